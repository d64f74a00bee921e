// Host check of pbr_slot.h: instance and triangle of a slot against integer
// division, for every mesh size of the band kernel, at every instance near the
// limit and near powers of two below it, and at every instance for a box.
// Prints "ok <cases>" or the first mismatch; exit code 1 on a mismatch.
#include <stdint.h>
#include <stdio.h>

#include "../../pybatchrender_amd/csrc/pbr_slot.h"

static long checked = 0;

static bool check(uint64_t i, int32_t ntri) {
  const float inv = 1.0f / (float)ntri;
  const int32_t at[4] = {0, ntri > 1 ? 1 : 0, ntri / 2, ntri - 1};
  for (int k = 0; k < 4; ++k) {
    const uint64_t local = i * (uint64_t)ntri + (uint64_t)at[k];
    if (i >= pbr_slot::kMaxInstances || local > 0xffffffffull) continue;
    uint32_t gi;
    int32_t gt;
    pbr_slot::split((uint32_t)local, ntri, inv, gi, gt);
    ++checked;
    if (gi != (uint32_t)i || gt != at[k]) {
      printf("mismatch ntri %d instance %llu triangle %d: %u %d\n", ntri, (unsigned long long)i,
             at[k], gi, gt);
      return false;
    }
  }
  return true;
}

int main() {
  for (int32_t ntri = 1; ntri <= 256; ++ntri) {
    for (uint64_t p = 1; p <= pbr_slot::kMaxInstances; p *= 2)
      for (int64_t d = -600; d <= 600; ++d)
        if ((int64_t)p + d >= 0 && !check((uint64_t)((int64_t)p + d), ntri)) return 1;
    for (uint64_t i = pbr_slot::kMaxInstances - 6000; i < pbr_slot::kMaxInstances; ++i)
      if (!check(i, ntri)) return 1;
  }
  for (uint64_t i = 0; i < pbr_slot::kMaxInstances; ++i)
    if (!check(i, 12)) return 1;
  printf("ok %ld\n", checked);
  return 0;
}
