// pbr_slot.h - a node's slot as instance and mesh triangle, shared by the
// band and backward kernels and its host-side test.
#pragma once

#include <stdint.h>

// The header is plain arithmetic: hipcc builds it for host and device, the
// host test builds it with a C++ compiler.
#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define PBR_SLOT_HD __host__ __device__
#else
#define PBR_SLOT_HD
#endif

namespace pbr_slot {

// Instances of a node up to which split() is exact.
constexpr uint32_t kMaxInstances = 1u << 22;

// Instance i and triangle t of a node's slot `local` = i * ntri + t, inv =
// 1.0f / ntri.  The slot's conversion, the reciprocal and the product each
// round by at most 2^-24 of the value, so that the product is within 3 * 2^-24
// of the quotient's size of it: less than one for i < 2^22.  Truncated it is
// off by at most one then, and one step corrects it.  (An integer division by a
// run-time value is some twenty instructions.)
PBR_SLOT_HD inline void split(uint32_t local, int32_t ntri, float inv, uint32_t& i, int32_t& t) {
  i = (uint32_t)((float)local * inv);
  t = (int32_t)(local - i * (uint32_t)ntri);
  if (t < 0) {
    --i;
    t += ntri;
  } else if (t >= ntri) {
    ++i;
    t -= ntri;
  }
}

}  // namespace pbr_slot
