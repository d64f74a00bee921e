// pbr_bands.hip - the band path: one workgroup draws one band of full rows of
// one scene from the scene's instances, with no records in device memory.
//
//   setup + raster  the scene's instances are dealt to the workgroup's eight or
//                   sixteen waves in chunks (as many instances of one node as
//                   the wave's vertex table holds).  A wave transforms and snaps the chunk's
//                   vertices once into its LDS table, drops the chunk if all
//                   of them lie outside one plane, off the band or between two
//                   pixel centres, tests each triangle on three table entries,
//                   queues the live ones and sets up 64 of them at a time.  A
//                   set-up triangle is rasterised at once - a small one by its
//                   lane, others by rows dealt to the lanes - into the band's
//                   64-bit pixel keys in LDS: atomicMin of depth bits << 32 |
//                   slot << 3 | sub-triangle, the winner the in-order
//                   strict-less depth test picks whatever the order of the
//                   fragments.  Triangles that straddle a clip plane wait in a
//                   queue that all waves clip and draw at the end.
//   resolve         covered pixels are queued per wave and shaded 64 at a
//                   time from the winner's instance and vertices, which are
//                   transformed again (fewer pixels are covered than triangles
//                   are set up, so keeping shading data per triangle costs
//                   more than making it per pixel); colours narrower than
//                   their key replace it in LDS and leave as whole dwords.
//
// Bound by vector instructions (8192 scenes of 84 x 84 with up to 256
// instances: 93% of the issue slots; 1585 us with the tile path's records, 535
// so); float frames of flat scenes also by the stores that follow setup (1024
// scenes of 128 x 128 with 64 boxes: 166 and 112).
//
// The arithmetic is the shared code of pbr_device.h, so the output is
// bit-identical to the other kernels.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>

#include "../../include/pbr_abi.h"
#include "pbr_device.h"
#include "pbr_host.h"
#include "pbr_slot.h"

using namespace pbr_host;

namespace {

constexpr int kBandWaves = 8;     // waves of a workgroup, two workgroups on a CU
constexpr int kWideWaves = 16;    // or one workgroup with all the waves of a CU, for
                                  // at most one workgroup a CU (see bands_plan)
constexpr int kBandVerts = 136;   // vertices a wave's table holds at most
constexpr int kBandTris = 256;    // triangles of one chunk (8-bit queue entries)
constexpr int kBandTable = 512;   // triangles of all meshes (LDS index table) at most
constexpr int kMaxBands = 4;      // bands per scene at most: each repeats the vertex work
constexpr int kBandPixels = 8192;
constexpr int kBandLds = 80 * 1024;  // half a CU's LDS: two workgroups share a CU
constexpr int kClipQueue = 128;   // clipped triangles that wait for the whole workgroup
constexpr int kSmallPixels = 12;  // box pixels one lane rasterises alone
constexpr uint32_t kDepthOne = 0x3f800000u;
// Sub-triangle number of a triangle that no plane clips (a clipped polygon has
// at most seven, 0 to 6), so that shading knows it without testing vertices.
constexpr uint32_t kUnclipped = 7;

// Per-node launch constants.
struct BandNode {
  uint32_t group;    // instances per chunk
  uint32_t inv_nv;   // ceil(2^16 / vertices): v / vertices = v * inv_nv >> 16
  uint32_t inv_nt;   // the same for triangles
};

struct BandFrame {
  int W, H, th, bands;
  float guard;
  uint32_t max_slots;  // slots of the largest scene
  uint32_t budget;     // slots drawn of the whole batch at most
  int uniform;         // 1: no node has per-scene counts
  int waves;           // of a workgroup
  int verts;           // entries of a wave's vertex table
  int ntab;            // triangles in the LDS index table
  int vec;             // 1: four pixels of a plane are whole aligned dwords / float4s
  BandNode node[PBR_MAX_NODES];
};

// Node facts a workgroup keeps in LDS.
struct NodeLds {
  const float* trans;
  const float* cols;
  uint32_t base, chunk0;  // first slot and first chunk of the node in this scene
  uint32_t cnt;           // active instances
  int32_t ntri, voff, ioff, ips;
  float inv_nt;           // 1 / ntri
  uint32_t flags;         // bit 0: shared, bit 1: flat
};

// A vertex table entry is the snapped position and the depth's bits.  A vertex
// that is outside a clip plane or did not snap (in a chunk that holds one) has
// this NaN | kNotSnapped | its outcode for the depth, which is finite in every
// other: a vertex inside the planes has a depth of 0 to 1.
constexpr uint32_t kCodeTag = 0xffc00000u;
constexpr uint32_t kOutMask = 0x3fu, kNotSnapped = 0x40u;
__device__ __forceinline__ uint32_t vertex_code(uint32_t d) {
  return d >= kCodeTag ? d & (kOutMask | kNotSnapped) : 0u;
}

// Lanes of m below this one.
__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Snapped extents (1/256 pixel) up to which edge values are evaluated in 32
// bits: coordinate differences are at most 2^14, their products 2^28, and
// the two products, the fill-rule bias and the overshoot of a block of
// pixels stay below 2^30.
constexpr int kIntExtent = 1 << 14;

typedef const __attribute__((address_space(1))) float global_cfloat;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) f32x4 global_cfloat4;

__device__ __forceinline__ void load_mat4_global(const float* src, float M[16]) {
  global_cfloat4* q = (global_cfloat4*)(uintptr_t)src;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const f32x4 v = q[r];
    M[4 * r] = v.x;
    M[4 * r + 1] = v.y;
    M[4 * r + 2] = v.z;
    M[4 * r + 3] = v.w;
  }
}

// Six floats of mesh vertex v.
__device__ __forceinline__ void load_vertex(const float* vertices, int v, float out[6]) {
  global_cfloat* p = (global_cfloat*)(uintptr_t)vertices + (size_t)v * 6;
#pragma unroll
  for (int q = 0; q < 6; ++q) out[q] = p[q];
}

// Vertex indices a | b << 8 | c << 16 of triangle q of the index pool.
__device__ __forceinline__ uint32_t pool_triangle(const pbr_scene_desc& D, int q) {
  const int32_t* t = D.indices + (size_t)q * 3;
  return (uint32_t)t[0] | ((uint32_t)t[1] << 8) | ((uint32_t)t[2] << 16);
}

// A value of lane `src`.
__device__ __forceinline__ int from_lane(int src, int v) {
  return __builtin_amdgcn_ds_bpermute(src << 2, v);
}
__device__ __forceinline__ float from_lane(int src, float v) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(src << 2, __float_as_int(v)));
}
// Sends v to lane `dst`; the lane's result is 0 if no lane sends to it.
__device__ __forceinline__ float to_lane(int dst, float v) {
  return __int_as_float(__builtin_amdgcn_ds_permute(dst << 2, __float_as_int(v)));
}

struct BandCtx {
  int s, W;
  int j0, j1;  // GL rows of the band; LDS row 0 is j1
};

// Depth test of one fragment: LDS atomicMin on the key (depth bits, rank).
// No read before it: with few fragments per pixel the read's latency costs
// more than the atomics it would save.
__device__ __forceinline__ void band_fragment(unsigned long long* q, float z, uint32_t rank) {
  atomicMin(q, ((unsigned long long)__float_as_uint(z) << 32) | rank);
}

// Edge function steps in 1/256 pixel: edge k is opposite vertex k,
// e_k(x, y) = A_k (x - X_a) + B_k (y - Y_a) - bias_k, inside <=> e_k >= 0.
// Num is int32_t (see kIntExtent) or double (every term an integer below
// 2^53, so the arithmetic is exact in either).
template <typename Num>
struct BandEdges {
  Num A[3], B[3], e[3];  // e at the first pixel centre
};

template <typename Num>
__device__ __forceinline__ void band_edges(const FixTri& T, int i, int j, BandEdges<Num>& E) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int a = (k + 1) % 3, b = (k + 2) % 3;
    const int32_t A = T.Y[a] - T.Y[b], B = T.X[b] - T.X[a];
    const int32_t dx = 256 * i + 128 - T.X[a], dy = 256 * j + 128 - T.Y[a];
    const int32_t bias = (int32_t)((T.bias >> k) & 1u);
    if constexpr (sizeof(Num) == 4) {
      E.e[k] = __mul24(A, dx) + __mul24(B, dy) - bias;
      E.A[k] = A * 256;
      E.B[k] = B * 256;
    } else {
      E.e[k] = fma((double)A, (double)dx, (double)B * (double)dy) - (double)bias;
      E.A[k] = (double)A * 256.0;
      E.B[k] = (double)B * 256.0;
    }
  }
}

__device__ __forceinline__ bool band_inside(const int32_t e[3]) { return (e[0] | e[1] | e[2]) >= 0; }

// One lane, the whole box.
__device__ __forceinline__ void band_raster_lane(unsigned long long* pix, const BandCtx& t,
                                                 const FixTri& T, uint32_t rank) {
  BandEdges<int32_t> E;
  band_edges(T, T.i0, T.j0, E);
  const float x0 = (float)T.i0 + 0.5f;
  unsigned long long* row = pix + (t.j1 - T.j0) * t.W + T.i0;
  const int w = T.i1 - T.i0;
  float y = (float)T.j0 + 0.5f;
  for (int h = T.j1 - T.j0; h >= 0; --h) {
    int32_t e[3] = {E.e[0], E.e[1], E.e[2]};
    const float tz = fmaf(T.zy, y, T.zc);
    float x = x0;
    for (int i = 0; i <= w; ++i) {
      if (band_inside(e)) band_fragment(row + i, clamp_depth(fmaf(T.zx, x, tz)), rank);
#pragma unroll
      for (int k = 0; k < 3; ++k) e[k] += E.A[k];
      x += 1.0f;  // exact: a pixel centre
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) E.e[k] += E.B[k];
    y += 1.0f;
    row -= t.W;
  }
}

// Pixels lo .. hi of a row of w + 1 that lie inside the three edges (e at the
// row's first pixel): each edge's crossing from a reciprocal estimate, off by
// less than a pixel's half, and one exact evaluation at the nearest pixel.
__device__ __forceinline__ void row_span(const BandEdges<double>& E, int w, int& lo, int& hi) {
  lo = 0;
  hi = w;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double A = E.A[k], e = E.e[k];
    const double q = rint(-e * __builtin_amdgcn_rcp(A));
    // in range before it becomes an integer (A = 0: any value)
    const double c = fmin(fmax(q, -1.0), (double)(w + 1));
    const bool out = __builtin_fma(A, c, e) < 0.0;
    const int i = (int)c;
    if (A > 0.0) lo = max(lo, out ? i + 1 : i);
    else if (A < 0.0) hi = min(hi, out ? i - 1 : i);
    else if (e < 0.0) hi = -1;
  }
}

// The rows of the lanes' triangles (`has`) dealt to the lanes of the wave, 64
// rows at a time: a lane finds its triangle by a binary search of the running
// row counts and walks the row.  Triangles of more than a few pixels keep the
// whole wave busy this way, where a lane per triangle would walk as long as
// the largest box.  Num int32_t (extents within kIntExtent) tests each pixel
// of the box's row; double, for the long thin triangles that reach out of the
// frame, walks the row's span: in blocks of 8 x 8 pixels of the box they took
// a steering scene's wave longest of all.
template <typename Num>
__device__ __forceinline__ void band_raster_rows(unsigned long long* pix, const BandCtx& t,
                                                 int lane, bool has, const FixTri& T,
                                                 uint32_t rank) {
  const int incl = wave_scan_add(has ? T.j1 - T.j0 + 1 : 0);
  const int total = __builtin_amdgcn_readlane(incl, 63);
  // columns (W <= 8192) and fill-rule bias in one word
  const int box = T.i0 | (T.i1 << 13) | (int)(T.bias << 26);
  for (int r0 = 0; r0 < total; r0 += 64) {
    const int r = min(r0 + lane, total - 1);
    int l = 0;  // the first lane whose running count exceeds r
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) l = from_lane(l + d - 1, incl) <= r ? l + d : l;
    FixTri U;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      U.X[k] = from_lane(l, T.X[k]);
      U.Y[k] = from_lane(l, T.Y[k]);
    }
    const float zx = from_lane(l, T.zx), zy = from_lane(l, T.zy), zc = from_lane(l, T.zc);
    const int b = from_lane(l, box);
    const int j = from_lane(l, T.j1) - (from_lane(l, incl) - 1 - r);
    const uint32_t ur = (uint32_t)from_lane(l, (int)rank);
    U.bias = (uint32_t)b >> 26;
    const int i0 = b & 0x1fff, w = ((b >> 13) & 0x1fff) - i0;
    BandEdges<Num> E;
    band_edges(U, i0, j, E);
    const float tz = fmaf(zy, (float)j + 0.5f, zc);
    unsigned long long* q = pix + (t.j1 - j) * t.W + i0;
    if (r0 + lane >= total) continue;
    if constexpr (sizeof(Num) == 4) {
      float x = (float)i0 + 0.5f;
      for (int i = 0; i <= w; ++i) {
        if (band_inside(E.e)) band_fragment(q + i, clamp_depth(fmaf(zx, x, tz)), ur);
#pragma unroll
        for (int k = 0; k < 3; ++k) E.e[k] += E.A[k];
        x += 1.0f;
      }
    } else {
      int lo, hi;
      row_span(E, w, lo, hi);
      float x = (float)(i0 + lo) + 0.5f;
      for (int i = lo; i <= hi; ++i) {
        band_fragment(q + i, clamp_depth(fmaf(zx, x, tz)), ur);
        x += 1.0f;
      }
    }
  }
}

// Bit p: not inside clip plane p (NaN distances count as outside, as the
// clipper takes them).
__device__ __forceinline__ uint32_t outcode(const CVert& v, float guard) {
  uint32_t oc = 0;
#pragma unroll
  for (int p = 0; p < 6; ++p) oc |= plane_dist(v, p, guard) >= 0.0f ? 0u : 1u << p;
  return oc;
}

// Sutherland-Hodgman on four polygons at once, one per group of 16 lanes: lane
// k of a group holds vertex k < n (every lane of the wave takes part; NC = 4
// clips positions, 7 normals too).  The same planes, order, intersections and
// vertex limit as clip_polygon; a plane that has every vertex inside leaves
// the polygons as they are and is skipped.  In registers: clip_polygon's
// arrays lie in scratch memory, where clipping 64 triangles at a time took
// most of the 95 us a steering scene's workgroup spent on setup.
template <int NC>
__device__ __forceinline__ void clip_groups(float v[NC], int& n, float guard, int lane) {
  const int k = lane & 15, base = lane & 48;
  for (int plane = 0; plane < 6; ++plane) {
    CVert a, b;
#pragma unroll
    for (int c = 0; c < 4; ++c) a.p[c] = v[c];
    const float da = plane_dist(a, plane, guard);
    const bool act = k < n, ina = act && da >= 0.0f;
    if (!__ballot(act && !ina)) continue;
    const int nx = base + (k + 1 >= n ? 0 : k + 1);
    float w[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) w[c] = from_lane(nx, v[c]);
#pragma unroll
    for (int c = 0; c < 4; ++c) b.p[c] = w[c];
    const float db = plane_dist(b, plane, guard);
    const bool cross = act && ina != (db >= 0.0f);
    const float di = ina ? da : db, dout = ina ? db : da;
    const float t = di / (di - dout);
    float r[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const float vi = ina ? v[c] : w[c], vo = ina ? w[c] : v[c];
      r[c] = vi + t * (vo - vi);
    }
    const uint32_t mi = (uint32_t)(__ballot(ina) >> base) & 0xffffu;
    const uint32_t mx = (uint32_t)(__ballot(cross) >> base) & 0xffffu;
    const uint32_t below = (1u << k) - 1u;
    const int pa = __popc(mi & below) + __popc(mx & below), px = pa + (ina ? 1 : 0);
    // lane 15 of a group takes what goes nowhere (a polygon has <= 9 vertices)
    const int ta = base + (ina && pa < kMaxPoly ? pa : 15);
    const int tx = base + (cross && px < kMaxPoly ? px : 15);
    const bool is_x = to_lane(tx, 1.0f) != 0.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const float va = to_lane(ta, v[c]), vx = to_lane(tx, r[c]);
      v[c] = is_x ? vx : va;
    }
    n = min(__popc(mi) + __popc(mx), kMaxPoly);
  }
}

// Vertices (clip position, world normal) of the mesh triangles of four slots,
// vertex k of group g's triangle in lane 16 g + k (k < 3).
__device__ __forceinline__ void group_vertex(const pbr_scene_desc& D, const float* trans,
                                             size_t row, int voff, uint32_t tri,
                                             const float VP[16], int lane, CVert& cv) {
  const int k = lane & 15;
  const uint32_t id = k == 0 ? tri & 0xffu : (k == 1 ? (tri >> 8) & 0xffu : tri >> 16);
  float M[16], vv[6];
  load_mat4_global(trans + row * 16, M);
  load_vertex(D.vertices, voff + (int)id, vv);
  transform_vertex(M, VP, vv, cv);
}

// A slot's node, its instance row in the node's buffers and its mesh triangle.
struct SlotRef {
  const float* trans;
  const float* cols;
  size_t row;
  int voff;
  uint32_t tri;    // vertex indices a | b << 8 | c << 16
  uint32_t flags;  // the node's (NodeLds)
};

__device__ __forceinline__ SlotRef band_slot(int s, const NodeLds* nodes, int nn,
                                             const uint32_t* tab, uint32_t slot) {
  int nj = 0;
  for (int k = 1; k < nn; ++k) nj = slot >= nodes[k].base ? k : nj;
  const NodeLds& nd = nodes[nj];
  const uint32_t local = slot - nd.base;
  uint32_t i;
  int32_t t;
  pbr_slot::split(local, nd.ntri, nd.inv_nt, i, t);
  SlotRef R;
  R.trans = nd.trans;
  R.cols = nd.cols;
  R.row = (nd.flags & 1u) ? (size_t)i : (size_t)s * (size_t)nd.ips + i;
  R.voff = nd.voff;
  R.tri = tab[nd.ioff + t];
  R.flags = nd.flags;
  return R;
}

// Colours of the pixels in lanes 0 .. take - 1 (GL pixel (x, j), winner `slot`
// and sub-triangle q).

// Flat scenes: every lane shades its own winner's first normal.
__device__ __forceinline__ void band_shade_flat(const pbr_scene_desc& D, const Light& lt, int s,
                                                const NodeLds* nodes, int nn, const uint32_t* tab,
                                                int lane, uint32_t take, uint32_t slot,
                                                float col[4]) {
  if ((uint32_t)lane >= take) return;
  const SlotRef R = band_slot(s, nodes, nn, tab, slot);
  float M[16], v[6], nw[3], n[3];
  load_mat4_global(R.trans + R.row * 16, M);
  const f32x4 c4 = ((global_cfloat4*)(uintptr_t)R.cols)[R.row];
  const float rgba[4] = {c4.x, c4.y, c4.z, c4.w};
  load_vertex(D.vertices, R.voff + (int)(R.tri & 0xffu), v);
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const float a = M[r * 4 + 0] * v[3] + M[r * 4 + 1] * v[4];
    nw[r] = a + M[r * 4 + 2] * v[5];
  }
  normalize3(nw, n);
  shade(n, rgba, lt, col);
}

// Smooth scenes.  Runs of pixels with one winner share its vertices when the
// pixels form at most kShadeRuns runs: lane 3 u + k transforms vertex k of
// the u-th run's triangle, and every pixel of the run reads the three back.
// With more runs (triangles of a pixel or two) every lane transforms its own
// winner's three vertices.  `heads` is 64 bytes of the wave's LDS.
constexpr int kShadeRuns = 21;
__device__ __forceinline__ void band_shade_smooth(const pbr_scene_desc& D, const BandFrame& F,
                                                  const Light& lt, int s, const float VP[16],
                                                  const NodeLds* nodes, int nn,
                                                  const uint32_t* tab, int lane, uint32_t take,
                                                  uint32_t slot, int q, int x, int j,
                                                  uint8_t* heads, float col[4]) {
  const bool mine = (uint32_t)lane < take;
  const int prev = from_lane(lane > 0 ? lane - 1 : 0, (int)slot);
  const bool head = mine && (lane == 0 || (uint32_t)prev != slot);
  const uint64_t hm = __ballot(head);
  const int runs = __popcll(hm);
  int32_t X[3] = {0, 0, 0}, Y[3] = {0, 0, 0};
  float iw[3] = {0.0f, 0.0f, 0.0f}, n[3][3] = {}, base[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  uint32_t fl = 0;  // the winner's node flags
  if (runs <= kShadeRuns) {
    const int run = __popcll(hm & ((2ull << lane) - 1ull)) - 1;
    if (head) heads[run] = (uint8_t)lane;
    wave_fence();
    const int u = (lane * 86) >> 8, k = lane - 3 * u;
    CVert cv = {};
    SnapVert sv = {};
    uint32_t vf = 0;
    float rgba[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    // every lane takes part in the reads of other lanes' slots
    const uint32_t vslot = (uint32_t)from_lane(u < runs ? (int)heads[u] : 0, (int)slot);
    if (u < runs) {
      const SlotRef R = band_slot(s, nodes, nn, tab, vslot);
      const f32x4 c4 = ((global_cfloat4*)(uintptr_t)R.cols)[R.row];
      rgba[0] = c4.x;
      rgba[1] = c4.y;
      rgba[2] = c4.z;
      rgba[3] = c4.w;
      const uint32_t id = k == 0 ? R.tri & 0xffu : (k == 1 ? (R.tri >> 8) & 0xffu : R.tri >> 16);
      float M[16], vv[6];
      load_mat4_global(R.trans + R.row * 16, M);
      load_vertex(D.vertices, R.voff + (int)id, vv);
      transform_vertex(M, VP, vv, cv);
      snap_vertex(cv, F.W, F.H, sv);
      vf = R.flags;
    }
    const int src = mine ? 3 * run : 0;
#pragma unroll
    for (int v = 0; v < 3; ++v) {
      X[v] = from_lane(src + v, sv.X);
      Y[v] = from_lane(src + v, sv.Y);
      iw[v] = from_lane(src + v, sv.invw);
#pragma unroll
      for (int c = 0; c < 3; ++c) n[v][c] = from_lane(src + v, cv.n[c]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) base[c] = from_lane(src, rgba[c]);
    fl = (uint32_t)from_lane(src, (int)vf);
  } else if (mine) {
    const SlotRef R = band_slot(s, nodes, nn, tab, slot);
    const f32x4 c4 = ((global_cfloat4*)(uintptr_t)R.cols)[R.row];
    base[0] = c4.x;
    base[1] = c4.y;
    base[2] = c4.z;
    base[3] = c4.w;
    float M[16];
    load_mat4_global(R.trans + R.row * 16, M);
    fl = R.flags;
#pragma unroll
    for (int v = 0; v < 3; ++v) {
      float vv[6];
      load_vertex(D.vertices, R.voff + (int)((R.tri >> (8 * v)) & 0xffu), vv);
      CVert cv;
      SnapVert sv;
      transform_vertex(M, VP, vv, cv);
      snap_vertex(cv, F.W, F.H, sv);
      X[v] = sv.X;
      Y[v] = sv.Y;
      iw[v] = sv.invw;
#pragma unroll
      for (int c = 0; c < 3; ++c) n[v][c] = cv.n[c];
    }
  }
  const bool flat = (fl & 2u) != 0u;

  // winners that straddle a clip plane: their polygons, four slots at a time
  bool clipped = mine && !flat && q != (int)kUnclipped;
  for (uint64_t cm = __ballot(clipped); cm; cm = __ballot(clipped)) {
    uint32_t gs = 0;
    int group = -1, count = 0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (!cm) break;
      const uint32_t sl = (uint32_t)__builtin_amdgcn_readlane(
          (int)slot, __ffsll((unsigned long long)cm) - 1);
      if ((lane >> 4) == g) gs = sl;
      const bool hit = clipped && slot == sl;
      if (hit) group = g;
      cm &= ~__ballot(hit);
      ++count;
    }
    CVert p = {};
    int pn = 0;
    if ((lane >> 4) < count) {
      pn = 3;
      if ((lane & 15) < 3) {
        const SlotRef R = band_slot(s, nodes, nn, tab, gs);
        group_vertex(D, R.trans, R.row, R.voff, R.tri, VP, lane, p);
      }
    }
    float v[7] = {p.p[0], p.p[1], p.p[2], p.p[3], p.n[0], p.n[1], p.n[2]};
    clip_groups<7>(v, pn, F.guard, lane);
#pragma unroll
    for (int c = 0; c < 4; ++c) p.p[c] = v[c];
    SnapVert ps;
    snap_vertex(p, F.W, F.H, ps);
    const int at = group < 0 ? 0 : group * 16;
    const int from[3] = {at, at + q + 1, at + q + 2};
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const int px = from_lane(from[e], ps.X), py = from_lane(from[e], ps.Y);
      const float pw = from_lane(from[e], ps.invw);
      float pnm[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) pnm[c] = from_lane(from[e], v[4 + c]);
      if (group >= 0) {
        X[e] = px;
        Y[e] = py;
        iw[e] = pw;
#pragma unroll
        for (int c = 0; c < 3; ++c) n[e][c] = pnm[c];
      }
    }
    clipped = clipped && group < 0;
  }
  if (mine) {
    // weights e_k / w_k, e_k the edge function without the fill-rule bias:
    // every difference and product is an exact integer in double
    const int32_t cx = 256 * x + 128, cy = 256 * j + 128;
    float bw[3], nn3[3];
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const int a = (e + 1) % 3, b = (e + 2) % 3;
      const double ev = fma((double)(Y[a] - Y[b]), (double)(cx - X[a]),
                            (double)(X[b] - X[a]) * (double)(cy - Y[a]));
      bw[e] = (float)ev * iw[e];
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float a = bw[0] * n[0][c] + bw[1] * n[1][c];
      nn3[c] = flat ? n[0][c] : a + bw[2] * n[2][c];
    }
    shade(nn3, base, lt, col);
  }
}

// Byte c of each of four packed RGBA8 colours -> one dword.
__device__ __forceinline__ uint32_t band_gather(uint32_t p0, uint32_t p1, uint32_t p2, uint32_t p3,
                                                int c) {
  const uint32_t sel = (uint32_t)c | ((uint32_t)(4 + c) << 8) | 0x0c0c0000u;
  return __builtin_amdgcn_perm(__builtin_amdgcn_perm(p3, p2, sel),
                               __builtin_amdgcn_perm(p1, p0, sel), 0x05040100u);
}

// OM: 0 uint8, 1 bf16, 2 float32 colours.  Dynamic LDS: pixel keys
// [th][W], the waves' vertex tables (int2 [verts], float depth [verts]) and
// triangle queues, then the index table.
template <bool SMOOTH, int OM>
__global__ __launch_bounds__(kWideWaves * 64)
__attribute__((amdgpu_waves_per_eu(4))) void
bands_kernel(pbr_scene_desc D, pbr_frame_out O, BandFrame F, const uint32_t* scene_off,
             const uint32_t* order, uint32_t* hdr, Light lt, float4 bg) {
  extern __shared__ __align__(16) unsigned long long pix[];
  __shared__ NodeLds nodes[PBR_MAX_NODES];
  __shared__ uint32_t next_chunk, total_chunks, covered_n, clip_total;
  __shared__ uint32_t clip_queue[kClipQueue];
  const int tid = (int)threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int W = F.W, H = F.H, nn = D.num_nodes;
  const int waves = F.waves, block = waves * 64;
  BandCtx t;
  const uint32_t at = blockIdx.x / (uint32_t)F.bands;
  const int band = (int)(blockIdx.x - at * (uint32_t)F.bands);
  t.s = (int)(order ? order[at] : at);
  const int yo0 = band * F.th, rows = min(F.th, H - yo0);
  t.W = W;
  t.j1 = H - 1 - yo0;
  t.j0 = t.j1 - (rows - 1);
  const int npx = rows * W;
  int2* tables = reinterpret_cast<int2*>(pix + ((F.th * W + 1) & ~1));
  int2* vxy = tables + wave * F.verts;
  unsigned char* after = reinterpret_cast<unsigned char*>(tables + waves * F.verts);
  uint32_t* vd = reinterpret_cast<uint32_t*>(after) + wave * F.verts;
  after += sizeof(float) * (size_t)waves * F.verts;
  uint8_t* qu = after + wave * kBandTris;
  uint32_t* tab = reinterpret_cast<uint32_t*>(after + waves * kBandTris);

  if (F.uniform && blockIdx.x == 0 && tid == 0) hdr[0] = 0u;  // no overflow
  // slots of this scene that are drawn (all, unless the batch exceeds its
  // slot budget)
  uint32_t ndraw;
  if (F.uniform) {
    const uint64_t o = min((uint64_t)t.s * F.max_slots, (uint64_t)F.budget);
    ndraw = (uint32_t)min((uint64_t)F.max_slots, (uint64_t)F.budget - o);
  } else {
    const uint32_t o = min(scene_off[t.s], F.budget), e = min(scene_off[t.s + 1], F.budget);
    ndraw = e > o ? e - o : 0u;
  }
  // two keys per store (the key area is padded to an even count)
  for (int p = tid; p < (npx + 1) / 2; p += block)
    reinterpret_cast<uint4*>(pix)[p] = make_uint4(0u, kDepthOne, 0u, kDepthOne);
  for (int q = tid; q < F.ntab; q += block) tab[q] = pool_triangle(D, q);
  if (wave == 0) {
    uint32_t cnt = 0, nslot = 0, nchunk = 0;
    if (lane < nn) {
      const pbr_node& nd = D.nodes[lane];
      const pbr_mesh& me = D.meshes[nd.mesh];
      int c = nd.instances_per_scene;
      if (nd.counts) c = min(max(nd.counts[t.s], 0), nd.instances_per_scene);
      cnt = me.num_triangles > 0 ? (uint32_t)c : 0u;
      nslot = cnt * (uint32_t)me.num_triangles;
      const uint32_t g = F.node[lane].group;
      nchunk = (cnt + g - 1u) / g;
    }
    const uint32_t is = (uint32_t)wave_scan_add((int)nslot);
    const uint32_t ic = (uint32_t)wave_scan_add((int)nchunk);
    if (lane < nn) {
      const pbr_node& nd = D.nodes[lane];
      const pbr_mesh& me = D.meshes[nd.mesh];
      NodeLds e;
      e.trans = nd.transforms;
      e.cols = nd.colors;
      e.base = is - nslot;
      e.chunk0 = ic - nchunk;
      e.cnt = cnt;
      e.ntri = max(me.num_triangles, 1);
      e.inv_nt = 1.0f / (float)e.ntri;
      e.voff = me.vertex_offset;
      e.ioff = me.index_offset;
      e.ips = nd.instances_per_scene;
      e.flags = (nd.shared ? 1u : 0u) | (nd.flat ? 2u : 0u);
      nodes[lane] = e;
    }
    if (lane == 63) {
      next_chunk = 0u;
      covered_n = 0u;
      clip_total = 0u;
      total_chunks = ic;
    }
  }
  __syncthreads();

  float VP[16];
  load_mat4_uniform(D.view_proj + (size_t)t.s * 16, VP);

  // --- setup and raster --------------------------------------------------------
  const uint32_t chunks = __builtin_amdgcn_readfirstlane((int)total_chunks);
  // set-up triangles of the lanes (`has`) into the band's pixels
  auto draw = [&](bool has, const FixTri& T, uint32_t rank) {
    const bool fits =  // edge values fit 32 bits
        has &&
        max(T.X[0], max(T.X[1], T.X[2])) - min(T.X[0], min(T.X[1], T.X[2])) <= kIntExtent &&
        max(T.Y[0], max(T.Y[1], T.Y[2])) - min(T.Y[0], min(T.Y[1], T.Y[2])) <= kIntExtent;
    const int w = T.i1 - T.i0 + 1, h = T.j1 - T.j0 + 1;
    const bool small = fits && w * h <= kSmallPixels;
    if (small) band_raster_lane(pix, t, T, rank);
    const bool rows = fits && !small;
    if (__ballot(rows)) band_raster_rows<int32_t>(pix, t, lane, rows, T, rank);
    const bool far = has && !fits;
    if (__ballot(far)) band_raster_rows<double>(pix, t, lane, far, T, rank);
  };
  // four triangles that straddle a clip plane, one per group of 16 lanes, a
  // lane per sub-triangle
  auto draw_clipped = [&](uint32_t slot, bool some) {
    FixTri T;
    CVert cv = {};
    int pn = some ? 3 : 0;
    if (some && (lane & 15) < 3) {
      const SlotRef R = band_slot(t.s, nodes, nn, tab, slot);
      group_vertex(D, R.trans, R.row, R.voff, R.tri, VP, lane, cv);
    }
    clip_groups<4>(cv.p, pn, F.guard, lane);
    SnapVert S;
    snap_vertex(cv, W, H, S);
    const int lost = 0x7fffffff;  // X of a vertex that did not snap
    const int X = S.ok ? S.X : lost;
    const int at = lane & 48, q = lane & 15;
    const bool sub = q + 2 < pn;
    const int f1 = sub ? at + q + 1 : at, f2 = sub ? at + q + 2 : at;
    SnapVert V[3];
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const int f = e == 0 ? at : (e == 1 ? f1 : f2);
      V[e].X = from_lane(f, X);
      V[e].Y = from_lane(f, S.Y);
      V[e].d = from_lane(f, S.d);
      V[e].invw = 0.0f;
      V[e].ok = V[e].X != lost;
    }
    const bool has = sub && setup_snapped(V[0], V[1], V[2], W, H, t.j0, t.j1, T);
    const uint32_t rank = (slot << 3) | (uint32_t)q;
    draw(has, T, rank);
  };
  for (;;) {
    uint32_t c = 0;
    if (lane == 0) c = atomicAdd(&next_chunk, 1u);
    c = (uint32_t)__builtin_amdgcn_readfirstlane((int)c);
    if (c >= chunks) break;
    int j = 0;
    for (int k = 1; k < nn; ++k)
      j = c >= (uint32_t)__builtin_amdgcn_readfirstlane((int)nodes[k].chunk0) ? k : j;
    // the node's facts in scalar registers, loaded once per chunk
    const pbr_node& nd = D.nodes[j];
    const pbr_mesh& me = D.meshes[nd.mesh];
    const uint32_t group = F.node[j].group, inv_nv = F.node[j].inv_nv, inv_nt = F.node[j].inv_nt;
    const float* trans = nd.transforms;
    const int voff = me.vertex_offset;
    const uint32_t nt = (uint32_t)me.num_triangles, nv = (uint32_t)me.num_vertices;
    const uint32_t* mtab = tab + me.index_offset;
    const uint32_t cnt = (uint32_t)__builtin_amdgcn_readfirstlane((int)nodes[j].cnt);
    const uint32_t base = (uint32_t)__builtin_amdgcn_readfirstlane((int)nodes[j].base);
    const uint32_t i0 =
        (c - (uint32_t)__builtin_amdgcn_readfirstlane((int)nodes[j].chunk0)) * group;
    const uint32_t g = min(group, cnt - i0);
    const uint32_t slot0 = base + i0 * nt;
    if (slot0 >= ndraw) continue;
    const uint32_t n = min(g * nt, ndraw - slot0);
    const size_t row0 = nd.shared ? (size_t)i0 : (size_t)t.s * (size_t)nd.instances_per_scene + i0;

    // vertices of the chunk into the wave's table.  `dirty`: some vertex is
    // outside a clip plane or did not snap; only then are outcodes made
    // (`out`: the planes that all vertices lie outside of) and tested.
    bool dirty = false;
    uint32_t out = kOutMask;
    constexpr int kFar = 1 << 28;
    int xmin = kFar, xmax = -kFar, ymin = kFar, ymax = -kFar;
    auto vertex = [&](uint32_t v, uint32_t k, const float* M) {
      float vv[6];
      load_vertex(D.vertices, voff + (int)k, vv);
      CVert cv;
      transform_vertex(M, VP, vv, cv);
      // plane_dist is >= 0 on both sides of an axis just when this is (a sum's
      // sign is exact, and NaN fails in both)
      const float w = cv.p[3], gw = F.guard * w;
      const bool in = w - fabsf(cv.p[2]) >= 0.0f && gw - fabsf(cv.p[0]) >= 0.0f &&
                      gw - fabsf(cv.p[1]) >= 0.0f;
      // snap_vertex without its early returns
      const float iw = 1.0f / w;
      const float nx = cv.p[0] * iw, ny = cv.p[1] * iw, nz = cv.p[2] * iw;
      const float sx = (nx + 1.0f) * (0.5f * (float)W), sy = (ny + 1.0f) * (0.5f * (float)H);
      const bool ok = w > 0.0f && fabsf(sx) < 65536.0f && fabsf(sy) < 65536.0f;
      int X = (int)rintf(sx * 256.0f), Y = (int)rintf(sy * 256.0f);
      uint32_t d = __float_as_uint(nz * 0.5f + 0.5f), oc = 0u;
      if (__ballot(!(in && ok))) {
        dirty = true;
        oc = outcode(cv, F.guard);
        const uint32_t code = oc | (ok ? 0u : kNotSnapped);
        if (code) d = kCodeTag | code;
        X = ok ? X : 0;
        Y = ok ? Y : 0;
      }
      out &= oc;
      vxy[v] = make_int2(X, Y);
      vd[v] = d;
      xmin = min(xmin, X);
      xmax = max(xmax, X);
      ymin = min(ymin, Y);
      ymax = max(ymax, Y);
    };
    if (group == 1u) {
      float M[16];
      load_mat4_uniform(trans + row0 * 16, M);
      for (uint32_t v = (uint32_t)lane; v < nv; v += 64u) vertex(v, v, M);
    } else {
      for (uint32_t v = (uint32_t)lane; v < g * nv; v += 64u) {
        const uint32_t di = __umul24(v, inv_nv) >> 16;
        float M[16];
        load_mat4_global(trans + (row0 + di) * 16, M);
        vertex(v, v - __umul24(di, nv), M);
      }
    }
    // A chunk is dropped when all of it lies outside one plane, beside the
    // band, or between the same two columns or rows of pixel centres.
    bool gone = false;
    dirty = __ballot(dirty) != 0ull;  // lanes without a vertex in the last round too
    if (dirty) {
#pragma unroll
      for (int b = 0; b < 6; ++b) gone = gone || __ballot(!((out >> b) & 1u)) == 0ull;
    } else {
      // first and last centre of the lane's vertices; none where c1 < c0
      const int cx0 = (xmin + 127) >> 8, cx1 = (xmax - 128) >> 8;
      const int cy0 = (ymin + 127) >> 8, cy1 = (ymax - 128) >> 8;
      const int kx = __builtin_amdgcn_readfirstlane(cx0), ky = __builtin_amdgcn_readfirstlane(cy0);
      const bool any = xmin <= xmax;
      gone = !__ballot(cx1 >= 0) || !__ballot(cx0 < W) || !__ballot(cy1 >= t.j0) ||
             !__ballot(cy0 <= t.j1) || !__ballot(any && (cx0 != kx || cx1 >= kx)) ||
             !__ballot(any && (cy0 != ky || cy1 >= ky));
    }
    if (gone) continue;
    wave_fence();

    // triangles: every one is tested on its table entries; the live ones are
    // queued from the front, those that straddle a clip plane from the back
    uint32_t live_n = 0, clip_n = 0;
    for (uint32_t q0 = 0; q0 < n; q0 += 64u) {
      const uint32_t u = min(q0 + (uint32_t)lane, n - 1u);
      const uint32_t di = __umul24(u, inv_nt) >> 16;
      const uint32_t tri = mtab[u - __umul24(di, nt)];
      const uint32_t vb = __umul24(di, nv);
      const uint32_t ia = vb + (tri & 0xffu), ib = vb + ((tri >> 8) & 0xffu), ic = vb + (tri >> 16);
      const int2 a = vxy[ia], b = vxy[ib], cc = vxy[ic];
      const int32_t X[3] = {a.x, b.x, cc.x}, Y[3] = {a.y, b.y, cc.y};
      FixTri T;
      snapped_box(X, Y, W, t.j0, t.j1, T);
      const bool here = q0 + (uint32_t)lane < n;
      bool live = here && T.i0 <= T.i1 && T.j0 <= T.j1 && snapped_area(X, Y) > 0.0;
      if (dirty) {
        const uint32_t ca = vertex_code(vd[ia]), cb = vertex_code(vd[ib]), c3 = vertex_code(vd[ic]);
        const uint32_t some = ca | cb | c3;
        const bool clip = here && (some & kOutMask) && !(ca & cb & c3 & kOutMask);
        live = live && some == 0u;
        const uint64_t mc = __ballot(clip);
        if (clip) qu[kBandTris - 1u - (clip_n + lanes_below(mc))] = (uint8_t)u;
        clip_n += (uint32_t)__popcll(mc);
      }
      const uint64_t ml = __ballot(live);
      if (live) qu[live_n + lanes_below(ml)] = (uint8_t)u;
      live_n += (uint32_t)__popcll(ml);
    }
    wave_fence();

    // 64 live triangles are set up at a time and rasterised at once
    for (uint32_t k0 = 0; k0 < live_n; k0 += 64u) {
      FixTri T;
      bool has = false;
      uint32_t rank = 0;
      if (k0 + (uint32_t)lane < live_n) {
        const uint32_t u = qu[k0 + (uint32_t)lane];
        const uint32_t di = __umul24(u, inv_nt) >> 16;
        const uint32_t tri = mtab[u - __umul24(di, nt)];
        const uint32_t vb = __umul24(di, nv);
        const uint32_t ia = vb + (tri & 0xffu), ib = vb + ((tri >> 8) & 0xffu),
                       ic = vb + (tri >> 16);
        const int2 a = vxy[ia], b = vxy[ib], cc = vxy[ic];
        const int32_t X[3] = {a.x, b.x, cc.x}, Y[3] = {a.y, b.y, cc.y};
        const float d[3] = {__uint_as_float(vd[ia]), __uint_as_float(vd[ib]),
                            __uint_as_float(vd[ic])};
        snapped_box(X, Y, W, t.j0, t.j1, T);
        snapped_planes(X, Y, d, T);
        has = true;
        rank = ((slot0 + u) << 3) | kUnclipped;
      }
      draw(has, T, rank);
    }
    // clipped ones go to the workgroup's queue, so that a mesh which crosses
    // the near plane does not keep one wave while the others run out of
    // chunks; what does not fit is drawn at once
    if (clip_n) {
      uint32_t first = 0;
      if (lane == 0) first = atomicAdd(&clip_total, clip_n);
      first = (uint32_t)__builtin_amdgcn_readfirstlane((int)first);
      const uint32_t room = first < (uint32_t)kClipQueue ? kClipQueue - first : 0u;
      for (uint32_t k = (uint32_t)lane; k < min(clip_n, room); k += 64u)
        clip_queue[first + k] = slot0 + qu[kBandTris - 1u - k];
      for (uint32_t k0 = room; k0 < clip_n; k0 += 4u) {
        const uint32_t k = k0 + (uint32_t)(lane >> 4);
        draw_clipped(slot0 + qu[kBandTris - 1u - min(k, clip_n - 1u)], k < clip_n);
      }
    }
    wave_fence();  // the next chunk rewrites the table
  }
  __syncthreads();
  const uint32_t clips =
      min((uint32_t)__builtin_amdgcn_readfirstlane((int)clip_total), (uint32_t)kClipQueue);
  if (clips) {
    for (uint32_t k0 = (uint32_t)wave * 4u; k0 < clips; k0 += (uint32_t)waves * 4u) {
      const uint32_t k = k0 + (uint32_t)(lane >> 4);
      draw_clipped(clip_queue[min(k, clips - 1u)], k < clips);
    }
    __syncthreads();
  }

  // --- resolve -----------------------------------------------------------------
  const int C = O.channels;
  const size_t plane = (size_t)H * (size_t)W;
  const size_t pix0 = (size_t)yo0 * W;  // the band is contiguous in every plane
  float* dep = O.depth ? O.depth + (size_t)t.s * plane + pix0 : nullptr;
  int32_t* vis = O.vis ? O.vis + (size_t)t.s * plane + pix0 : nullptr;
  const float bgc[4] = {bg.x, bg.y, bg.z, bg.w};
  unsigned long long bgk = 0;
  if constexpr (OM == 0) bgk = pack_rgba8(bgc);
  if constexpr (OM == 1)
    bgk = (unsigned long long)(bf16_rne(bgc[0]) | (bf16_rne(bgc[1]) << 16)) |
          ((unsigned long long)(bf16_rne(bgc[2]) | (bf16_rne(bgc[3]) << 16)) << 32);
  float* fout = reinterpret_cast<float*>(O.color) + (size_t)t.s * C * plane + pix0;  // OM 2
  const float inv_w = 1.0f / (float)W;
  const int step = F.vec ? 4 : 1;  // pixels per lane of a scan
  const uint64_t below = (1ull << lane) - 1ull;
  // Scan of the 64 x step pixels from p0 (those below `end`): depths, ids and
  // backgrounds leave; bit k of the result: the lane's pixel k is covered
  // (pixels p0 + lane * step + k).
  auto scan = [&](int p0, int end) -> uint32_t {
    uint32_t cov = 0;
    const int p = p0 + lane * step;
    if (p >= end) return 0u;
    if (F.vec) {
      const ulonglong2 ka = *reinterpret_cast<const ulonglong2*>(pix + p);
      const ulonglong2 kb = *reinterpret_cast<const ulonglong2*>(pix + p + 2);
      const unsigned long long key[4] = {ka.x, ka.y, kb.x, kb.y};
#pragma unroll
      for (int k = 0; k < 4; ++k) cov |= (uint32_t)(key[k] >> 32) < kDepthOne ? 1u << k : 0u;
      if (dep) {
        float z[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          z[k] = (cov >> k) & 1u ? __uint_as_float((uint32_t)(key[k] >> 32)) : 1.0f;
        store_stream(dep + p, make_float4(z[0], z[1], z[2], z[3]));
      }
      if (vis) {
        int v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = (cov >> k) & 1u ? (int)((uint32_t)key[k] >> 3) : -1;
        store_stream(vis + p, make_int4(v[0], v[1], v[2], v[3]));
      }
      if constexpr (OM == 1) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (!((cov >> k) & 1u)) pix[p + k] = bgk;
      } else if constexpr (OM == 2) {
        if (cov == 0u) {
          for (int ch = 0; ch < C; ++ch)
            store_stream(fout + (size_t)ch * plane + p,
                         make_float4(bgc[ch], bgc[ch], bgc[ch], bgc[ch]));
        } else if (cov != 15u) {
          for (int ch = 0; ch < C; ++ch)
#pragma unroll
            for (int k = 0; k < 4; ++k)
              if (!((cov >> k) & 1u)) fout[(size_t)ch * plane + p + k] = bgc[ch];
        }
      }
    } else {
      const unsigned long long key = pix[p];
      const uint32_t zb = (uint32_t)(key >> 32);
      cov = zb < kDepthOne ? 1u : 0u;
      if (dep) dep[p] = cov ? __uint_as_float(zb) : 1.0f;
      if (vis) vis[p] = cov ? (int32_t)((uint32_t)key >> 3) : -1;
      if (!cov) {
        if constexpr (OM == 1) pix[p] = bgk;
        if constexpr (OM == 2)
          for (int ch = 0; ch < C; ++ch) fout[(size_t)ch * plane + p] = bgc[ch];
      }
    }
    return cov;
  };
  // Position of the lane's first covered pixel among the scan's, their number
  // in `sum`.
  auto place = [&](uint32_t cov, uint32_t& sum) -> uint32_t {
    uint32_t at = 0;
    sum = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k >= step) break;
      const uint64_t m = __ballot((cov >> k) & 1u);
      at += (uint32_t)__popcll(m & below);
      sum += (uint32_t)__popcll(m);
    }
    return at;
  };
  auto push = [&](uint16_t* q, uint32_t cov, int p0) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if ((cov >> k) & 1u) *q++ = (uint16_t)(p0 + lane * step + k);
  };
  // Shades the pixels q[0 .. take) (take <= 64).
  uint8_t* heads = reinterpret_cast<uint8_t*>(tab) - 64 * waves + 64 * wave;
  auto shade_batch = [&](const uint16_t* q, uint32_t take) {
    const int p = q[min((uint32_t)lane, take - 1u)];
    const uint32_t rank = (uint32_t)pix[p];
    float col[4];
    if constexpr (SMOOTH) {
      int y = (int)((float)p * inv_w);
      int x = p - y * W;
      if (x < 0) {
        --y;
        x += W;
      } else if (x >= W) {
        ++y;
        x -= W;
      }
      band_shade_smooth(D, F, lt, t.s, VP, nodes, nn, tab, lane, take, rank >> 3,
                        (int)(rank & 7u), x, t.j1 - y, heads, col);
    } else {
      band_shade_flat(D, lt, t.s, nodes, nn, tab, lane, take, rank >> 3, col);
    }
    if ((uint32_t)lane < take) {
      if constexpr (OM == 0) {
        pix[p] = pack_rgba8(col);
      } else if constexpr (OM == 1) {
        pix[p] = (unsigned long long)(bf16_rne(col[0]) | (bf16_rne(col[1]) << 16)) |
                 ((unsigned long long)(bf16_rne(col[2]) | (bf16_rne(col[3]) << 16)) << 32);
      } else {
#pragma unroll
        for (int ch = 0; ch < 4; ++ch)
          if (ch < C) fout[(size_t)ch * plane + p] = col[ch];
      }
    }
    wave_fence();
  };
  if constexpr (SMOOTH) {
    // one queue for the workgroup (in the space of the vertex tables and
    // triangle queues), so that only one batch per block of pixels is not
    // full; a block is what the queue holds
    uint16_t* pq = reinterpret_cast<uint16_t*>(tables);
    const int hold = (waves * (12 * F.verts + kBandTris - 64) / 2) & ~255;
    for (int b0 = 0; b0 < npx; b0 += hold) {
      const int bend = min(npx, b0 + hold);
      for (int p0 = b0 + wave * 64 * step; p0 < bend; p0 += block * step) {
        uint32_t sum;
        const uint32_t cov = scan(p0, bend), at = place(cov, sum);
        if (sum) {
          uint32_t first = 0;
          if (lane == 0) first = atomicAdd(&covered_n, sum);
          first = (uint32_t)__builtin_amdgcn_readfirstlane((int)first);
          push(pq + first + at, cov, p0);
        }
      }
      __syncthreads();
      const uint32_t total = (uint32_t)__builtin_amdgcn_readfirstlane((int)covered_n);
      for (uint32_t k0 = (uint32_t)wave * 64u; k0 < total; k0 += (uint32_t)block)
        shade_batch(pq + k0, min(total - k0, 64u));
      __syncthreads();
      if (bend < npx) {  // the next block starts with an empty queue
        if (tid == 0) covered_n = 0u;
        __syncthreads();
      }
    }
  } else {
    // a queue per wave: flat shading is cheap enough that partial batches
    // cost less than two more barriers
    uint16_t* pq = reinterpret_cast<uint16_t*>(vxy);
    uint32_t pend = 0;
    for (int p0 = wave * 64 * step; p0 < npx || pend > 0u;) {
      while (p0 < npx && pend < 64u) {  // at most 63 + 256 pixels are queued
        uint32_t sum;
        const uint32_t cov = scan(p0, npx), at = place(cov, sum);
        push(pq + pend + at, cov, p0);
        pend += sum;
        p0 += block * step;
      }
      wave_fence();
      uint32_t done = 0;
      while (done + 64u <= pend || (p0 >= npx && done < pend)) {
        const uint32_t take = min(pend - done, 64u);
        shade_batch(pq + done, take);
        done += take;
      }
      const uint16_t v = done + (uint32_t)lane < pend ? pq[done + lane] : (uint16_t)0;
      wave_fence();
      if (done + (uint32_t)lane < pend) pq[lane] = v;
      pend -= done;
      wave_fence();
    }
    __syncthreads();
  }
  if constexpr (OM == 2) return;
  unsigned char* cout = reinterpret_cast<unsigned char*>(O.color) +
                        ((size_t)t.s * C * plane + pix0) * (OM == 0 ? 1 : 2);
  // colour of pixel p as its plane's bytes; an uncovered pixel of a uint8
  // frame still holds its key
  auto pixel = [&](unsigned long long v) {
    if constexpr (OM == 0)
      return (uint32_t)(v >> 32) == kDepthOne ? (uint32_t)bgk : (uint32_t)v;
    else
      return v;
  };
  if (F.vec) {
    // four pixels of every channel from one read of their keys
    for (int p = tid * 4; p < npx; p += block * 4) {
      const ulonglong2 ka = *reinterpret_cast<const ulonglong2*>(pix + p);
      const ulonglong2 kb = *reinterpret_cast<const ulonglong2*>(pix + p + 2);
      const auto v0 = pixel(ka.x), v1 = pixel(ka.y), v2 = pixel(kb.x), v3 = pixel(kb.y);
      unsigned char* dst = cout + (size_t)p * (OM == 0 ? 1 : 2);
#pragma unroll 1
      for (int ch = 0; ch < C; ++ch) {
        if constexpr (OM == 0) {
          store_stream(dst + (size_t)ch * plane,
                       band_gather((uint32_t)v0, (uint32_t)v1, (uint32_t)v2, (uint32_t)v3, ch));
        } else {
          const int sh = 16 * ch;
          store_stream(dst + (size_t)ch * plane * 2,
                       make_uint2(((uint32_t)(v0 >> sh) & 0xffffu) | ((uint32_t)(v1 >> sh) << 16),
                                  ((uint32_t)(v2 >> sh) & 0xffffu) | ((uint32_t)(v3 >> sh) << 16)));
        }
      }
    }
    return;
  }
  // whole dwords of each channel plane: dword k of the plane's aligned range
  // starts at pixel k * PER - mis
  constexpr int PER = OM == 0 ? 4 : 2;
  constexpr size_t ES = OM == 0 ? 1 : 2;
  for (int ch = 0; ch < C; ++ch) {
    unsigned char* dst = cout + (size_t)ch * plane * ES;
    const int mis = (int)(((uintptr_t)dst & 3u) / ES);
    for (int k = tid; k * PER - mis < npx; k += block) {
      const int p = k * PER - mis;
      if (p >= 0 && p + PER <= npx) {
        uint32_t v;
        if constexpr (OM == 0) {
          v = band_gather(pixel(pix[p]), pixel(pix[p + 1]), pixel(pix[p + 2]), pixel(pix[p + 3]),
                          ch);
        } else {
          v = ((uint32_t)(pix[p] >> (16 * ch)) & 0xffffu) |
              ((uint32_t)(pix[p + 1] >> (16 * ch)) << 16);
        }
        store_stream(dst + (size_t)p * ES, v);
      } else {
#pragma unroll
        for (int b = 0; b < PER; ++b) {
          if (p + b < 0 || p + b >= npx) continue;
          if constexpr (OM == 0)
            dst[p + b] = (uint8_t)(pixel(pix[p + b]) >> (8 * ch));
          else
            reinterpret_cast<uint16_t*>(dst)[p + b] = (uint16_t)(pix[p + b] >> (16 * ch));
        }
      }
    }
  }
}

// --- host side ----------------------------------------------------------------

struct BandPlan {
  BandFrame F;
  size_t lds;
};

// Whether the scenes are few and each is much work.  A scene has at most kMaxBands
// workgroups, which each transform all its vertices, where the tile path spreads
// the scene's setup over the chip.  Which path draws sooner then depends on what is
// left after setup, which the host does not know: tile path's time over the band
// path's for objects of usual size / smaller than a pixel, frames of 32 x 32 to 160 x
// 160 (geometric means, boxes, UV spheres and cylinders):
//   vertices of a scene  1 scene      4            8            16           32
//   10 to 15 thousand    1.51 / 1.13  1.86 / 1.23  2.22 / 1.34  2.99 / 1.54  4.10 / 1.91
//   30 to 60             1.15 / 0.52  1.48 / 0.65  1.86 / 0.80  2.58 / 1.08  2.92 / 1.34
//   60 to 150            1.04 / 0.28  1.42 / 0.41  1.61 / 0.50  1.97 / 0.66  2.41 / 0.87
//   150 to 400           0.96 / 0.15  1.17 / 0.23  1.33 / 0.30  1.75 / 0.46  2.47 / 0.74
//   400 to 2000          1.07 / 0.10  1.23 / 0.18  1.47 / 0.29  1.92 / 0.49  2.57 / 0.82
// The line is where the mean over both is about one.  From 128 scenes on it is 1.8
// to 2.3, the lowest 0.74 (1024 scenes of 160 x 160 with 500 boxes below a pixel).
bool few_large_scenes(const pbr_scene_desc* D, const pbr_render_opts* opts, int64_t cus) {
  const int64_t n = D->num_scenes;
  if (n < 1 || 16 * n > cus) return false;
  double verts = 0.0;
  bool counts = false;
  for (int j = 0; j < D->num_nodes; ++j) {
    const pbr_node& nd = D->nodes[j];
    const pbr_mesh& me = D->meshes[nd.mesh];
    if (me.num_triangles > 0) verts += (double)nd.instances_per_scene * me.num_vertices;
    counts = counts || nd.counts;
  }
  // of a batch with instance counts the slot budget tells the mean scene's share
  const double most = (double)n * (double)max_slots(D);
  if (counts && opts && opts->slot_budget > 0 && (double)opts->slot_budget < most)
    verts *= (double)opts->slot_budget / most;
  return verts > 24576.0 + 6144.0 * (double)n;
}

// Whether the band path draws the batch, and its launch shape: default tile
// options (a tile size or bin capacity asks for the tile path), meshes that the
// wave tables hold, scenes whose setup its workgroups share out well, and frames of
// at most kMaxBands bands and kBandTable triangles.  Tile path's time over the band
// path's at three and four bands (160 x 160 and 176 x 176), 300 to 1024 scenes: 1.2
// to 2.9 for objects of usual size, 0.74 to 2.5 for objects smaller than a pixel.
// The two limits bound what was tested, they are no crossing: with both raised,
// five to fourteen bands (200 x 200 to 320 x 320) gave 1.04 to 4.2 and 0.62 to 2.4,
// and three to eight nodes with a sphere of 224 triangles each 1.3 to 4.5.
bool bands_plan(const pbr_scene_desc* D, const pbr_render_opts* opts, BandPlan& P) {
  if (opts && (opts->tile_size > 0 || opts->bin_capacity > 0)) return false;
  const int64_t cus = device_cus();
  if (few_large_scenes(D, opts, cus)) return false;
  memset(&P, 0, sizeof(P));
  BandFrame& F = P.F;
  F.W = D->width;
  F.H = D->height;
  int verts = 0, ntab = 0;
  for (int j = 0; j < D->num_nodes; ++j) {
    const pbr_mesh& me = D->meshes[D->nodes[j].mesh];
    F.node[j].group = 1;
    if (D->nodes[j].instances_per_scene == 0 || me.num_triangles == 0) continue;
    if (me.num_vertices < 1 || me.num_vertices > kBandVerts || me.num_triangles > kBandTris)
      return false;
    // shading finds a slot's instance by pbr_slot::split
    if (D->nodes[j].instances_per_scene > (int32_t)pbr_slot::kMaxInstances) return false;
    verts = std::max(verts, me.num_vertices);
    ntab = std::max(ntab, me.index_offset + me.num_triangles);
  }
  verts = (std::max(verts, 120) + 1) & ~1;  // tables and keys stay 16-byte aligned
  for (int j = 0; j < D->num_nodes; ++j) {
    const pbr_mesh& me = D->meshes[D->nodes[j].mesh];
    if (D->nodes[j].instances_per_scene == 0 || me.num_triangles == 0) continue;
    const int g = std::min(std::min(verts / me.num_vertices, kBandTris / me.num_triangles),
                           D->nodes[j].instances_per_scene);
    F.node[j].group = (uint32_t)std::max(1, g);
    F.node[j].inv_nv = (uint32_t)((65536 + me.num_vertices - 1) / me.num_vertices);
    F.node[j].inv_nt = (uint32_t)((65536 + me.num_triangles - 1) / me.num_triangles);
  }
  F.verts = verts;
  if (ntab > kBandTable) return false;
  F.ntab = ntab;
  const size_t stat = sizeof(NodeLds) * PBR_MAX_NODES + 4 * kClipQueue + 64;
  const auto rest = [&](int waves) {
    return (size_t)waves * ((size_t)verts * 12 + kBandTris) + 4 * (size_t)ntab;
  };
  const auto split = [&](int waves, int most, int bands) {
    F.waves = waves;
    F.bands = std::max((D->height + most - 1) / most, bands);
    F.th = (D->height + F.bands - 1) / F.bands;
    F.bands = (D->height + F.th - 1) / F.th;
    P.lds = (size_t)8 * ((F.th * F.W + 1) & ~1) + rest(waves);
  };
  const int px = std::min((int)((kBandLds - stat - rest(kBandWaves)) / 8), kBandPixels);
  if (D->width > px) return false;
  split(kBandWaves, px / D->width, 1);
  if (F.bands > kMaxBands) return false;
  // A batch that leaves CUs without a workgroup runs workgroups of twice the
  // waves and, while CUs are left, more bands.  Kernel time in us (8 waves /
  // 16 / 16 and bands): 64 scenes of 84 x 84 with up to 256 instances 99 / 68 /
  // 50, of 128 x 128 with 64 boxes 26 / 26 / 18, of 64 x 64 steering 50 / 47 /
  // 45; 512 steering scenes in one workgroup per CU at a time 96, not 73.
  const int64_t n = D->num_scenes;
  if (n * F.bands <= cus) {
    const int wide = (int)((2 * kBandLds - stat - rest(kWideWaves)) / 8);
    int bands = 1;
    while (bands < kMaxBands && 2 * n * bands <= cus && D->height / bands >= 16) bands *= 2;
    split(kWideWaves, std::min(wide, 2 * kBandPixels) / D->width, bands);
  }
  return true;
}

template <bool SMOOTH, int OM>
hipError_t launch_bands_t(const pbr_scene_desc* D, const pbr_frame_out* O, const BandPlan& P,
                          const uint32_t* scene_off, const uint32_t* order, uint32_t* hdr,
                          const Light& lt, float4 bg, uint32_t grid, hipStream_t st) {
  auto k = bands_kernel<SMOOTH, OM>;
  if (P.lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(
        (const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)P.lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k, dim3(grid), dim3(P.F.waves * 64), P.lds, st, *D, *O, P.F, scene_off,
                     order, hdr, lt, bg);
  return hipGetLastError();
}

}  // namespace

namespace pbr_host {

bool bands_supported(const pbr_scene_desc* D, const pbr_render_opts* opts) {
  BandPlan P;
  return bands_plan(D, opts, P);
}

int launch_bands(const pbr_scene_desc* D, const pbr_frame_out* O, const pbr_render_opts* opts,
                 uint32_t max_slots, uint32_t budget, bool uniform, const uint32_t* scene_off,
                 const uint32_t* order, uint32_t* hdr, hipStream_t st) {
  BandPlan P;
  if (!bands_plan(D, opts, P)) return fail(PBR_ERR_UNSUPPORTED, "band path cannot draw this batch");
  BandFrame& F = P.F;
  F.guard = 65536.0f / (float)(D->width > D->height ? D->width : D->height);
  F.max_slots = max_slots;
  F.budget = budget;
  F.uniform = uniform ? 1 : 0;
  // every channel plane, depth and id row of a band starts on a multiple of
  // four pixels from an aligned base, and the band is whole groups of four
  const uintptr_t align = O->dtype == PBR_DTYPE_U8 ? 3 : (O->dtype == PBR_DTYPE_BF16 ? 7 : 15);
  F.vec = (D->width * D->height) % 4 == 0 && (F.th * D->width) % 4 == 0 &&
          !((uintptr_t)O->color & align) && !((uintptr_t)O->depth & 15) &&
          !((uintptr_t)O->vis & 15);
  const uint64_t items = (uint64_t)D->num_scenes * (uint64_t)F.bands;
  if (items >= 0x7fffffffull) return fail(PBR_ERR_INVALID, "too many bands");
  const Light lt = host_light(D);
  const float4 bg = make_float4(D->background[0], D->background[1], D->background[2],
                                D->background[3]);
  const uint32_t grid = (uint32_t)items;
  hipError_t e;
  const bool smooth = any_smooth(D);
  switch (O->dtype) {
    case PBR_DTYPE_U8:
      e = smooth ? launch_bands_t<true, 0>(D, O, P, scene_off, order, hdr, lt, bg, grid, st)
                 : launch_bands_t<false, 0>(D, O, P, scene_off, order, hdr, lt, bg, grid, st);
      break;
    case PBR_DTYPE_BF16:
      e = smooth ? launch_bands_t<true, 1>(D, O, P, scene_off, order, hdr, lt, bg, grid, st)
                 : launch_bands_t<false, 1>(D, O, P, scene_off, order, hdr, lt, bg, grid, st);
      break;
    default:
      e = smooth ? launch_bands_t<true, 2>(D, O, P, scene_off, order, hdr, lt, bg, grid, st)
                 : launch_bands_t<false, 2>(D, O, P, scene_off, order, hdr, lt, bg, grid, st);
  }
  if (e != hipSuccess) return fail(PBR_ERR_LAUNCH, "band launch failed: %s", hipGetErrorString(e));
  return PBR_OK;
}

}  // namespace pbr_host
