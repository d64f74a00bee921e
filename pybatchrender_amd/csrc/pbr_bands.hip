// pbr_bands.hip - the band path: one workgroup draws one band of full rows of
// one scene from the scene's instances, with no records in device memory.
//
//   setup + raster  the scene's instances are dealt to the eight waves in
//                   chunks (as many instances of one node as the wave's vertex
//                   table holds).  A wave transforms and snaps the chunk's
//                   vertices once into its LDS table, drops the chunk if all
//                   of them lie outside one plane or off the band, tests each
//                   triangle on three table entries, queues the live ones and
//                   sets up 64 of them at a time.  A set-up triangle is
//                   rasterised at once - a small one by its lane, a large one
//                   by the whole wave - into the band's 64-bit pixel keys in
//                   LDS: atomicMin of depth bits << 32 | slot << 3 |
//                   sub-triangle, the winner the in-order strict-less depth
//                   test picks whatever the order of the fragments.
//   resolve         covered pixels are queued per wave and shaded 64 at a
//                   time from the winner's instance and vertices, which are
//                   transformed again (fewer pixels are covered than triangles
//                   are set up, so keeping shading data per triangle costs
//                   more than making it per pixel); colours narrower than
//                   their key replace it in LDS and leave as whole dwords.
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

using namespace pbr_host;

namespace {

constexpr int kBandBlock = 512;
constexpr int kBandWaves = kBandBlock / 64;
constexpr int kBandVerts = 136;   // vertices a wave's table holds at most
constexpr int kBandTris = 256;    // triangles of one mesh (8-bit queue entries)
constexpr int kBandTable = 512;   // triangles of the LDS index table at most
constexpr int kMaxBands = 4;      // bands per scene at most: each repeats the vertex work
constexpr int kBandPixels = 8192;
constexpr int kBandLds = 80 * 1024;  // half a CU's LDS: two workgroups share a CU
constexpr int kSmallPixels = 48;  // box pixels one lane rasterises alone
constexpr uint32_t kDepthOne = 0x3f800000u;

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
  int verts;           // entries of a wave's vertex table
  int ntab;            // triangles in the LDS index table (0: read from memory)
  BandNode node[PBR_MAX_NODES];
};

// Node facts a workgroup keeps in LDS.
struct NodeLds {
  const float* trans;
  const float* cols;
  uint32_t base, chunk0;  // first slot and first chunk of the node in this scene
  uint32_t cnt;           // active instances
  int32_t ntri, voff, ioff, ips;
  uint32_t flags;         // bit 0: shared, bit 1: flat
};

// Vertex table entry: X << 6 | outcode, Y << 6 | inside all planes << 1 |
// snapped.  |X|, |Y| <= 2^24 (snap_vertex), so both shifts fit 32 bits.
constexpr int kInAll = 2, kSnapped = 1;

typedef const __attribute__((address_space(4))) float const_float;
typedef const __attribute__((address_space(1))) float global_cfloat;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) f32x4 global_cfloat4;

// Sixteen floats at a wave-uniform address, by scalar loads.
__device__ __forceinline__ void load_mat4_uniform(const float* src, float M[16]) {
  const_float* p = (const_float*)(uintptr_t)src;
#pragma unroll
  for (int q = 0; q < 16; ++q) M[q] = p[q];
}

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

struct BandCtx {
  int s, W;
  int j0, j1;  // GL rows of the band; LDS row 0 is j1
};

__device__ __forceinline__ void band_fragment(unsigned long long* pix, const BandCtx& t, int i,
                                              int j, float z, uint32_t rank) {
  const unsigned long long key = ((unsigned long long)__float_as_uint(z) << 32) | rank;
  unsigned long long* q = pix + (t.j1 - j) * t.W + i;
  // keys only decrease, so a read that is already <= the key proves the
  // atomic would change nothing
  if (key < *q) atomicMin(q, key);
}

// Biased edge values e_k = A_k Px + B_k Py + C_k >= 0 <=> inside, at pixel
// (i, j); every term is an integer below 2^53.
struct BandEdges {
  double A[3], B[3], C[3];
};

__device__ __forceinline__ void band_edges(const int32_t X[3], const int32_t Y[3], uint32_t bias,
                                           BandEdges& E) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int a = (k + 1) % 3, b = (k + 2) % 3;
    E.A[k] = (double)(Y[a] - Y[b]);
    E.B[k] = (double)(X[b] - X[a]);
    E.C[k] = -fma(E.A[k], (double)X[a], E.B[k] * (double)Y[a]) - (double)((bias >> k) & 1u);
  }
}

// One lane, the whole box.
__device__ __forceinline__ void band_raster_lane(unsigned long long* pix, const BandCtx& t,
                                                 const FixTri& T, uint32_t rank) {
  BandEdges E;
  band_edges(T.X, T.Y, T.bias, E);
  const double px0 = (double)(256 * T.i0 + 128);
  for (int j = T.j0; j <= T.j1; ++j) {
    const double py = (double)(256 * j + 128);
    double e0 = fma(E.A[0], px0, fma(E.B[0], py, E.C[0]));
    double e1 = fma(E.A[1], px0, fma(E.B[1], py, E.C[1]));
    double e2 = fma(E.A[2], px0, fma(E.B[2], py, E.C[2]));
    const float tz = fmaf(T.zy, (float)j + 0.5f, T.zc);
    for (int i = T.i0; i <= T.i1; ++i) {
      if (e0 >= 0.0 && e1 >= 0.0 && e2 >= 0.0)
        band_fragment(pix, t, i, j, clamp_depth(fmaf(T.zx, (float)i + 0.5f, tz)), rank);
      e0 += E.A[0] * 256.0;
      e1 += E.A[1] * 256.0;
      e2 += E.A[2] * 256.0;
    }
  }
}

// The whole wave, in blocks of 8 x 8 pixels.  Every argument is uniform.
__device__ __forceinline__ void band_raster_wave(unsigned long long* pix, const BandCtx& t,
                                                 int lane, const FixTri& T, uint32_t rank) {
  BandEdges E;
  band_edges(T.X, T.Y, T.bias, E);
  const int li = lane & 7, lj = lane >> 3;
  for (int jb = T.j0; jb <= T.j1; jb += 8) {
    const int j = jb + lj;
    const double py = (double)(256 * j + 128);
    const double px = (double)(256 * (T.i0 + li) + 128);
    double e0 = fma(E.A[0], px, fma(E.B[0], py, E.C[0]));
    double e1 = fma(E.A[1], px, fma(E.B[1], py, E.C[1]));
    double e2 = fma(E.A[2], px, fma(E.B[2], py, E.C[2]));
    const float tz = fmaf(T.zy, (float)j + 0.5f, T.zc);
    for (int ib = T.i0; ib <= T.i1; ib += 8) {
      const int i = ib + li;
      if (i <= T.i1 && j <= T.j1 && e0 >= 0.0 && e1 >= 0.0 && e2 >= 0.0)
        band_fragment(pix, t, i, j, clamp_depth(fmaf(T.zx, (float)i + 0.5f, tz)), rank);
      e0 += E.A[0] * 2048.0;
      e1 += E.A[1] * 2048.0;
      e2 += E.A[2] * 2048.0;
    }
  }
}

__device__ __forceinline__ int rl(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ float rlf(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// Clip polygon of slot `local` of node j; only triangles that straddle a clip
// plane get here.
__device__ __noinline__ int band_clip(const pbr_scene_desc* D, float guard, int s, int j,
                                      uint32_t local, CVert* poly) {
  CVert cv[3];
  float rgba[4];
  bool flat;
  fetch_node_triangle(*D, s, j, local, cv, rgba, flat);
  poly[0] = cv[0];
  poly[1] = cv[1];
  poly[2] = cv[2];
  return clip_polygon(poly, guard);
}

__device__ __noinline__ bool band_clip_sub(const CVert* poly, int q, int W, int H, int j0, int j1,
                                           FixTri* T) {
  return setup_fixed(poly[0], poly[q + 1], poly[q + 2], W, H, j0, j1, *T);
}

// Smooth colour of sub-triangle q of a clipped slot at pixel centre (px, py).
__device__ __noinline__ void band_clipped_colour(const pbr_scene_desc* D, float guard, int s,
                                                 int j, uint32_t local, int q, const float* rgba,
                                                 Light lt, double px, double py, float* col) {
  CVert poly[kMaxPoly];
  const int n = band_clip(D, guard, s, j, local, poly);
  FixTri T;
  if (q + 2 >= n || !band_clip_sub(poly, q, D->width, D->height, 0, D->height - 1, &T)) return;
  double A[3], B[3], C[3];
  edges_from_fixed(T.X, T.Y, T.bias, A, B, C);
  const CVert* v[3] = {&poly[0], &poly[q + 1], &poly[q + 2]};
  float sh[kShadeFloats];
  for (int k = 0; k < 3; ++k) {
    for (int c = 0; c < 3; ++c) sh[3 * k + c] = v[k]->n[c];
    sh[9 + k] = T.invw[k];
  }
  for (int c = 0; c < 4; ++c) sh[12 + c] = rgba[c];
  shade_smooth(A, B, C, T.bias, sh, px, py, lt, col);
}

// Colour of the pixel whose winner is slot `slot`, sub-triangle q, of node j.
template <bool SMOOTH>
__device__ __forceinline__ void band_shade(const pbr_scene_desc& D, const BandFrame& F,
                                           const Light& lt, int s, const float VP[16],
                                           const NodeLds* nodes, int nn, const uint32_t* tab,
                                           uint32_t slot, int q, int x, int j, float col[4]) {
  int nj = 0;
  for (int k = 1; k < nn; ++k) nj = slot >= nodes[k].base ? k : nj;
  const NodeLds& nd = nodes[nj];
  const uint32_t local = slot - nd.base, nt = (uint32_t)nd.ntri;
  // local / nt from a float reciprocal: the quotient is below 2^24, so the
  // truncated product is off by at most one and one step corrects it
  uint32_t i = (uint32_t)((float)local * (1.0f / (float)nt));
  int32_t t = (int32_t)(local - i * nt);
  if (t < 0) {
    --i;
    t += (int32_t)nt;
  } else if (t >= (int32_t)nt) {
    ++i;
    t -= (int32_t)nt;
  }
  const size_t row = (nd.flags & 1u) ? (size_t)i : (size_t)s * (size_t)nd.ips + i;
  float M[16];
  load_mat4_global(nd.trans + row * 16, M);
  const f32x4 c4 = ((global_cfloat4*)(uintptr_t)nd.cols)[row];
  const float rgba[4] = {c4.x, c4.y, c4.z, c4.w};
  const uint32_t tri = F.ntab ? tab[nd.ioff + t] : pool_triangle(D, nd.ioff + t);
  float v[6];
  load_vertex(D.vertices, nd.voff + (int)(tri & 0xffu), v);
  if (!SMOOTH || (nd.flags & 2u)) {
    float nw[3], n[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const float a = M[r * 4 + 0] * v[3] + M[r * 4 + 1] * v[4];
      nw[r] = a + M[r * 4 + 2] * v[5];
    }
    normalize3(nw, n);
    shade(n, rgba, lt, col);
    return;
  }
  if constexpr (SMOOTH) {
    float v1[6], v2[6];
    load_vertex(D.vertices, nd.voff + (int)((tri >> 8) & 0xffu), v1);
    load_vertex(D.vertices, nd.voff + (int)(tri >> 16), v2);
    VertRec r[3];
    vertex_record(M, VP, v, F.W, F.H, F.guard, r[0]);
    vertex_record(M, VP, v1, F.W, F.H, F.guard, r[1]);
    vertex_record(M, VP, v2, F.W, F.H, F.guard, r[2]);
    if ((((r[0].bits & r[1].bits & r[2].bits) >> 1) & 0x3fu) != 0x3fu) {
      const double px = (double)(256 * x + 128), py = (double)(256 * j + 128);
      col[0] = col[1] = col[2] = col[3] = 0.0f;
      band_clipped_colour(kernarg_scene(), F.guard, s, nj, local, q, rgba, lt, px, py, col);
      return;
    }
    // e_k = A_k Px + B_k Py + C_k without the fill-rule bias: edge k runs from
    // vertex k + 1 to vertex k + 2, and every difference and product is an
    // exact integer in double
    const int32_t X[3] = {r[0].X, r[1].X, r[2].X}, Y[3] = {r[0].Y, r[1].Y, r[2].Y};
    const int32_t cx = 256 * x + 128, cy = 256 * j + 128;
    float bw[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int a = (k + 1) % 3, b = (k + 2) % 3;
      const double e = fma((double)(Y[a] - Y[b]), (double)(cx - X[a]),
                           (double)(X[b] - X[a]) * (double)(cy - Y[a]));
      bw[k] = (float)e * r[k].invw;
    }
    float n[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float a = bw[0] * r[0].n[c] + bw[1] * r[1].n[c];
      n[c] = a + bw[2] * r[2].n[c];
    }
    shade(n, rgba, lt, col);
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
// [th][W], per wave a vertex table (int2 [verts], float depth [verts]) and a
// queue of 128 bytes, then the index table.  D stays the first parameter: the
// out-of-line clipper reads it through the kernarg segment (kernarg_scene).
template <bool SMOOTH, int OM>
__global__ __launch_bounds__(kBandBlock)
__attribute__((amdgpu_waves_per_eu(4))) void bands_kernel(pbr_scene_desc D, pbr_frame_out O,
                                                          BandFrame F, const uint32_t* scene_off,
                                                          uint32_t* hdr, Light lt, float4 bg) {
  extern __shared__ unsigned long long pix[];
  __shared__ NodeLds nodes[PBR_MAX_NODES];
  __shared__ uint32_t next_chunk, total_chunks;
  const int tid = (int)threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int W = F.W, H = F.H, nn = D.num_nodes;
  BandCtx t;
  t.s = (int)(blockIdx.x / (uint32_t)F.bands);
  const int band = (int)(blockIdx.x - (uint32_t)t.s * (uint32_t)F.bands);
  const int yo0 = band * F.th, rows = min(F.th, H - yo0);
  t.W = W;
  t.j1 = H - 1 - yo0;
  t.j0 = t.j1 - (rows - 1);
  const int npx = rows * W;
  int2* vxy = reinterpret_cast<int2*>(pix + F.th * W) + wave * F.verts;
  float* vd = reinterpret_cast<float*>(reinterpret_cast<int2*>(pix + F.th * W) +
                                       kBandWaves * F.verts) + wave * F.verts;
  uint8_t* qu = reinterpret_cast<uint8_t*>(reinterpret_cast<int2*>(pix + F.th * W) +
                                           kBandWaves * F.verts) +
                sizeof(float) * kBandWaves * F.verts + wave * 128;
  uint32_t* tab = reinterpret_cast<uint32_t*>(
      reinterpret_cast<uint8_t*>(reinterpret_cast<int2*>(pix + F.th * W) + kBandWaves * F.verts) +
      sizeof(float) * kBandWaves * F.verts + kBandWaves * 128);

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
  for (int p = tid; p < npx; p += kBandBlock) pix[p] = (unsigned long long)kDepthOne << 32;
  for (int q = tid; q < F.ntab; q += kBandBlock) tab[q] = pool_triangle(D, q);
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
      e.voff = me.vertex_offset;
      e.ioff = me.index_offset;
      e.ips = nd.instances_per_scene;
      e.flags = (nd.shared ? 1u : 0u) | (nd.flat ? 2u : 0u);
      nodes[lane] = e;
    }
    if (lane == 63) {
      next_chunk = 0u;
      total_chunks = ic;
    }
  }
  __syncthreads();

  float VP[16];
  load_mat4_uniform(D.view_proj + (size_t)t.s * 16, VP);

  // --- setup and raster --------------------------------------------------------
  const uint32_t chunks = __builtin_amdgcn_readfirstlane((int)total_chunks);
  // pixel-centre limits in 1/256 pixel: a chunk wholly below / above / left /
  // right of them touches no pixel centre of the band
  const int ylo = 256 * t.j0 + 128, yhi = 256 * t.j1 + 128, xhi = 256 * (W - 1) + 128;
  for (;;) {
    uint32_t c = 0;
    if (lane == 0) c = atomicAdd(&next_chunk, 1u);
    c = (uint32_t)__builtin_amdgcn_readfirstlane((int)c);
    if (c >= chunks) break;
    int j = 0;
    for (int k = 1; k < nn; ++k)
      j = c >= (uint32_t)__builtin_amdgcn_readfirstlane((int)nodes[k].chunk0) ? k : j;
    const pbr_node& nd = D.nodes[j];
    const pbr_mesh& me = D.meshes[nd.mesh];
    const BandNode bn = F.node[j];
    const uint32_t cnt = (uint32_t)__builtin_amdgcn_readfirstlane((int)nodes[j].cnt);
    const uint32_t base = (uint32_t)__builtin_amdgcn_readfirstlane((int)nodes[j].base);
    const uint32_t i0 = (c - (uint32_t)__builtin_amdgcn_readfirstlane((int)nodes[j].chunk0)) *
                        bn.group;
    const uint32_t g = min(bn.group, cnt - i0);
    const uint32_t nt = (uint32_t)me.num_triangles, nv = (uint32_t)me.num_vertices;
    const uint32_t slot0 = base + i0 * nt;
    if (slot0 >= ndraw) continue;
    const uint32_t n = min(g * nt, ndraw - slot0);
    const size_t row0 = nd.shared ? (size_t)i0 : (size_t)t.s * (size_t)nd.instances_per_scene + i0;

    // vertices of the chunk into the wave's table; `out` gathers what all of
    // them lie outside of (bits 0-5 clip planes, 6-9 the band's sides)
    uint32_t out = 0x3ffu;
    for (uint32_t v = (uint32_t)lane; v < g * nv; v += 64u) {
      const uint32_t di = (v * bn.inv_nv) >> 16, k = v - di * nv;
      float M[16], vv[6];
      load_mat4_global(nd.transforms + (row0 + di) * 16, M);
      load_vertex(D.vertices, me.vertex_offset + (int)k, vv);
      VertRec r;
      vertex_record(M, VP, vv, W, H, F.guard, r);
      const uint32_t oc = (r.bits >> 7) & 0x3fu;
      const bool in = ((r.bits >> 1) & 0x3fu) == 0x3fu;
      vxy[v] = make_int2((int)(((uint32_t)r.X << 6) | oc),
                         (int)(((uint32_t)r.Y << 6) | (in ? (uint32_t)kInAll : 0u) |
                               (r.bits & 1u)));
      vd[v] = r.d;
      uint32_t side = 0;
      if (in && (r.bits & 1u))
        side = (r.Y < ylo ? 64u : 0u) | (r.Y > yhi ? 128u : 0u) | (r.X < 128 ? 256u : 0u) |
               (r.X > xhi ? 512u : 0u);
      out &= oc | side;
    }
    bool gone = false;
#pragma unroll
    for (int b = 0; b < 10; ++b) gone = gone || __ballot(!((out >> b) & 1u)) == 0ull;
    if (gone) continue;
    wave_fence();

    // triangles: test, queue, set up 64 queued ones at a time, rasterise.
    // Sub-triangles of clipped ones take the place of a set-up round.
    uint32_t pend = 0, q0 = 0;
    int nsub = 0;  // vertices of this lane's clip polygon
    int sub = 0, subs = 0;  // sub-triangle rounds done and due
    uint32_t clip_slot = 0;
    CVert poly[kMaxPoly];
    for (;;) {
      FixTri T;
      bool has = false;
      uint32_t rank = 0;
      if (sub < subs) {
        const int q = sub++;
        if (q + 2 < nsub) {
          FixTri S;
          has = band_clip_sub(poly, q, W, H, t.j0, t.j1, &S);
          T = S;
          rank = (clip_slot << 3) | (uint32_t)q;
        }
      } else if (pend >= 64u || (q0 >= n && pend > 0u)) {
        const uint32_t take = min(pend, 64u);
        if ((uint32_t)lane < take) {
          const uint32_t u = qu[lane];
          const uint32_t di = (u * bn.inv_nt) >> 16, tt = u - di * nt;
          const uint32_t tri = F.ntab ? tab[me.index_offset + (int)tt]
                                      : pool_triangle(D, me.index_offset + (int)tt);
          const uint32_t vb = di * nv;
          const uint32_t ia = vb + (tri & 0xffu), ib = vb + ((tri >> 8) & 0xffu),
                         ic = vb + (tri >> 16);
          const int2 a = vxy[ia], b = vxy[ib], cc = vxy[ic];
          const SnapVert sa = {a.x >> 6, a.y >> 6, vd[ia], 0.0f, true};
          const SnapVert sb = {b.x >> 6, b.y >> 6, vd[ib], 0.0f, true};
          const SnapVert sc = {cc.x >> 6, cc.y >> 6, vd[ic], 0.0f, true};
          has = setup_snapped(sa, sb, sc, W, H, t.j0, t.j1, T);
          rank = (slot0 + u) << 3;
        }
        uint8_t rest = 0;
        if ((uint32_t)lane + 64u < pend) rest = qu[lane + 64];
        wave_fence();
        if ((uint32_t)lane + 64u < pend) qu[lane] = rest;
        pend -= take;
        wave_fence();
      } else if (q0 < n) {
        const uint32_t u = q0 + (uint32_t)lane;
        bool live = false, clip = false;
        if (u < n) {
          const uint32_t di = (u * bn.inv_nt) >> 16, tt = u - di * nt;
          const uint32_t tri = F.ntab ? tab[me.index_offset + (int)tt]
                                      : pool_triangle(D, me.index_offset + (int)tt);
          const uint32_t vb = di * nv;
          const int2 a = vxy[vb + (tri & 0xffu)], b = vxy[vb + ((tri >> 8) & 0xffu)],
                     cc = vxy[vb + (tri >> 16)];
          const int fl = a.y & b.y & cc.y;
          if ((a.x & b.x & cc.x & 0x3f) == 0) {
            if (!(fl & kInAll)) {
              clip = true;
            } else if (fl & kSnapped) {
              const int32_t X0 = a.x >> 6, X1 = b.x >> 6, X2 = cc.x >> 6;
              const int32_t Y0 = a.y >> 6, Y1 = b.y >> 6, Y2 = cc.y >> 6;
              const double area = (double)(X1 - X0) * (double)(Y2 - Y0) -
                                  (double)(X2 - X0) * (double)(Y1 - Y0);
              const int32_t xmin = min(X0, min(X1, X2)), xmax = max(X0, max(X1, X2));
              const int32_t ymin = min(Y0, min(Y1, Y2)), ymax = max(Y0, max(Y1, Y2));
              const int32_t a0 = max((xmin + 127) >> 8, 0), a1 = min((xmax - 128) >> 8, W - 1);
              const int32_t b0 = max((ymin + 127) >> 8, t.j0), b1 = min((ymax - 128) >> 8, t.j1);
              live = area > 0.0 && a0 <= a1 && b0 <= b1;
            }
          }
        }
        const uint64_t m = __ballot(live);
        if (live) qu[pend + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint8_t)u;
        pend += (uint32_t)__popcll(m);
        q0 += 64u;
        if (__ballot(clip)) {
          nsub = 0;
          if (clip) {
            clip_slot = slot0 + u;
            nsub = band_clip(kernarg_scene(), F.guard, t.s, j, clip_slot - base, poly);
          }
          sub = subs = 0;
          while (__ballot(subs + 2 < nsub)) ++subs;
        }
        wave_fence();
        continue;
      } else {
        break;
      }
      // rasterise the lanes' triangles
      const bool small = has && (T.i1 - T.i0 + 1) * (T.j1 - T.j0 + 1) <= kSmallPixels;
      if (small) band_raster_lane(pix, t, T, rank);
      for (uint64_t m = __ballot(has && !small); m; m &= m - 1ull) {
        const int l = __ffsll((unsigned long long)m) - 1;
        FixTri U;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          U.X[k] = rl(T.X[k], l);
          U.Y[k] = rl(T.Y[k], l);
        }
        U.zx = rlf(T.zx, l);
        U.zy = rlf(T.zy, l);
        U.zc = rlf(T.zc, l);
        U.i0 = rl(T.i0, l);
        U.i1 = rl(T.i1, l);
        U.j0 = rl(T.j0, l);
        U.j1 = rl(T.j1, l);
        U.bias = (uint32_t)rl((int)T.bias, l);
        band_raster_wave(pix, t, lane, U, (uint32_t)rl((int)rank, l));
      }
    }
    wave_fence();  // the next chunk rewrites the table
  }
  __syncthreads();

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
  uint16_t* pq = reinterpret_cast<uint16_t*>(vxy);  // covered pixels awaiting their shading
  uint32_t pend = 0;
  for (int p0 = wave * 64; p0 < npx || pend > 0u;) {
    if (p0 < npx && pend < 64u) {
      const int p = p0 + lane;
      bool covered = false;
      if (p < npx) {
        const unsigned long long key = pix[p];
        const uint32_t zb = (uint32_t)(key >> 32);
        covered = zb < kDepthOne;
        if (dep) dep[p] = covered ? __uint_as_float(zb) : 1.0f;
        if (vis) vis[p] = covered ? (int32_t)((uint32_t)key >> 3) : -1;
        if (!covered) {
          if constexpr (OM < 2) {
            pix[p] = bgk;
          } else {
            for (int ch = 0; ch < C; ++ch) fout[(size_t)ch * plane + p] = bgc[ch];
          }
        }
      }
      const uint64_t m = __ballot(covered);
      if (covered) pq[pend + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)p;
      pend += (uint32_t)__popcll(m);
      p0 += kBandBlock;
      wave_fence();
      continue;
    }
    const uint32_t take = min(pend, 64u);
    if ((uint32_t)lane < take) {
      const int p = pq[lane];
      const uint32_t rank = (uint32_t)pix[p];
      int y = (int)((float)p * (1.0f / (float)W));
      int x = p - y * W;
      if (x < 0) {
        --y;
        x += W;
      } else if (x >= W) {
        ++y;
        x -= W;
      }
      float col[4];
      band_shade<SMOOTH>(D, F, lt, t.s, VP, nodes, nn, tab, rank >> 3, (int)(rank & 7u), x,
                         t.j1 - y, col);
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
    uint16_t rest = 0;
    if ((uint32_t)lane + 64u < pend) rest = pq[lane + 64];
    wave_fence();
    if ((uint32_t)lane + 64u < pend) pq[lane] = rest;
    pend -= take;
    wave_fence();
  }
  if constexpr (OM == 2) return;
  __syncthreads();
  // the band's colours as whole dwords of each channel plane: dword k of the
  // plane's aligned range starts at pixel k * PER - mis
  constexpr int PER = OM == 0 ? 4 : 2;
  constexpr size_t ES = OM == 0 ? 1 : 2;
  unsigned char* cout = reinterpret_cast<unsigned char*>(O.color) +
                        ((size_t)t.s * C * plane + pix0) * ES;
  for (int ch = 0; ch < C; ++ch) {
    unsigned char* dst = cout + (size_t)ch * plane * ES;
    const int mis = (int)(((uintptr_t)dst & 3u) / ES);
    for (int k = tid; k * PER - mis < npx; k += kBandBlock) {
      const int p = k * PER - mis;
      if (p >= 0 && p + PER <= npx) {
        uint32_t v;
        if constexpr (OM == 0) {
          v = band_gather((uint32_t)pix[p], (uint32_t)pix[p + 1], (uint32_t)pix[p + 2],
                          (uint32_t)pix[p + 3], ch);
        } else {
          v = ((uint32_t)(pix[p] >> (16 * ch)) & 0xffffu) |
              ((uint32_t)(pix[p + 1] >> (16 * ch)) << 16);
        }
        *reinterpret_cast<uint32_t*>(dst + (size_t)p * ES) = v;
      } else {
#pragma unroll
        for (int b = 0; b < PER; ++b) {
          if (p + b < 0 || p + b >= npx) continue;
          if constexpr (OM == 0)
            dst[p + b] = (uint8_t)(pix[p + b] >> (8 * ch));
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

// Whether the band path draws the batch, and its launch shape: default tile
// options (a tile size or bin capacity asks for the tile path), meshes the
// wave tables hold, and few enough bands that repeating the scene's vertex
// work per band stays below what the tile path's records cost.
bool bands_plan(const pbr_scene_desc* D, const pbr_render_opts* opts, BandPlan& P) {
  if (opts && (opts->tile_size > 0 || opts->bin_capacity > 0)) return false;
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
    verts = std::max(verts, me.num_vertices);
    ntab = std::max(ntab, me.index_offset + me.num_triangles);
  }
  verts = std::max(verts, 120);
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
  F.ntab = ntab <= kBandTable ? ntab : 0;
  const size_t stat = sizeof(NodeLds) * PBR_MAX_NODES + 64;
  const size_t rest = (size_t)kBandWaves * ((size_t)verts * 12 + 128) + 4 * (size_t)F.ntab;
  const int fit = (int)((kBandLds - stat - rest) / 8);
  const int px = std::min(fit, kBandPixels);
  if (D->width > px) return false;
  const int most = px / D->width;
  F.bands = (D->height + most - 1) / most;
  if (F.bands > kMaxBands) return false;
  F.th = (D->height + F.bands - 1) / F.bands;
  F.bands = (D->height + F.th - 1) / F.th;
  P.lds = (size_t)8 * F.th * F.W + rest;
  return true;
}

template <bool SMOOTH, int OM>
hipError_t launch_bands_t(const pbr_scene_desc* D, const pbr_frame_out* O, const BandPlan& P,
                          const uint32_t* scene_off, uint32_t* hdr, const Light& lt, float4 bg,
                          uint32_t grid, hipStream_t st) {
  auto k = bands_kernel<SMOOTH, OM>;
  if (P.lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(
        (const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)P.lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k, dim3(grid), dim3(kBandBlock), P.lds, st, *D, *O, P.F, scene_off, hdr, lt,
                     bg);
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
                 uint32_t* hdr, hipStream_t st) {
  BandPlan P;
  if (!bands_plan(D, opts, P)) return fail(PBR_ERR_UNSUPPORTED, "band path cannot draw this batch");
  BandFrame& F = P.F;
  F.guard = 65536.0f / (float)(D->width > D->height ? D->width : D->height);
  F.max_slots = max_slots;
  F.budget = budget;
  F.uniform = uniform ? 1 : 0;
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
      e = smooth ? launch_bands_t<true, 0>(D, O, P, scene_off, hdr, lt, bg, grid, st)
                 : launch_bands_t<false, 0>(D, O, P, scene_off, hdr, lt, bg, grid, st);
      break;
    case PBR_DTYPE_BF16:
      e = smooth ? launch_bands_t<true, 1>(D, O, P, scene_off, hdr, lt, bg, grid, st)
                 : launch_bands_t<false, 1>(D, O, P, scene_off, hdr, lt, bg, grid, st);
      break;
    default:
      e = smooth ? launch_bands_t<true, 2>(D, O, P, scene_off, hdr, lt, bg, grid, st)
                 : launch_bands_t<false, 2>(D, O, P, scene_off, hdr, lt, bg, grid, st);
  }
  if (e != hipSuccess) return fail(PBR_ERR_LAUNCH, "band launch failed: %s", hipGetErrorString(e));
  return PBR_OK;
}

}  // namespace pbr_host
