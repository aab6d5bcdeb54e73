// Device helpers shared by the kernel files: wavefront synchronisation,
// counts of a captured pipeline, sign predicates, tet planes.
#pragma once
#include <hip/hip_runtime.h>

#include "rpd_device.h"
#include "rpd_capi.h"

namespace rpd {

constexpr uint32_t kEnd = 255;

__device__ __forceinline__ void wsync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ uint64_t ballot(bool p) {
  return __ballot(p);
}

__device__ __forceinline__ rpd_d4 ld4(const double4* p) {
  double4 v = *p;
  return rpd_d4{v.x, v.y, v.z, v.w};
}

// Counts of a captured pipeline (hipGraph): a launch is sized by its
// capacity and reads the count the previous kernels left on the device;
// without a device count the host's count is exact.
__device__ __forceinline__ int64_t dev_count(int64_t cap, const int64_t* d,
                                             int64_t sub = 0) {
  return d ? min(cap, *d - sub) : cap;
}
__device__ __forceinline__ int64_t dev_count32(int64_t cap, const int32_t* d,
                                               int64_t sub = 0) {
  return d ? min(cap, (int64_t)*d - sub) : cap;
}

// --------------------------------------------------------- predicates
// det4x4(p1.x, p2.x, p3.x, e.x, p1.y, ..., p1.w, p2.w, p3.w, e.w) in the
// reference's evaluation order (convex_cell.cu:458-459,
// common_cuda.h:195-213), with a semi-static filter: every monomial passes
// through at most 9 roundings, |err| <= gamma_9 * 24 * prod_r max_c |a_rc|,
// 24 * gamma_9 = 2.398e-14; 2.5e-14 covers the rounding of the bound.
// Products may fuse with the following sum: a fused monomial passes
// through fewer roundings, so the bound holds, and a decided sign is the
// exact one either way (undecided signs go to the exact predicate).
// The caller passes the bound eps, computed from row maxima that dominate
// the four columns': the clip kernel keeps, per cell, the largest |a|,
// |b|, |c|, |d| over all planes it has added, so each row's maximum over a
// vertex's three planes and the new plane e is at most max(cell maximum,
// |e|) -- one bound per clip step, no smaller than the per-vertex one.
// Returns +1 conflict, -1 no conflict, 0 undecided.
__device__ __forceinline__ int conflict_filtered_eps(const rpd_d4& p1,
                                                     const rpd_d4& p2,
                                                     const rpd_d4& p3,
                                                     const rpd_d4& e,
                                                     double eps) {
#pragma clang fp contract(fast)
  const double a11 = p1.x, a12 = p2.x, a13 = p3.x, a14 = e.x;
  const double a21 = p1.y, a22 = p2.y, a23 = p3.y, a24 = e.y;
  const double a31 = p1.z, a32 = p2.z, a33 = p3.z, a34 = e.z;
  const double a41 = p1.w, a42 = p2.w, a43 = p3.w, a44 = e.w;
  double m12 = a21 * a12 - a11 * a22;
  double m13 = a31 * a12 - a11 * a32;
  double m14 = a41 * a12 - a11 * a42;
  double m23 = a31 * a22 - a21 * a32;
  double m24 = a41 * a22 - a21 * a42;
  double m34 = a41 * a32 - a31 * a42;
  double m123 = m23 * a13 - m13 * a23 + m12 * a33;
  double m124 = m24 * a13 - m14 * a23 + m12 * a43;
  double m134 = m34 * a13 - m14 * a33 + m13 * a43;
  double m234 = m34 * a23 - m24 * a33 + m23 * a43;
  double det = m234 * a14 - m134 * a24 + m124 * a34 - m123 * a44;
  if (det > eps) return 1;
  if (det < -eps) return -1;
  return 0;
}

__device__ __noinline__ int conflict_exact(rpd_d4 p1, rpd_d4 p2, rpd_d4 p3,
                                           rpd_d4 e) {
  return rpd_exact_det4_sign(p1, p2, p3, e);
}

// sign of det3(normals) == 0 ? (is_vertex_perturb, convex_cell.cu:274-316)
// returns 1 degenerate, 0 fine, -1 undecided
__device__ __forceinline__ int perturb_filtered(const rpd_d4& p1,
                                                const rpd_d4& p2,
                                                const rpd_d4& p3) {
  double d, q;
  rpd_det3p(p1.x, p1.y, p1.z, p2.x, p2.y, p2.z, p3.x, p3.y, p3.z, d, q);
  if (!(q < 1e280)) return -1;
  double eps = 6.0e-16 * q + 1e-290;
  if (d > eps || d < -eps) return 0;
  if (q == 0.0) return 1;  // all products zero: exactly degenerate
  return -1;
}

__device__ __noinline__ int perturb_exact(rpd_d4 p1, rpd_d4 p2, rpd_d4 p3) {
  return rpd_exact_w_sign(p1, p2, p3) == 0 ? 1 : 0;
}

// --------------------------------------------------------- tet planes
// face k opposite vertex k with vertices tet_faces_lvid[k]
// (convex_cell.h:24-25): {2,1,3}, {0,2,3}, {1,0,3}, {0,1,2}
__device__ __forceinline__ rpd_d4 tri(const double4& a, const double4& b,
                                      const double4& c) {
  return rpd_tri_plane(a.x, a.y, a.z, b.x, b.y, b.z, c.x, c.y, c.z);
}
__device__ __forceinline__ void tet_planes(const double4 V[4], rpd_d4 pl[4]) {
  pl[0] = tri(V[2], V[1], V[3]);
  pl[1] = tri(V[0], V[2], V[3]);
  pl[2] = tri(V[1], V[0], V[3]);
  pl[3] = tri(V[0], V[1], V[2]);
}
// initial dual triangles (convex_cell.cu:183-186)
__constant__ uint8_t c_init_ver[4][3] = {{1, 3, 2}, {0, 2, 3}, {0, 3, 1},
                                         {0, 1, 2}};
// initial edges for local vertex pairs (0,1),(0,2),(0,3),(1,2),(1,3),(2,3)
// (convex_cell.cu:202-207)
__constant__ uint8_t c_init_edge[6][2] = {{2, 3}, {1, 3}, {1, 2},
                                          {0, 3}, {0, 2}, {0, 1}};

__device__ __forceinline__ uint32_t meta_byte(const TetMeta& m, int k) {
  // k in [0,16): x:0-3, y:4-7, z:8-11, w:12-15
  uint32_t w = k < 4 ? m.x : (k < 8 ? m.y : (k < 12 ? m.z : m.w));
  return (w >> (8 * (k & 3))) & 255u;
}

// 1/x: hardware reciprocal estimate refined by two Newton steps (relative
// error ~1 ulp for the normal, finite x used here)
__device__ __forceinline__ double rcp64(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = fma(-x, r, 1.0);
  r = fma(r, e, r);
  e = fma(-x, r, 1.0);
  return fma(r, e, r);
}
// binary search in a sorted u64 array
__device__ __forceinline__ bool has_key(const uint64_t* keys, int64_t n,
                                        uint64_t k) {
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (keys[mid] < k)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo < n && keys[lo] == k;
}

// ------------------------------------- polytopes held by one wavefront
// Vertex slot 64 q + lane is slot q of a lane: its plane triple in tr[q] as
// bytes a | b << 8 | c << 16; alive[q] marks the slots in use.
// v of lane l (l the same in every lane)
__device__ __forceinline__ double lane_value(double v, int l) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)u, l);
  const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), l);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
__device__ __forceinline__ float lane_value(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ uint32_t lane_value(uint32_t v, int l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
__device__ __forceinline__ int lanes_below(uint64_t m, int lane) {
  return __popcll(m & ((1ull << lane) - 1));
}
// The edges that a plane cuts when it removes the vertices out: the pairs
// (removed, kept) that share two planes.  Every lane compares its own
// triples with one removed vertex at a time.  s_new[0 .. n_new) receives
// the shared planes a | b << 8 (as far as 64 kVS); n_edge counts the edges
// at removed vertices, three each in a sound polytope.
template <int kVS>
__device__ __forceinline__ void cut_edges(const uint32_t (&tr)[kVS],
                                          const uint64_t (&alive)[kVS],
                                          const uint64_t (&out)[kVS],
                                          int lane, uint32_t* s_new,
                                          int& n_new, int& n_edge) {
  n_new = n_edge = 0;
#pragma unroll
  for (int q = 0; q < kVS; ++q) {
    uint64_t todo = out[q];
    while (todo) {
      const int r = __ffsll((long long)todo) - 1;
      todo &= todo - 1;
      const uint32_t t = lane_value(tr[q], r);
      const uint32_t a = t & 255, b = (t >> 8) & 255, c = (t >> 16) & 255;
#pragma unroll
      for (int u = 0; u < kVS; ++u) {
        if (alive[u] == 0) continue;
        const uint32_t x = tr[u] & 255, y = (tr[u] >> 8) & 255,
                       z = (tr[u] >> 16) & 255;
        const bool ha = x == a || y == a || z == a;
        const bool hb = x == b || y == b || z == b;
        const bool hc = x == c || y == c || z == c;
        const bool two = ha ? hb != hc : hb && hc;
        const uint64_t edge = ballot(two) & alive[u];
        n_edge += __popcll(edge);
        const uint64_t nw = edge & ~out[u];
        const int at = n_new + lanes_below(nw, lane);
        if (((nw >> lane) & 1) && at < 64 * kVS)
          s_new[at] = !ha ? b | (c << 8) : !hb ? a | (c << 8) : a | (b << 8);
        n_new += __popcll(nw);
      }
    }
  }
}

}  // namespace rpd
