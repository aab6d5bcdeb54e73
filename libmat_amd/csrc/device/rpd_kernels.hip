// The convex-cell clip: G cells per wavefront, 64/G lanes per cell, cell
// state in LDS: the reference clip loop (convex_cell.cu:680-774) with
// lane-parallel conflict tests (ballot), serial cavity boundary walk,
// lane-parallel edge/vertex creation and FP64 geometry.
//
// The kernel has many shapes; the file is compiled once per RPD_CLIP_PART
// (0..3: the small tier's four capacities, 4: full capacity and the exact
// tier) so that they build side by side.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "rpd_capi.h"
#include "rpd_clip.h"
#include "rpd_geom.h"

#ifndef RPD_CLIP_PART
#error "RPD_CLIP_PART selects the shapes to compile"
#endif

namespace rpd {

// 128-bit vertex masks as (lo, hi) words
__device__ __forceinline__ bool mbit(uint64_t lo, uint64_t hi, int v) {
  return v < 64 ? (lo >> v) & 1 : (hi >> (v - 64)) & 1;
}
__device__ __forceinline__ uint64_t low_bits(int n) {  // bits [0, n), n <= 64
  return n >= 64 ? ~0ull : (1ull << n) - 1;
}
// bits [a, b), 0 <= a <= b <= 128
__device__ __forceinline__ void mrange(int a, int b, uint64_t& lo,
                                       uint64_t& hi) {
  lo = low_bits(min(b, 64)) & ~low_bits(min(a, 64));
  hi = low_bits(max(b, 64) - 64) & ~low_bits(max(a, 64) - 64);
}
// position of the k-th lowest (k >= 1) set bit
__device__ __forceinline__ int mkth_low(uint64_t lo, uint64_t hi, int k) {
  const int nl = __popcll(lo);
  uint64_t w = lo;
  int base = 0;
  if (k > nl) {
    k -= nl;
    w = hi;
    base = 64;
  }
  for (int i = 1; i < k; ++i) w &= w - 1;
  return base + __ffsll((long long)w) - 1;
}
// position of the k-th highest (k >= 1) set bit
__device__ __forceinline__ int mkth_high(uint64_t lo, uint64_t hi, int k) {
  const int nh = __popcll(hi);
  uint64_t w = hi;
  int base = 64;
  if (k > nh) {
    k -= nh;
    w = lo;
    base = 0;
  }
  for (int i = 1; i < k; ++i) w &= ~(1ull << (63 - __clzll((long long)w)));
  return base + 63 - __clzll((long long)w);
}

template <int L>
__device__ __forceinline__ uint64_t group_bits(uint64_t b, int g) {
  if constexpr (L == 64) {
    return b;
  } else {
    return (b >> (g * L)) & ((1ull << L) - 1);
  }
}

// ---- sums and ORs over the L lanes of a cell's group, butterfly with
// offsets L/2, ..., 1.  Groups of 4 lanes are quads: their exchanges are
// DPP quad permutations (one VALU move per 32 bits) instead of LDS-routed
// lane shuffles.
template <int C>
__device__ __forceinline__ uint32_t quad_perm(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, C, 0xF, 0xF, false);
}
template <int C>
__device__ __forceinline__ double quad_perm(double v) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const uint64_t lo = quad_perm<C>((uint32_t)u);
  const uint64_t hi = quad_perm<C>((uint32_t)(u >> 32));
  return __longlong_as_double((long long)((hi << 32) | lo));
}
constexpr int kXor2 = 0x4E;  // quad lanes (2, 3, 0, 1)
constexpr int kXor1 = 0xB1;  // quad lanes (1, 0, 3, 2)
template <int L>
__device__ __forceinline__ double group_sum(double x) {
  if constexpr (L == 4) {
    x += quad_perm<kXor2>(x);
    x += quad_perm<kXor1>(x);
  } else {
#pragma unroll
    for (int off = L / 2; off > 0; off >>= 1) x += __shfl_xor(x, off);
  }
  return x;
}
template <int L>
__device__ __forceinline__ uint32_t group_or(uint32_t x) {
  if constexpr (L == 4) {
    x |= quad_perm<kXor2>(x);
    x |= quad_perm<kXor1>(x);
  } else {
#pragma unroll
    for (int off = L / 2; off > 0; off >>= 1) x |= __shfl_xor(x, off);
  }
  return x;
}

// ---- FP64 geometry helpers (tolerance-checked, not bit-compared)
// foot F = C - s n_p of C on plane p, given 1/|n_p|^2; returns s =
// (n_p.C + d_p) / |n_p|^2
__device__ __forceinline__ double foot_plane(const rpd_d4& p, double inv_nn,
                                             const double C[3], double F[3]) {
#pragma clang fp contract(fast)
  const double s = (p.x * C[0] + p.y * C[1] + p.z * C[2] + p.w) * inv_nn;
  F[0] = C[0] - s * p.x;
  F[1] = C[1] - s * p.y;
  F[2] = C[2] - s * p.z;
  return s;
}
// foot of C on the line through A with direction n_p x n_q
__device__ __forceinline__ void foot_line(const rpd_d4& p, const rpd_d4& q,
                                          const double A[3], const double C[3],
                                          double E[3]) {
#pragma clang fp contract(fast)
  const double d0 = p.y * q.z - p.z * q.y;
  const double d1 = p.z * q.x - p.x * q.z;
  const double d2 = p.x * q.y - p.y * q.x;
  const double dd = d0 * d0 + d1 * d1 + d2 * d2;
  const double s =
      ((C[0] - A[0]) * d0 + (C[1] - A[1]) * d1 + (C[2] - A[2]) * d2) *
      rcp64(dd);
  E[0] = A[0] + s * d0;
  E[1] = A[1] + s * d1;
  E[2] = A[2] + s * d2;
}
// twice the signed area of triangle (P, Q, A) along the (unnormalised)
// normal n
__device__ __forceinline__ double tri_area2(const double P[3],
                                            const double Q[3],
                                            const double A[3],
                                            const rpd_d4& n) {
#pragma clang fp contract(fast)
  const double u0 = Q[0] - P[0], u1 = Q[1] - P[1], u2 = Q[2] - P[2];
  const double v0 = A[0] - P[0], v1 = A[1] - P[1], v2 = A[2] - P[2];
  return (u1 * v2 - u2 * v1) * n.x + (u2 * v0 - u0 * v2) * n.y +
         (u0 * v1 - u1 * v0) * n.z;
}
__device__ __forceinline__ void vertex_pos(const rpd_d4& a, const rpd_d4& b,
                                           const rpd_d4& c, double A[3]) {
  rpd_d4 X, Q;
  rpd_vertex_homog(a, b, c, X, Q);
  const double r = rcp64(X.w);
  A[0] = X.x * r;
  A[1] = X.y * r;
  A[2] = X.z * r;
}

// resident wavefronts per SIMD the compiler must allow: 4 for the 16-cell
// shape with the tightest capacities (its register count otherwise lands
// just above the 4-wave limit of 128; measured 8 % faster), no constraint
// otherwise (the same hint slows the 8-cell shapes)
template <int G, class C>
constexpr int clip_min_waves() {
  return (G == 16 && C::V <= 16) ? 4 : 1;
}

// kCert: the learned path's launches, which evaluate the completeness
// certificate on every final cell (a.cert); the plain path's launches are
// compiled without it
template <int G, class C, bool kExact, bool kCert>
__global__ __launch_bounds__(64, (clip_min_waves<G, C>())) void k_clip(
    ClipArgs a) {
  constexpr int L = 64 / G;
  static_assert(L >= 4, "the tet's four planes are set up one per lane");
  constexpr int V = C::V, P = C::P, E = C::E;
  constexpr int VS = (V + L - 1) / L;
  constexpr bool kFull = (P == RPD_MAX_P);
  __shared__ double4 s_pl[G][P];
  __shared__ int32_t s_src[G][P];
  __shared__ uint8_t s_h[G][P];
  // the cavity boundary: successor bytes of the serial walk; up to 16
  // planes, first the planes' directed edges (16 out, 16 in), and the cycle
  // is packed in a register
  constexpr bool kPacked = P <= 16;
  __shared__ uint32_t s_bd[G][kPacked ? P : (P + 3) / 4];
  __shared__ uint8_t s_cyc[kPacked ? 1 : G][P + 1];
  uint8_t(*const s_bn)[sizeof(s_bd[0])] =
      reinterpret_cast<uint8_t(*)[sizeof(s_bd[0])]>(s_bd);
  __shared__ uint32_t s_ver[G][V];
  // s_adj[p]: bit q (q < p) set iff the edge list holds the pair (q, p)
  using AdjT = typename std::conditional<
      (P <= 16), uint16_t,
      typename std::conditional<(P <= 32), uint32_t, uint64_t>::type>::type;
  __shared__ AdjT s_adj[G][P];
  // per cell: the largest |a|, |b|, |c|, |d| over its planes (filter bound)
  __shared__ double s_mx[G][4];

  const int lane = threadIdx.x;
  const int g = lane / L, j = lane % L;
  // XCD-aware order: consecutive items stay on one XCD (8 XCDs,
  // round-robin dispatch of workgroups)
  const int64_t nb = gridDim.x;
  int64_t blk = blockIdx.x;
  if (nb >= 8 && !a.slot_by_cell) {
    const int64_t per = nb / 8;
    const int64_t xcd = blk % 8, pos = blk / 8;
    if (pos < per) blk = xcd * per + pos;
  }
  const int64_t item = blk * G + g;
  const int64_t n_items =
      a.n_items_d64 ? dev_count(a.n_items, a.n_items_d64)
                    : dev_count32(a.n_items, a.n_items_d32, a.n_sub);
  if (item >= n_items) return;
  const int64_t cidx = a.items ? a.items[item] : a.item_base + item;
  const int64_t slot = a.slot_by_cell ? cidx : a.slot_base + item;
  // the slot's edge records are written at its start as the edges are
  // appended (the reference never removes an edge), so they need no LDS
  // copy; the vertices and plane sources follow the last one at the end
  uint32_t* const wslot = a.out.words + slot * a.out.stride_words;
  uint32_t* const wedge = wslot;
  const Cand cd = a.cand[cidx];
  const int t = cd.tet, s = cd.seed;
  const int4 tv = a.M.tet_v[t];
  const TetMeta tm = a.M.tet_meta[t];
  const int64_t k0 = a.S.knn_off[s];
  const int deg = (int)(a.S.knn_off[s + 1] - k0);
  uint64_t m0 = a.use_mask ? cd.m0 : ~0ull;
  uint64_t m1 = a.use_mask ? cd.m1 : ~0ull;

  // ---- init the cell as its tet (convex_cell.cu:116-214)
  {
    if (j < 4) {
      // face j = tet_faces_lvid[j]: {2,1,3}, {0,2,3}, {1,0,3}, {0,1,2}
      const int ia = j == 0 ? tv.z : (j == 2 ? tv.y : tv.x);
      const int ib = j == 0 ? tv.y : (j == 1 ? tv.z : (j == 2 ? tv.x : tv.y));
      const int ic = j == 3 ? tv.z : tv.w;
      const rpd_d4 p = tri(a.M.vert[ia], a.M.vert[ib], a.M.vert[ic]);
      s_pl[g][j] = make_double4(p.x, p.y, p.z, p.w);
      s_src[g][j] = -1 - j;
      s_h[g][j] = (uint8_t)meta_byte(tm, j);
      s_ver[g][j] = c_init_ver[j][0] | (c_init_ver[j][1] << 8) |
                    (c_init_ver[j][2] << 16) | (meta_byte(tm, 4 + j) << 24);
      s_adj[g][j] = (AdjT)((1u << j) - 1u);  // the six edges of the tet
    }
    for (int q = j; q < 6; q += L)
      wedge[q] = c_init_edge[q][0] | (c_init_edge[q][1] << 8) |
                 (meta_byte(tm, 8 + q) << 16);
  }
  wsync();
  if (j < 4) {  // row maxima of the four tet planes, one row per lane
    double m = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const double4 pq = s_pl[g][q];
      const double v = j == 0 ? pq.x : j == 1 ? pq.y : j == 2 ? pq.z : pq.w;
      m = fmax(m, fabs(v));
    }
    s_mx[g][j] = m;
  }
  wsync();
  int nb_v = 4, nb_p = 4, nb_e = 6;
  uint32_t status = RPD_SUCCESS;
  uint32_t n_det = 0, n_bis = 0, n_exd = 0;  // executed work (count_work)
  bool on_plane = false;  // exact tier: a vertex lay exactly on a plane
  // next neighbour position after k that may cut the cell
  auto next_pos = [&](int k) {
    int nk = k + 1;
    if (nk < 64) {
      uint64_t r = m0 >> nk;
      if (r)
        nk += __ffsll((long long)r) - 1;
      else
        nk = 64;
    }
    if (nk >= 64 && nk < 128) {
      uint64_t r = m1 >> (nk - 64);
      if (r)
        nk += __ffsll((long long)r) - 1;
      else
        nk = 128;
    }
    return nk;
  };
  // the plane of the next step is loaded one step ahead (the masks fix the
  // positions in advance), so its latency overlaps the current step
  int k = -1;
  int kp = next_pos(-1);
  int mp = -1;
  rpd_d4 ep{0, 0, 0, 0};
  if (kp < deg) {
    mp = a.S.knn_ids[k0 + kp];
    ep = ld4(a.S.knn_bis + k0 + kp);
  }
  for (;;) {
    // at the reference's plane capacity every further neighbour overflows,
    // whether or not it can cut (new_plane checks the count before the
    // plane is tested, convex_cell.cu:561-565), so a masked one does too
    if (kFull && nb_p >= P && k + 1 < deg) {
      status = RPD_VERTEX_OVERFLOW;
      break;
    }
    k = kp;
    if (k >= deg) break;
    if (nb_p >= P) {
      status = kFull ? RPD_VERTEX_OVERFLOW : kStatusRerunLarge;
      break;
    }
    const int m = mp;
    const rpd_d4 e = ep;
    kp = next_pos(k);
    if (kp < deg) {
      mp = a.S.knn_ids[k0 + kp];
      ep = ld4(a.S.knn_bis + k0 + kp);
    }
    if (m == -1) break;
    const int cur = nb_p;
    n_bis += 1;
    n_det += nb_v;

    // ---- conflict tests, lane-parallel (convex_cell.cu:706-721); one
    // filter bound per step from the cell's row maxima and the new plane
    const double mx = fmax(s_mx[g][0], fabs(e.x));
    const double my = fmax(s_mx[g][1], fabs(e.y));
    const double mz = fmax(s_mx[g][2], fabs(e.z));
    const double mw = fmax(s_mx[g][3], fabs(e.w));
    const double bnd = (mx * my) * (mz * mw);
    // an unrepresentable bound leaves every sign undecided
    const double eps = bnd < 1e280 ? 2.5e-14 * bnd + 1e-290 : INFINITY;
    uint64_t conf_lo = 0, conf_hi = 0;
    bool undecided = false;
#pragma unroll
    for (int q = 0; q < VS; ++q) {
      // slots no cell of the wavefront has reached are not issued
      if (q > 0 && ballot(nb_v > q * L) == 0) break;
      const int v = q * L + j;
      int c = -1;
      if (v < nb_v) {
        const uint32_t w = s_ver[g][v];
        const rpd_d4 p1 = ld4(&s_pl[g][w & 255]);
        const rpd_d4 p2 = ld4(&s_pl[g][(w >> 8) & 255]);
        const rpd_d4 p3 = ld4(&s_pl[g][(w >> 16) & 255]);
        c = a.force_exact ? 0 : conflict_filtered_eps(p1, p2, p3, e, eps);
        if (kExact && c == 0) {
          const int sg = conflict_exact(p1, p2, p3, e);
          on_plane = on_plane || sg == 0;
          c = sg > 0 ? 1 : -1;
          ++n_exd;
        }
      }
      const uint64_t bc = group_bits<L>(ballot(c > 0), g);
      const uint64_t bu = group_bits<L>(ballot(c == 0), g);
      if (q * L < 64)
        conf_lo |= bc << (q * L);
      else
        conf_hi |= bc << (q * L - 64);
      undecided = undecided || bu != 0;
    }
    if (undecided) {
      status = kStatusRerunExact;
      break;
    }
    const int nr = __popcll(conf_lo) + __popcll(conf_hi);
    if (nr == 0) continue;  // the plane does not cut: popped (nb_p--)
    if (nr == nb_v) {
      status = RPD_NO_INTERSECTION;
      break;
    }
    if (j == 0) {
      s_pl[g][cur] = make_double4(e.x, e.y, e.z, e.w);
      s_src[g][cur] = m;
      s_h[g][cur] = 1;  // F_CELL_ADJ_DEFAULT
      s_adj[g][cur] = 0;
      s_mx[g][0] = mx;
      s_mx[g][1] = my;
      s_mx[g][2] = mz;
      s_mx[g][3] = mw;
    }
    nb_p = cur + 1;

    // ---- move conflicting vertices to the tail exactly as the serial
    // swap loop does (i scans from the front, end from the back, a
    // conflicting vertex at i is swapped with the one at end - 1), in
    // closed form: with nk = nb_v - nr kept vertices, the front pass reads
    // F = [0, m), m = nk + (vertex nk conflicts), the back pass reads
    // B = [m, nb_v) downwards.  A kept vertex of F stays; the j-th
    // conflicting vertex of F goes to nb_v - 1 (j = 1) or just below the
    // (j-1)-th kept vertex of B; the k-th kept vertex of B takes the place
    // of the k-th conflicting vertex of F; a conflicting vertex v of B goes
    // to v - 1.  (Up to 32 vertices the masks are one word.)
    if constexpr (V <= 32) {
      const uint32_t cm = (uint32_t)conf_lo;
      const int keep = nb_v - nr;
      const int m = keep + (int)((cm >> keep) & 1);
      // (m <= nb_v: all but the last vertex kept; nb_v < V <= 32)
      const uint32_t lo_m = (1u << m) - 1u;
      const uint32_t f = cm & lo_m;
      const uint32_t b = ~cm & ~lo_m & (nb_v >= 32 ? ~0u : (1u << nb_v) - 1u);
      uint32_t val[VS];
      int dst[VS];
#pragma unroll
      for (int q = 0; q < VS; ++q) {
        val[q] = 0;
        dst[q] = -1;
      }
#pragma unroll
      for (int q = 0; q < VS; ++q) {
        if (q > 0 && ballot(nb_v > q * L) == 0) break;
        const int v = q * L + j;
        if (v < nb_v) {
          val[q] = s_ver[g][v];
          const bool c = (cm >> v) & 1;
          const bool front = v < m;
          // conflicting in F: the jj-th one of F; kept in B: the kk-th
          // highest of B takes the kk-th lowest of F's places
          const int jj = __popc(f & ((2u << v) - 1u));
          const int kk = __popc(b >> v);
          int n = front ? jj - 1 : kk;  // set bits to take
          uint32_t w = front ? __brev(b) : f;
          dst[q] = front ? v : v - 1;
          if (front == c && n > 0) {
            for (int i = 1; i < n; ++i) w &= w - 1;
            const int at = __ffs((int)w) - 1;
            dst[q] = front ? 30 - at : at;
          } else if (front && c) {
            dst[q] = nb_v - 1;
          }
        }
      }
      wsync();
#pragma unroll
      for (int q = 0; q < VS; ++q)
        if (dst[q] >= 0) s_ver[g][dst[q]] = val[q];
      wsync();
    } else {
      const int nk = nb_v - nr;
      const int m = nk + (int)mbit(conf_lo, conf_hi, nk);
      uint64_t f_lo, f_hi, b_lo, b_hi;  // F's conflicts, B's kept vertices
      mrange(0, m, f_lo, f_hi);
      mrange(m, nb_v, b_lo, b_hi);
      f_lo &= conf_lo;
      f_hi &= conf_hi;
      b_lo &= ~conf_lo;
      b_hi &= ~conf_hi;
      uint32_t val[VS];
      int dst[VS];
#pragma unroll
      for (int q = 0; q < VS; ++q) {
        val[q] = 0;
        dst[q] = -1;
      }
#pragma unroll
      for (int q = 0; q < VS; ++q) {
        if (q > 0 && ballot(nb_v > q * L) == 0) break;
        const int v = q * L + j;
        if (v < nb_v) {
          val[q] = s_ver[g][v];
          const bool c = mbit(conf_lo, conf_hi, v);
          if (v < m) {
            if (!c) {
              dst[q] = v;
            } else {
              uint64_t r_lo, r_hi;
              mrange(0, v + 1, r_lo, r_hi);
              const int jj = __popcll(f_lo & r_lo) + __popcll(f_hi & r_hi);
              dst[q] = jj == 1 ? nb_v - 1 : mkth_high(b_lo, b_hi, jj - 1) - 1;
            }
          } else if (!c) {
            uint64_t r_lo, r_hi;
            mrange(v, nb_v, r_lo, r_hi);
            const int kk = __popcll(b_lo & r_lo) + __popcll(b_hi & r_hi);
            dst[q] = mkth_low(f_lo, f_hi, kk);
          } else {
            dst[q] = v - 1;
          }
        }
      }
      wsync();
#pragma unroll
      for (int q = 0; q < VS; ++q)
        if (dst[q] >= 0) s_ver[g][dst[q]] = val[q];
      wsync();
    }
    const int nv_old = nb_v;
    nb_v -= nr;
    (void)nv_old;

    // ---- cavity boundary (convex_cell.cu:618-678) and its cycle
    // The reference grows the removed region triangle by triangle (the
    // serial walk below: one dependent LDS round trip after another, for the
    // longest of the wavefront's cells).  Where the removed triangles form a
    // disk -- their directed edges without a reverse make one cycle -- the
    // walk always ends with that cycle (a disk's triangulation can be grown
    // in any order), so up to 16 planes it is built at once: every lane adds
    // its triangles' edges to the planes' masks, lanes then read their
    // planes' successors, and all lanes hold the cycle, 4 bits a plane.  It
    // starts at the first removed triangle's first plane; if that plane is
    // cut off altogether, the reference moves the start to the plane before
    // it in the last triangle added around it, the second of three when
    // there are three.  Everything else takes the walk.
    // (1.57 M tets: 1.77 -> 1.70 ms, the 8-cell shape of 32 vertices 0.90 ->
    // 0.64 ms on 16 uneven instances, together with the one-word vertex move
    // and the area sums below.  Growing larger fans for their start in
    // registers cost more than the walk, 1.76 ms; masks of 32 and 64 bits for
    // the shapes over 16 planes gave nothing: their walks are few.)
    uint32_t first = kEnd;
    uint64_t cyc = 0;
    int nbd = 0;
    bool walk = true;
    // the plane before plane p in the triangle w (kEnd: p is not in it)
    auto before = [](uint32_t w, uint32_t p) -> uint32_t {
      const uint32_t a = w & 255, b = (w >> 8) & 255, c = (w >> 16) & 255;
      return a == p ? c : b == p ? a : c == p ? b : kEnd;
    };
    if constexpr (kPacked) {
      for (int p = j; p < P; p += L) s_bd[g][p] = 0;
      wsync();
      for (int q = j; q < nr; q += L) {
        const uint32_t w = s_ver[g][nb_v + q];
        const uint32_t a = w & 255, b = (w >> 8) & 255, c = (w >> 16) & 255;
        atomicOr(&s_bd[g][a], (1u << b) | (65536u << c));
        atomicOr(&s_bd[g][b], (1u << c) | (65536u << a));
        atomicOr(&s_bd[g][c], (1u << a) | (65536u << b));
      }
      wsync();
      uint32_t nx_lo = 0, nx_hi = 0, on = 0;  // bit 16 of on: no simple cycle
      for (int p = j; p < P; p += L) {
        const uint32_t w = s_bd[g][p];
        const uint32_t o = w & ~(w >> 16) & 0xffffu;
        if (o != 0) {
          const uint64_t n = (uint64_t)(uint32_t)(__ffs((int)o) - 1) << (4 * p);
          nx_lo |= (uint32_t)n;
          nx_hi |= (uint32_t)(n >> 32);
          on |= (1u << p) | ((o & (o - 1)) ? 65536u : 0u);
        }
      }
      nx_lo = group_or<L>(nx_lo);
      nx_hi = group_or<L>(nx_hi);
      on = group_or<L>(on);
      const uint64_t nx = ((uint64_t)nx_hi << 32) | nx_lo;
      const int len = __popc(on & 0xffffu);
      auto next = [&](uint32_t p) { return (uint32_t)(nx >> (4 * p)) & 15u; };
      uint32_t at = s_ver[g][nb_v] & 255;
      if (!((on >> at) & 1) && nr == 3)  // all three lie around it
        at = before(s_ver[g][nb_v + 1], at) & 31u;
      if ((on >> at) & 1) {
        uint32_t p = at;
        do {
          cyc |= (uint64_t)p << (4 * nbd);
          ++nbd;
          p = next(p);
        } while (p != at && nbd < len);
        walk = p != at || nbd != len || on > 0xffffu;
        first = at;
      }
    }
    if (walk) {
      first = kEnd;
      wsync();
      for (int p = j; p < P; p += L) s_bn[g][p] = kEnd;
      wsync();
      {
        int iter = 0, t = nb_v, r = nr;
        while (r > 0) {
          if (iter++ > 65535) {
            status = RPD_INCONSISTENT_BOUNDARY;
            break;
          }
          const uint32_t tw = s_ver[g][t];
          const uint32_t pa = tw & 255, pb = (tw >> 8) & 255,
                         pc = (tw >> 16) & 255;
          const uint32_t ba = s_bn[g][pa], bb = s_bn[g][pb], bc = s_bn[g][pc];
          const bool in0 = ba != kEnd, in1 = bb != kEnd, in2 = bc != kEnd;
          const bool n0 = bb == pa, n1 = bc == pb, n2 = ba == pc;
          bool simple = true;
          if (!n0 && !n1 && in1) simple = false;
          if (!n1 && !n2 && in2) simple = false;
          if (!n2 && !n0 && in0) simple = false;
          if (!n0 && !n1 && !n2) {
            if (first == kEnd) {
              wsync();
              s_bn[g][pa] = pb;
              s_bn[g][pb] = pc;
              s_bn[g][pc] = pa;
              first = pa;
              wsync();
            } else {
              simple = false;
            }
          }
          if (!simple) {
            ++t;
            if (t == nb_v + r) t = nb_v;
            continue;
          }
          wsync();
          if (!n0) s_bn[g][pa] = pb;
          if (!n1) s_bn[g][pb] = pc;
          if (!n2) s_bn[g][pc] = pa;
          wsync();
          if (n0 && n1) {
            if (first == pb) first = s_bn[g][pb];
            wsync();
            s_bn[g][pb] = kEnd;
            wsync();
          }
          if (n1 && n2) {
            if (first == pc) first = s_bn[g][pc];
            wsync();
            s_bn[g][pc] = kEnd;
            wsync();
          }
          if (n2 && n0) {
            if (first == pa) first = s_bn[g][pa];
            wsync();
            s_bn[g][pa] = kEnd;
            wsync();
          }
          const int last = nb_v + r - 1;
          const uint32_t lw = s_ver[g][last];
          wsync();
          s_ver[g][t] = lw;
          s_ver[g][last] = tw;
          wsync();
          t = nb_v;
          --r;
        }
      }
    }
    if (status != RPD_SUCCESS) break;
    if (first == kEnd) {
      if (kFull && nb_p >= RPD_MAX_P && k + 1 < deg) {
        status = RPD_VERTEX_OVERFLOW;
        break;
      }
      continue;
    }
    if (walk) {
      cyc = 0;
      nbd = 0;
      uint32_t cir = first;
      do {
        if (nbd >= P || cir >= (uint32_t)P) break;
        if constexpr (kPacked)
          cyc |= (uint64_t)cir << (4 * nbd);
        else if (j == 0)
          s_cyc[g][nbd] = (uint8_t)cir;
        ++nbd;
        cir = s_bn[g][cir];
      } while (cir != first);
      if (cir != first) {
        status = RPD_INCONSISTENT_BOUNDARY;
        break;
      }
    }
    wsync();
    // plane q of the cycle
    auto cycle = [&](int q) -> uint32_t {
      if constexpr (kPacked)
        return (uint32_t)(cyc >> (4 * q)) & 15u;
      else
        return s_cyc[g][q];
    };
    // ---- new edges (cur, cir) (convex_cell.cu:604-616, 752-758)
    if (nb_e + nbd > E) {
      status = kFull ? RPD_EDGE_OVERFLOW : kStatusRerunLarge;
      break;
    }
    const uint32_t hcur = s_h[g][cur];
    uint32_t adj_lo = 0, adj_hi = 0;  // the planes now joined to cur
    for (int q = j; q < nbd; q += L) {
      const uint32_t c2 = cycle(q);
      const uint32_t hz = max(hcur, (uint32_t)s_h[g][c2]);
      const uint32_t lo = min((uint32_t)cur, c2), hi = max((uint32_t)cur, c2);
      wedge[nb_e + q] = lo | (hi << 8) | (hz << 16);
      if (P <= 32 || c2 < 32)
        adj_lo |= 1u << (c2 & 31);
      else
        adj_hi |= 1u << (c2 - 32);
    }
    adj_lo = group_or<L>(adj_lo);
    if constexpr (P > 32) adj_hi = group_or<L>(adj_hi);
    if (j == 0) s_adj[g][cur] = (AdjT)(((uint64_t)adj_hi << 32) | adj_lo);
    wsync();
    // ---- new vertices (cur, cir, next(cir)) (convex_cell.cu:760-772)
    int first_bad = 1 << 30;   // first index failing overflow or perturb
    int bad_kind = 0;          // 1 overflow, 2 perturb, 3 edge lookup, 4 undecided
    for (int q0 = 0; q0 < nbd; q0 += L) {
      const int q = q0 + j;
      int kind = 0;
      if (q < nbd) {
        const uint32_t c1 = cycle(q);
        const uint32_t c2 = cycle(q + 1 < nbd ? q + 1 : 0);
        if (nb_v + q + 1 >= V) {
          kind = 1;
        } else {
          // adjacency = max over the three edges (first match in list)
          // the new edges (cur, c1), (cur, c2) carry max(h_cur, h_c)
          const uint32_t z1 = max(hcur, (uint32_t)s_h[g][c1]);
          const uint32_t z2 = max(hcur, (uint32_t)s_h[g][c2]);
          const uint32_t lo = min(c1, c2), hi = max(c1, c2);
          // the edge (lo, hi), without a scan of the list: a pair of tet
          // faces is one of the six initial records (list positions 0-5,
          // pairs (2,3), (1,3), (1,2), (0,3), (0,2), (0,1)); a pair with a
          // bisector was appended once, when its later plane was clipped,
          // with z = max of the two planes' adjacency bytes
          const bool found = (s_adj[g][hi] >> lo) & 1;
          uint32_t z3 = 0;
          if (found) {
            if (hi < 4)
              z3 = meta_byte(tm, 8 + 5 - (lo * (7 - lo) / 2 + (hi - lo - 1)));
            else
              z3 = max((uint32_t)s_h[g][lo], (uint32_t)s_h[g][hi]);
          }
          if (!found) {
            kind = 3;
          } else {
            const rpd_d4 pc = ld4(&s_pl[g][cur]);
            const rpd_d4 p1 = ld4(&s_pl[g][c1]);
            const rpd_d4 p2 = ld4(&s_pl[g][c2]);
            int pf = a.force_exact ? -1 : perturb_filtered(pc, p1, p2);
            if (kExact && pf < 0) pf = perturb_exact(pc, p1, p2);
            if (pf == 1)
              kind = 2;
            else if (pf < 0)
              kind = 4;
            const uint32_t z = max(max(z1, z2), z3);
            s_ver[g][nb_v + q] = cur | (c1 << 8) | (c2 << 16) | (z << 24);
          }
        }
      }
      // first failing index in this pass (in order), kinds by priority of
      // position; overflow at q stops before the perturb test of q
      const uint64_t bad = group_bits<L>(ballot(kind != 0), g);
      if (bad && first_bad == (1 << 30)) {
        const int qb = q0 + __ffsll((long long)bad) - 1;
        first_bad = qb;
        // broadcast the kind of lane (qb - q0) of this group
        bad_kind = __shfl(kind, g * L + (qb - q0));
      }
    }
    wsync();
    if (first_bad != (1 << 30)) {
      if (bad_kind == 1)
        status = kFull ? RPD_TRIANGLE_OVERFLOW : kStatusRerunLarge;
      else if (bad_kind == 2)
        status = RPD_NEEDS_PERTURB;
      else if (bad_kind == 3)
        status = RPD_INCONSISTENT_BOUNDARY;
      else
        status = kStatusRerunExact;
      break;
    }
    nb_e += nbd;
    nb_v += nbd;
    if (kFull && nb_p >= RPD_MAX_P && k + 1 < deg) {
      status = RPD_VERTEX_OVERFLOW;
      break;
    }
  }

  // ---- write the slot
  const SlotView& o = a.out;
  if (status == RPD_SUCCESS && a.geometry) {
    // (tolerance-checked arithmetic: products and sums may fuse)
#pragma clang fp contract(fast)
    // FP64 geometry in one pass over the vertices.  Around each vertex A
    // lie 6 tets (C, X, Y, A) whose bases (X, Y, A) tile A's corner of its
    // three faces: X, Y run over the feet of C on A's 3 planes and on its 3
    // edge lines (the decomposition of the reference's
    // get_tet_decomposition_of_vertex, convex_cell.cu:986-1006).  Their
    // volumes give the cell volume and centroid, their bases the facet
    // areas (signed along each plane normal, so feet outside a face
    // cancel).  C is the cell's vertex 0, so rounding scales with the cell.
    // A base (X, Y, A) lies in A's plane p, so six times the signed volume
    // of (X, Y, C, A) is -area2(X, Y, A; n_p) * s_p, with s_p the foot
    // parameter of C on p (C - F_p = s_p n_p): one product per tet.
    double Cc[3];
    {
      const uint32_t w0 = s_ver[g][0];
      vertex_pos(ld4(&s_pl[g][w0 & 255]), ld4(&s_pl[g][(w0 >> 8) & 255]),
                 ld4(&s_pl[g][(w0 >> 16) & 255]), Cc);
    }
    constexpr int PA = (P + L - 1) / L;  // planes per lane
    double acc[PA];
#pragma unroll
    for (int q = 0; q < PA; ++q) acc[q] = 0.0;
    double vol6 = 0, mx = 0, my = 0, mz = 0;
    for (int q0 = 0; q0 < nb_v; q0 += L) {
      const int v = q0 + j;
      uint32_t ia = kEnd, ib = kEnd, ic = kEnd;
      double ca = 0, cb = 0, cc = 0;
      if (v < nb_v) {
        const uint32_t w = s_ver[g][v];
        ia = w & 255;
        ib = (w >> 8) & 255;
        ic = (w >> 16) & 255;
        const rpd_d4 pa = ld4(&s_pl[g][ia]);
        const rpd_d4 pb = ld4(&s_pl[g][ib]);
        const rpd_d4 pc = ld4(&s_pl[g][ic]);
        double A[3];
        vertex_pos(pa, pb, pc, A);
        // walk the six (foot, foot) pairs around A so that each foot dies
        // after its two tets and base triangles
        double Fa[3], Xp[3], Xn[3];
        const double sa = foot_plane(
            pa, rcp64(pa.x * pa.x + pa.y * pa.y + pa.z * pa.z), Cc, Fa);
#define RPD_ACC(P0, P1, PL, SP, CONTRIB)                         \
  {                                                              \
    const double ar2 = tri_area2(P0, P1, A, PL);                 \
    const double tvl = -ar2 * SP;                                \
    vol6 += tvl;                                                 \
    mx += tvl * (((P0[0] + P1[0]) + Cc[0]) + A[0]);              \
    my += tvl * (((P0[1] + P1[1]) + Cc[1]) + A[1]);              \
    mz += tvl * (((P0[2] + P1[2]) + Cc[2]) + A[2]);              \
    CONTRIB += ar2;                                              \
  }
        foot_line(pa, pb, A, Cc, Xp);                               // Eab
        RPD_ACC(Fa, Xp, pa, sa, ca)
        const double sb = foot_plane(
            pb, rcp64(pb.x * pb.x + pb.y * pb.y + pb.z * pb.z), Cc, Xn);
        RPD_ACC(Xp, Xn, pb, sb, cb)                                 // Eab, Fb
        foot_line(pb, pc, A, Cc, Xp);                               // Ebc
        RPD_ACC(Xn, Xp, pb, sb, cb)                                 // Fb, Ebc
        const double sc = foot_plane(
            pc, rcp64(pc.x * pc.x + pc.y * pc.y + pc.z * pc.z), Cc, Xn);
        RPD_ACC(Xp, Xn, pc, sc, cc)                                 // Ebc, Fc
        foot_line(pc, pa, A, Cc, Xp);                               // Eca
        RPD_ACC(Xn, Xp, pc, sc, cc)                                 // Fc, Eca
        RPD_ACC(Xp, Fa, pa, sa, ca)                                 // Eca, Fa
#undef RPD_ACC
      }
      // per-plane sums over the group's lanes (fixed butterfly order);
      // lane p % L keeps plane p
      if constexpr (L == 4) {
        // a quad's lanes read each other's three contributions (DPP
        // broadcasts) and pick those of their own planes: every lane works
        // for its planes, instead of all four summing each plane in turn
        // (12 planes: 148 instead of 264 instructions)
        const uint32_t pk = ia | (ib << 8) | (ic << 16);
        const uint32_t pk_s[4] = {quad_perm<0x00>(pk), quad_perm<0x55>(pk),
                                  quad_perm<0xAA>(pk), quad_perm<0xFF>(pk)};
        const double ca_s[4] = {quad_perm<0x00>(ca), quad_perm<0x55>(ca),
                                quad_perm<0xAA>(ca), quad_perm<0xFF>(ca)};
        const double cb_s[4] = {quad_perm<0x00>(cb), quad_perm<0x55>(cb),
                                quad_perm<0xAA>(cb), quad_perm<0xFF>(cb)};
        const double cc_s[4] = {quad_perm<0x00>(cc), quad_perm<0x55>(cc),
                                quad_perm<0xAA>(cc), quad_perm<0xFF>(cc)};
#pragma unroll
        for (int pi = 0; pi < PA; ++pi) {
          if (pi > 0 && ballot(nb_p > pi * L) == 0) break;
          const uint32_t p = (uint32_t)(pi * L + j);
          double c[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            c[u] = (pk_s[u] >> 16) == p ? cc_s[u] : 0.0;
            c[u] = ((pk_s[u] >> 8) & 255) == p ? cb_s[u] : c[u];
            c[u] = (pk_s[u] & 255) == p ? ca_s[u] : c[u];
          }
          acc[pi] += (c[0] + c[2]) + (c[1] + c[3]);
        }
      } else
#pragma unroll
      for (int pi = 0; pi < PA; ++pi) {
#pragma unroll
        for (int pj = 0; pj < L; ++pj) {
          const uint32_t p = (uint32_t)(pi * L + pj);
          if (p < (uint32_t)P && p < (uint32_t)nb_p) {
            double sp = (ia == p ? ca : 0.0) + (ib == p ? cb : 0.0) +
                        (ic == p ? cc : 0.0);
            sp = group_sum<L>(sp);
            if (j == pj) acc[pi] += sp;
          }
        }
      }
    }
    vol6 = group_sum<L>(vol6);
    mx = group_sum<L>(mx);
    my = group_sum<L>(my);
    mz = group_sum<L>(mz);
    if (j == 0) {
      double* gm = o.geom + 4 * slot;
      const double vol = vol6 / 6.0;
      const double inv = vol6 != 0 ? 1.0 / (4.0 * vol6) : 0.0;
      gm[0] = fabs(vol);
      gm[1] = mx * inv;
      gm[2] = my * inv;
      gm[3] = mz * inv;
    }
#pragma unroll
    for (int pi = 0; pi < PA; ++pi) {
      const int p = pi * L + j;
      if (p < nb_p) {
        const rpd_d4 pp = ld4(&s_pl[g][p]);
        const double nn = pp.x * pp.x + pp.y * pp.y + pp.z * pp.z;
        o.areas[slot * o.stride_areas + p] =
            fabs(acc[pi]) * 0.5 / sqrt(nn);
      }
    }
  }
  if (status == RPD_SUCCESS) {
    // vertices and plane sources right after the edges (in place)
    for (int v = j; v < nb_v; v += L) wslot[nb_e + v] = s_ver[g][v];
    for (int p = j; p < nb_p; p += L)
      wslot[nb_e + nb_v + p] = (uint32_t)s_src[g][p];
  }
  if constexpr (kExact) {
    // a vertex exactly on a plane: the configuration is degenerate and a
    // sphere whose cell meets the tet only in a face, an edge or a point
    // (a zero-volume cell, which the plain path emits) may touch this cell
    // without leaving an active facet here; the certificate cannot see it,
    // so the tet goes to the full relation (the exact tier runs one cell
    // per wavefront, so the ballot covers exactly this cell's lanes)
    if (kCert && ballot(on_plane) != 0 && j == 0) a.cert.flag[t] = 1;
  }
  if (kCert && status != kStatusRerunLarge && status != kStatusRerunExact &&
      status != RPD_NO_INTERSECTION) {
    const CertArgs& c = a.cert;
    if (status != RPD_SUCCESS) {
      if (j == 0) c.flag[t] = 1;
    } else {
      if (j == 0) c.has_cell[t] = 1;
      // planes with a vertex (the active facets), OR over the group
      uint64_t act0 = 0, act1 = 0;
      for (int v = j; v < nb_v; v += L) {
        const uint32_t w = s_ver[g][v];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const uint32_t p = (w >> (8 * q)) & 255u;
          if (p < 64)
            act0 |= 1ull << p;
          else
            act1 |= 1ull << (p - 64);
        }
      }
#pragma unroll
      for (int off = L / 2; off > 0; off >>= 1) {
        act0 |= (uint64_t)__shfl_xor((unsigned long long)act0, off);
        act1 |= (uint64_t)__shfl_xor((unsigned long long)act1, off);
      }
      const int64_t o0 = c.tet_off[t], o1 = c.tet_off[t + 1];
      for (int p = j; p < nb_p; p += L) {
        const bool active =
            p < 64 ? ((act0 >> p) & 1) : ((act1 >> (p - 64)) & 1);
        const int32_t src = s_src[g][p];
        if (!active || src < 0) continue;
        int64_t lo = o0, hi = o1;
        while (lo < hi) {
          const int64_t mid = (lo + hi) >> 1;
          if (c.mem_ids[mid] < src)
            lo = mid + 1;
          else
            hi = mid;
        }
        if (lo < o1 && c.mem_ids[lo] == src) continue;
        const uint64_t key = ((uint64_t)(uint32_t)t << 32) | (uint32_t)src;
        if (c.n_ext && has_key(c.ext, c.n_ext, key)) continue;
        const int r = atomicAdd(c.n_miss, 1);
        const int64_t cap =
            c.cap_n ? min((int64_t)c.cap, max((int64_t)4096, 2 * *c.cap_n))
                    : (int64_t)c.cap;
        if (r < cap)
          c.miss[r] = key;
        else
          c.flag[t] = 1;
      }
    }
  }
  if (a.work) {
    if (kExact) {  // exact determinants are per lane: sum over the group
#pragma unroll
      for (int d = 1; d < L; d <<= 1) n_exd += __shfl_xor(n_exd, d, 64);
    }
    if (j == 0) {
      unsigned long long* w = a.work + 4 * (blockIdx.x & 63);
      atomicAdd(w + 0, (unsigned long long)n_det);
      atomicAdd(w + 1, (unsigned long long)n_bis);
      if (status == RPD_SUCCESS) atomicAdd(w + 2, (unsigned long long)nb_v);
      if (n_exd) atomicAdd(w + 3, (unsigned long long)n_exd);
    }
  }
  if (j == 0) {
    o.hdr[slot] = (uint32_t)nb_v | ((uint32_t)nb_p << 8) |
                  ((uint32_t)nb_e << 16) | (status << 24);
    if (status == kStatusRerunLarge) {
      int r = atomicAdd(a.n_rerun_large, 1);
      if (r < a.cap_large)
        a.rerun_large[r] = (int32_t)cidx;
      else
        a.overflow[0] = 1;
    } else if (status == kStatusRerunExact) {
      int r = atomicAdd(a.n_rerun_exact, 1);
      if (r < a.cap_exact)
        a.rerun_exact[r] = (int32_t)cidx;
      else
        a.overflow[0] = 1;
    }
  }
}

// ------------------------------------------------------------- launches
template <int G, class C, bool kExact>
static void launch_shape(hipStream_t s, const ClipArgs& a) {
  const int blocks = (int)((a.n_items + G - 1) / G);
  if (a.cert.tet_off)
    hipLaunchKernelGGL((k_clip<G, C, kExact, true>), dim3(blocks), dim3(64), 0,
                       s, a);
  else
    hipLaunchKernelGGL((k_clip<G, C, kExact, false>), dim3(blocks), dim3(64),
                       0, s, a);
}
// any G of {1, 2, 4, 8, 16}; kMin: the smallest one compiled
template <class C, int kMin>
static void launch_small(hipStream_t s, int G, const ClipArgs& a) {
  if constexpr (kMin <= 1)
    if (G == 1) return launch_shape<1, C, false>(s, a);
  if constexpr (kMin <= 2)
    if (G == 2) return launch_shape<2, C, false>(s, a);
  switch (G) {
    case 4: return launch_shape<4, C, false>(s, a);
    case 8: return launch_shape<8, C, false>(s, a);
    default: return launch_shape<16, C, false>(s, a);
  }
}

void clip_part0(hipStream_t s, int G, const ClipArgs& a);
void clip_part1(hipStream_t s, int G, const ClipArgs& a);
void clip_part2(hipStream_t s, int G, const ClipArgs& a);
void clip_part3(hipStream_t s, int G, const ClipArgs& a);

#if RPD_CLIP_PART == 0
void clip_part0(hipStream_t s, int G, const ClipArgs& a) {
  launch_small<SmallCaps, 1>(s, G, a);
}
#elif RPD_CLIP_PART == 1
void clip_part1(hipStream_t s, int G, const ClipArgs& a) {
  launch_small<WideCaps, 1>(s, G, a);
}
#elif RPD_CLIP_PART == 2
void clip_part2(hipStream_t s, int G, const ClipArgs& a) {
  launch_small<TightCaps, 4>(s, G, a);
}
#elif RPD_CLIP_PART == 3
void clip_part3(hipStream_t s, int G, const ClipArgs& a) {
  launch_small<MidCaps, 4>(s, G, a);
}
#else
hipError_t clip_launch(hipStream_t s, int tier, int G, const ClipArgs& a,
                       int caps_id) {
  if (tier == 0) {
    switch (caps_id) {
      case 1: clip_part1(s, G, a); break;
      case 2: clip_part2(s, G, a); break;
      case 3: clip_part3(s, G, a); break;
      default: clip_part0(s, G, a); break;
    }
  } else if (tier == 1) {
    switch (G) {
      case 1: launch_shape<1, LargeCaps, false>(s, a); break;
      case 2: launch_shape<2, LargeCaps, false>(s, a); break;
      default: launch_shape<4, LargeCaps, false>(s, a); break;
    }
  } else {
    launch_shape<1, LargeCaps, true>(s, a);
  }
  return hipGetLastError();
}
#endif

}  // namespace rpd
