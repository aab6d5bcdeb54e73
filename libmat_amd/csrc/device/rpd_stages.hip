// HIP kernels of the restricted power diagram (RPD) for CDNA4 (gfx950).
//
// Pipeline of one rpd_run (see rpd_engine.hip for the host side):
//   k_site_bbox    one wavefront per flagged sphere: clips the domain box by
//                  the neighbour bisectors pushed outwards by the largest
//                  tet radius; the bbox of that polytope contains the
//                  centroid of every tet the sphere can relate to
//   k_tet_bin*     the mesh's tets in the order of a uniform grid of their
//                  centroids (once per mesh or tet subset)
//   k_rel_pairs    wavefronts per sphere: the reference's tet-sphere relation
//                  (voronoi.cu:154-193) over the tets of the grid rows that
//                  its polytope reaches
//   k_pair_*       the related pairs in tet order, ascending site id
//   k_cand_mask    the mask of neighbour planes that may cut the tet
//   k_clip         (rpd_kernels.hip) the clip; tiers: small capacity, full
//                  capacity, full capacity with exact arithmetic
//   k_compact_*    deterministic compaction into the output stream
#include <hip/hip_runtime.h>

#include "rpd_capi.h"
#include "rpd_clip.h"
#include "rpd_device.h"
#include "rpd_geom.h"

namespace rpd {

__global__ __launch_bounds__(256) void k_fill32(int32_t* p, int64_t n,
                                                int32_t v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// A captured run's re-run lists (cnt[1] small-tier overflows, cnt[2] exact
// re-runs, cnt[6] middle-tier overflows): after a clip launch's tiers the
// counts are checked against the list positions the host reserved
// (*overflow otherwise); with next_large >= 0 the counters then start at
// the positions reserved for the next launch.
__global__ void k_check_rerun_counts(int32_t* cnt, int32_t lim_large,
                                     int32_t lim_exact, int32_t lim_full,
                                     int32_t* overflow, int32_t next_large,
                                     int32_t next_exact, int32_t next_full) {
  if (threadIdx.x != 0) return;
  if (cnt[1] > lim_large || cnt[2] > lim_exact || cnt[6] > lim_full)
    *overflow = 1;
  if (next_large >= 0) {
    cnt[1] = next_large;
    cnt[2] = next_exact;
    cnt[6] = next_full;
  }
}

// ================================================= candidate gathering
struct BinGrid {
  double org[3];
  double inv_bs;
  int32_t dim[3];
  int32_t pad;
};

// One instance of a batch: its domain box, the largest distance of a tet
// corner from its tet's centroid (rho, with margin), and its candidate bin
// grid, whose bins are numbered from bin_base in the batch-wide bin space.
// The grid's first axis, along which its rows run, is the one with the most
// bins: axis k of g and of gdom (dom in that order) is axis ax[k] of the
// coordinates.  A flat or long mesh then has few long rows (3 x 297 instead
// of 297 x 297 of 3 bins: one sphere on 1.57 M tets, boxes and relation
// 2.0 -> 0.16 ms, graded by the third power along them 15.1 -> 0.15 ms).
struct InstInfo {
  BinGrid g;
  int64_t bin_base;
  double gdom[6];
  int32_t ax[4];
  double dom[6];
  double rho;
  BinGrid sg;        // grid of sphere centres (learned proposals)
  int64_t sg_base;
  int32_t site_off;  // first site of the instance, number of sites
  int32_t n_site;
};

__device__ __forceinline__ int bin_coord(double x, double org, double inv,
                                         int dim) {
  double f = floor((x - org) * inv);
  int c = f < 0 ? 0 : (f >= dim ? dim - 1 : (int)f);
  return c;
}

// One wavefront per sphere.  Polytope = domain box clipped by the
// neighbour bisectors, each pushed out by rho (max tet circum-radius about
// the centroid plus a margin).  Output bbox (lo, hi); empty if lo > hi.
// The bisectors are applied nearest first (ascending signed distance of
// the sphere centre to the bisector), so the polytope shrinks early and
// later planes rarely cut; the relation test takes the planes in that order
// too, to meet a rejecting neighbour early (its outcome does not depend on
// the order).
// The chain of clips bounds it (one site's wavefront is as long as the
// kernel for small sets), so the vertices stay in registers, two slots per
// lane, and a clip's edges are found by comparing all of them with each
// removed one (cut_edges).  With the vertices in LDS and one lane scanning
// all of them per removed vertex: 309 -> 39 us
// for 500 sites, 1,646 -> 153 us for 18,000.
constexpr int kBoxV = 128;      // vertices (overflow: whole-domain box)
constexpr int kBoxP = 128;      // 6 box planes + 122 neighbours
constexpr int kNearMax = 128;   // longest list ranked (else kept as is)

// inline neighbour word: the site id, with bit 31 set when the site is not
// flagged (it bounds cells but has none of its own)
constexpr uint32_t kNearUnflagged = 0x80000000u;
__device__ __forceinline__ int32_t near_word(const DevSites& S, int m) {
  return (int32_t)((uint32_t)m | (S.flags[m] == 1u ? 0u : kNearUnflagged));
}
__device__ __forceinline__ int near_id(int32_t w) { return w & 0x7fffffff; }

// component a of (x, y, z)
template <class T>
__device__ __forceinline__ T axis(T x, T y, T z, int a) {
  return a == 0 ? x : a == 1 ? y : z;
}

// bin range of a sphere's candidate box; false if empty
__device__ __forceinline__ bool bin_range(const double* b, const BinGrid& g,
                                          int r[6]) {
  if (b[0] > b[3] || b[1] > b[4] || b[2] > b[5]) return false;
  for (int a = 0; a < 3; ++a) {
    r[a] = bin_coord(b[a], g.org[a], g.inv_bs, g.dim[a]);
    r[3 + a] = bin_coord(b[3 + a], g.org[a], g.inv_bs, g.dim[a]);
  }
  return true;
}

// A sphere's relation test is cut into parts of up to kPartTets of the tets
// in the grid rows (y, z) of its box and of up to kRelRows rows, whose ranges
// a wavefront finds at once.  Where the tets are spread evenly a part is a
// fixed number of rows (part_rows[i] > 0), as many as keep the fullest rows
// within kPartTets.  Where that would make more than about twice the parts
// that the tets need (graded meshes, meshes that fill little of their box,
// subsets), parts are cut by count (part_rows[i] = 0), row by row, a row
// counting for no fewer than kRowTets; finding a part's rows then takes a
// pass over the rows before it.
// (1.57 M tets, the relation alone, up to 16 rows of together 170 bins | by
// count alone | so: 18,000 sites 0.51 | 0.55 | 0.49 ms; the grid graded by
// the fourth power, where one bin holds 69,000 tets, 7.7 | 3.4 | 3.3 ms, with
// 100 sites 5.4 | 0.17 | 0.17 ms.)
constexpr int kPartTets = 1024;
constexpr int kRelRows = 16;
constexpr int kRowTets = kPartTets / kRelRows;

// tets of row `row` of the box r (y fastest) and the first of them
__device__ __forceinline__ int row_tets(const int32_t* __restrict__ first,
                                        int64_t bin_base, const BinGrid& g,
                                        const int r[6], int row, int& f0) {
  const int ny = r[4] - r[1] + 1;
  const int y = r[1] + row % ny, z = r[2] + row / ny;
  const int64_t base =
      bin_base + (int64_t)g.dim[0] * (y + (int64_t)g.dim[1] * z);
  f0 = first[base + r[0]];
  return first[base + r[3] + 1] - f0;
}

// A bisector for the relation test: binary32 coefficients about the centre
// of the instance's domain box, aux.x a bound of the error of its computed
// value at any point of the box (three fused products and the rounding of
// plane and point: 5 u sum |e_a| h_a + 4 u |d|, h the box's half extents,
// u = 2^-24; 4e-7 covers it) plus the rounding of the two binary64 power
// distances that decide the relation and what coefficients, points and
// products below the normal range lose, aux.y the distance term of a tet's
// corners from its centroid.  Beyond aux.x the sign is the relation's.
// Where a value could leave binary32's range (d and the power distances grow
// with the square of the coordinates, so from extents of about 1e18 on) the
// plane is zero and its bound infinite: it narrows no row and decides no
// tet.
constexpr double kRelMax = 1e37;
__device__ __forceinline__ void rel_plane(const rpd_d4& e, const rpd_d4& si,
                                          const double4& sm, double nrm,
                                          double rho, const double* dom,
                                          float4& pl, float2& aux) {
  const double sum = fabs(e.x) + fabs(e.y) + fabs(e.z);
  double d = e.w, h = 0, far2 = 0, half = 0;
  for (int a = 0; a < 3; ++a) {
    const double ea = a == 0 ? e.x : a == 1 ? e.y : e.z;
    const double c = 0.5 * (dom[a] + dom[3 + a]);
    const double m = fmax(fabs(dom[a]), fabs(dom[3 + a]));
    const double ha = (dom[3 + a] - dom[a]) * 0.5;
    d += ea * c;
    h += fabs(ea) * ha;
    half += ha;
    far2 += m * m;
  }
  const double s2 = si.x * si.x + si.y * si.y + si.z * si.z + fabs(si.w) +
                    sm.x * sm.x + sm.y * sm.y + sm.z * sm.z + fabs(sm.w);
  const double eps =
      4e-7 * (h + fabs(d)) + 1e-14 * (far2 + s2) + 1.2e-38 * (half + sum);
  const double far = nrm * rho;
  // (negated, so that a NaN is out of range too)
  if (!(h + fabs(d) + half + sum + eps + far < kRelMax)) {
    pl = make_float4(0.f, 0.f, 0.f, 0.f);
    aux = make_float2(INFINITY, 0.f);
    return;
  }
  pl = make_float4((float)e.x, (float)e.y, (float)e.z, (float)d);
  aux.x = (float)eps + 1e-36f;
  aux.y = (float)far * 1.000001f;
}

__global__ __launch_bounds__(64) void k_site_bbox(DevSites S,
                                                  const InstInfo* inst,
                                                  const int32_t* site_inst,
                                                  double* bbox,  // 6/site
                                                  float4* rel_pl,
                                                  float2* rel_aux,
                                                  const int32_t* first,
                                                  int64_t* parts,
                                                  int32_t* part_rows,
                                                  unsigned long long* reg64,
                                                  int32_t* n_fallback) {
  constexpr int kVS = kBoxV / 64;
  __shared__ double4 s_pl[kBoxP];
  __shared__ double s_key[kNearMax];
  __shared__ int32_t s_near[kNearMax];
  __shared__ uint32_t s_new[kBoxV];
  const int i = blockIdx.x;
  const int lane = threadIdx.x;
  if (i >= S.n_site) {  // the block past the last site ends the part counts
    if (lane == 0) parts[i] = 0;
    return;
  }
  const InstInfo& I = inst[site_inst[i]];
  const double* dom = I.dom;
  const double rho = I.rho;
  double* out = bbox + 6 * (int64_t)i;
  // the box in the grid's axes, the parts that the tets of its grid rows
  // make, and its bins (a statistic); every lane calls it
  const int ax0 = I.ax[0], ax1 = I.ax[1], ax2 = I.ax[2];
  auto finish = [&](const double box[6]) {
    const double b[6] = {axis(box[0], box[1], box[2], ax0),
                         axis(box[0], box[1], box[2], ax1),
                         axis(box[0], box[1], box[2], ax2),
                         axis(box[3], box[4], box[5], ax0),
                         axis(box[3], box[4], box[5], ax1),
                         axis(box[3], box[4], box[5], ax2)};
    int r[6], rows = 0;
    if (bin_range(b, I.g, r)) rows = (r[4] - r[1] + 1) * (r[5] - r[2] + 1);
    int64_t tets = 0;
    int most = 1;
    for (int q = lane; q < rows; q += 64) {
      int f0;
      const int n = row_tets(first, I.bin_base, I.g, r, q, f0);
      tets += max(kRowTets, n);
      most = max(most, n);
    }
    for (int off = 32; off > 0; off >>= 1) {
      tets += __shfl_xor(tets, off);
      most = max(most, __shfl_xor(most, off));
    }
    if (lane != 0) return;
    for (int a = 0; a < 6; ++a) out[a] = b[a];
    if (rows > 0)
      atomicAdd(reg64 + (blockIdx.x & 63),
                (unsigned long long)((int64_t)rows * (r[3] - r[0] + 1)));
    const int per = max(1, min(kRelRows, kPartTets / most));
    const int64_t by_rows = (rows + per - 1) / per;
    const int64_t by_count = (tets + kPartTets - 1) / kPartTets;
    const bool even = most <= kPartTets && by_rows <= 2 * by_count + 2;
    parts[i] = even ? by_rows : by_count;
    part_rows[i] = even ? per : 0;
  };
  const double none[6] = {1.0, 1.0, 1.0, -1.0, -1.0, -1.0};
  if (S.flags[i] != 1u) {
    finish(none);
    return;
  }
  const int64_t k0 = S.knn_off[i];
  const int deg = (int)(S.knn_off[i + 1] - k0);
  bool fail = deg > kBoxP - 6;
  const rpd_d4 si = ld4(S.site + i);
  const bool ranked = deg <= kNearMax;
  if (ranked) {
    for (int k = lane; k < deg; k += 64) {
      const rpd_d4 e = rpd_bisector(si, ld4(S.site + S.knn_ids[k0 + k]));
      const double nn = e.x * e.x + e.y * e.y + e.z * e.z;
      double key = (e.x * si.x + e.y * si.y + e.z * si.z + e.w) / sqrt(nn);
      if (!(key == key)) key = -INFINITY;  // keep a strict total order
      s_key[k] = key;
    }
    wsync();
    // rank = position in ascending (key, index) order: a permutation
    for (int k = lane; k < deg; k += 64) {
      const double kk = s_key[k];
      int r = 0;
      for (int u = 0; u < deg; ++u) {
        const double ku = s_key[u];
        r += (ku < kk) || (ku == kk && u < k);
      }
      s_near[r] = S.knn_ids[k0 + k];
    }
    wsync();
  }
  for (int k = lane; k < deg; k += 64) {
    const double4 sm = S.site[ranked ? s_near[k] : S.knn_ids[k0 + k]];
    const rpd_d4 e = rpd_bisector(si, rpd_d4{sm.x, sm.y, sm.z, sm.w});
    const double nrm = sqrt(e.x * e.x + e.y * e.y + e.z * e.z);
    if (k < kBoxP - 6)  // the pushed bisector
      s_pl[6 + k] = make_double4(e.x, e.y, e.z, e.w + nrm * rho);
    float4 pl;
    rel_plane(e, si, sm, nrm, rho, dom, pl, rel_aux[k0 + k]);
    rel_pl[k0 + k] =
        make_float4(axis(pl.x, pl.y, pl.z, ax0), axis(pl.x, pl.y, pl.z, ax1),
                    axis(pl.x, pl.y, pl.z, ax2), pl.w);
  }
  // box planes: x >= x0, x <= x1, y >= y0, y <= y1, z >= z0, z <= z1
  if (lane < 6) {
    int a = lane >> 1;
    double4 p = make_double4(0, 0, 0, 0);
    double* pp = &p.x;
    if ((lane & 1) == 0) {
      pp[a] = 1.0;
      p.w = -dom[a];
    } else {
      pp[a] = -1.0;
      p.w = dom[3 + a];
    }
    s_pl[lane] = p;
  }
  wsync();
  rpd_d4 X[kVS];        // homogeneous, X.w >= 0
  uint32_t tr[kVS];
  uint64_t alive[kVS];
  auto set_vertex = [&](rpd_d4& Xq, uint32_t& trq, uint32_t a, uint32_t b,
                        uint32_t c) {
    rpd_d4 Y, Q;
    rpd_vertex_homog(ld4(&s_pl[a]), ld4(&s_pl[b]), ld4(&s_pl[c]), Y, Q);
    Xq = Y.w < 0 ? rpd_d4{-Y.x, -Y.y, -Y.z, -Y.w} : Y;
    trq = a | (b << 8) | (c << 16);
  };
#pragma unroll
  for (int q = 0; q < kVS; ++q) {
    X[q] = rpd_d4{0, 0, 0, 1};
    tr[q] = 0;
    alive[q] = q == 0 ? 0xffull : 0;
  }
  int nv = 8;
  if (lane < 8)
    set_vertex(X[0], tr[0], lane & 1, 2 + ((lane >> 1) & 1),
               4 + ((lane >> 2) & 1));
  bool empty = false;
  for (int k = 0; k < deg && !fail; ++k) {
    const uint32_t p = (uint32_t)(6 + k);
    const rpd_d4 e = ld4(&s_pl[p]);
    uint64_t gone[kVS];
    int n_out = 0;
#pragma unroll
    for (int q = 0; q < kVS; ++q) {
      const double s =
          e.x * X[q].x + e.y * X[q].y + e.z * X[q].z + e.w * X[q].w;
      gone[q] = ballot(s < 0 && X[q].w > 0) & alive[q];
      n_out += __popcll(gone[q]);
    }
    if (n_out == 0) continue;
    if (n_out == nv) {
      empty = true;
      break;
    }
    int n_new, n_edge;
    cut_edges<kVS>(tr, alive, gone, lane, s_new, n_new, n_edge);
    if (n_edge != 3 * n_out || nv - n_out + n_new > kBoxV) {
      fail = true;
      break;
    }
    wsync();
    int base = 0;  // the new vertices take the free slots
#pragma unroll
    for (int q = 0; q < kVS; ++q) {
      alive[q] &= ~gone[q];
      const uint64_t fr = ~alive[q];
      const int at = base + lanes_below(fr, lane);
      const bool take = ((fr >> lane) & 1) && at < n_new;
      if (take) {
        const uint32_t ab = s_new[at];
        set_vertex(X[q], tr[q], ab & 255, ab >> 8, p);
      }
      alive[q] |= ballot(take);
      base += __popcll(fr);
    }
    wsync();
    nv += n_new - n_out;
  }
  if (fail) {
    if (lane == 0) atomicAdd(n_fallback, 1);
    finish(dom);
    return;
  }
  if (empty) {
    finish(none);
    return;
  }
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
#pragma unroll
  for (int q = 0; q < kVS; ++q) {
    if (!((alive[q] >> lane) & 1)) continue;
    const double x = X[q].x / X[q].w, y = X[q].y / X[q].w,
                 z = X[q].z / X[q].w;
    lo[0] = fmin(lo[0], x);
    lo[1] = fmin(lo[1], y);
    lo[2] = fmin(lo[2], z);
    hi[0] = fmax(hi[0], x);
    hi[1] = fmax(hi[1], y);
    hi[2] = fmax(hi[2], z);
  }
  for (int off = 32; off > 0; off >>= 1)
    for (int a = 0; a < 3; ++a) {
      lo[a] = fmin(lo[a], __shfl_xor(lo[a], off));
      hi[a] = fmax(hi[a], __shfl_xor(hi[a], off));
    }
  const double ext =
      fmax(fmax(dom[3] - dom[0], dom[4] - dom[1]), dom[5] - dom[2]);
  const double eps = 1e-7 * ext;  // covers the rounding of the vertices
  const double b[6] = {lo[0] - eps, lo[1] - eps, lo[2] - eps,
                       hi[0] + eps, hi[1] + eps, hi[2] + eps};
  finish(b);
}

// bin_start[b] = first key of bin >= b in the sorted keys (sphere grid)
__global__ __launch_bounds__(256) void k_bin_starts(int64_t n_bins,
                                                    int64_t n_reg_cap,
                                                    const uint64_t* keys,
                                                    int32_t* bin_start,
                                                    int32_t* bin_ids,
                                                    const int64_t* n_reg_dev) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t n_reg = dev_count(n_reg_cap, n_reg_dev);
  if (b < n_reg) bin_ids[b] = (int32_t)(keys[b] & 0xffffffffu);
  if (b > n_bins) return;
  int64_t lo = 0, hi = n_reg;  // first index with key >> 32 >= b
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)(keys[mid] >> 32) < b)
      lo = mid + 1;
    else
      hi = mid;
  }
  bin_start[b] = (int32_t)lo;
}

struct TetLoad {
  double4 V[4];
  int4 tv;
};

__device__ __forceinline__ void load_tet(const DevMesh& M, int t,
                                         TetLoad& L) {
  L.tv = M.tet_v[t];
  L.V[0] = M.vert[L.tv.x];
  L.V[1] = M.vert[L.tv.y];
  L.V[2] = M.vert[L.tv.z];
  L.V[3] = M.vert[L.tv.w];
}

// reference relation test (voronoi.cu:154-193) in binary64: sphere i
// relates to the tet iff for every neighbour m some corner v has
// pd(v, m) > pd(v, i).  The neighbours are visited nearest bisector first
// (the outcome does not depend on the order), their spheres read inline,
// one ahead.
__device__ __forceinline__ bool relation(const DevSites& S, const TetLoad& L,
                                         int i) {
  if (S.flags[i] != 1u) return false;
  const rpd_d4 si = ld4(S.site + i);
  double pdi[4];
  for (int k = 0; k < 4; ++k)
    pdi[k] = rpd_power_dist(L.V[k].x, L.V[k].y, L.V[k].z, si);
  const int64_t k0 = S.knn_off[i], k1 = S.knn_off[i + 1];
  if (k0 == k1) return true;
  double4 nxt = S.knn_site_near[k0];
  for (int64_t q = k0; q < k1; ++q) {
    const rpd_d4 sm{nxt.x, nxt.y, nxt.z, nxt.w};
    if (q + 1 < k1) nxt = S.knn_site_near[q + 1];
    bool ok = false;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      ok = ok || rpd_power_dist(L.V[k].x, L.V[k].y, L.V[k].z, sm) > pdi[k];
    if (!ok) return false;
  }
  return true;
}

__device__ __forceinline__ void tet_centroid(const TetLoad& L, double c[3]) {
  c[0] = (((L.V[0].x + L.V[1].x) + L.V[2].x) + L.V[3].x) * 0.25;
  c[1] = (((L.V[0].y + L.V[1].y) + L.V[2].y) + L.V[3].y) * 0.25;
  c[2] = (((L.V[0].z + L.V[1].z) + L.V[2].z) + L.V[3].z) * 0.25;
}

__device__ __forceinline__ int64_t tet_bin(const double c[3],
                                           const BinGrid& g) {
  int x = bin_coord(c[0], g.org[0], g.inv_bs, g.dim[0]);
  int y = bin_coord(c[1], g.org[1], g.inv_bs, g.dim[1]);
  int z = bin_coord(c[2], g.org[2], g.inv_bs, g.dim[2]);
  return x + (int64_t)g.dim[0] * (y + (int64_t)g.dim[1] * z);
}

// The tets in grid order: bin b (its x fastest, then y, then z) holds
// positions [first[b], first[b + 1]); per position the tet and its corners,
// binary32 about the centre of the domain box, in the grid's axes: (x0 y0 z0
// x1), (y1 z1 x2 y2), (z2 x3 y3 z3).
struct MeshBins {
  const int32_t* first;
  const int32_t* tet;
  const float4* c0;
  const float4* c1;
  const float4* c2;
};

// bin of every (selected) tet and its rank there; bin_n was cleared.  The
// ranks follow the atomics' order, which nothing depends on.
__global__ __launch_bounds__(256) void k_tet_bin(DevMesh M,
                                                 const InstInfo* inst,
                                                 const int32_t* tet_inst,
                                                 const uint8_t* tet_sel,
                                                 int32_t* bin_n,
                                                 int2* tet_bin_rank) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= M.n_tet || (tet_sel && !tet_sel[t])) return;
  TetLoad L;
  load_tet(M, t, L);
  double m[3];
  tet_centroid(L, m);
  const InstInfo& I = inst[tet_inst[t]];
  const double c[3] = {axis(m[0], m[1], m[2], I.ax[0]),
                       axis(m[0], m[1], m[2], I.ax[1]),
                       axis(m[0], m[1], m[2], I.ax[2])};
  const int32_t b = (int32_t)(I.bin_base + tet_bin(c, I.g));
  tet_bin_rank[t] = make_int2(b, atomicAdd(bin_n + b, 1));
}

__global__ __launch_bounds__(256) void k_tet_bin_fill(
    DevMesh M, const InstInfo* inst, const int32_t* tet_inst,
    const uint8_t* tet_sel, const int2* tet_bin_rank, const int32_t* first,
    int32_t* tet, float4* c0, float4* c1, float4* c2) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= M.n_tet || (tet_sel && !tet_sel[t])) return;
  const int2 br = tet_bin_rank[t];
  const int32_t p = first[br.x] + br.y;
  TetLoad L;
  load_tet(M, t, L);
  const InstInfo& I = inst[tet_inst[t]];
  float v[12];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double c = 0.5 * (I.gdom[a] + I.gdom[3 + a]);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      v[3 * k + a] =
          (float)(axis(L.V[k].x, L.V[k].y, L.V[k].z, I.ax[a]) - c);
  }
  tet[p] = t;
  c0[p] = make_float4(v[0], v[1], v[2], v[3]);
  c1[p] = make_float4(v[4], v[5], v[6], v[7]);
  c2[p] = make_float4(v[8], v[9], v[10], v[11]);
}

// the relation in binary64 over the neighbour list as it is (for the few
// pairs that the binary32 planes leave open)
__device__ __noinline__ bool relation_exact(const DevMesh& M,
                                            const DevSites& S, int t, int i) {
  TetLoad L;
  load_tet(M, t, L);
  const rpd_d4 si = ld4(S.site + i);
  double pdi[4];
  for (int k = 0; k < 4; ++k)
    pdi[k] = rpd_power_dist(L.V[k].x, L.V[k].y, L.V[k].z, si);
  for (int64_t q = S.knn_off[i]; q < S.knn_off[i + 1]; ++q) {
    const rpd_d4 sm = ld4(S.site + S.knn_ids[q]);
    bool ok = false;
    for (int k = 0; k < 4; ++k)
      ok = ok || rpd_power_dist(L.V[k].x, L.V[k].y, L.V[k].z, sm) > pdi[k];
    if (!ok) return false;
  }
  return true;
}

// Tet-sphere relation (voronoi.cu:154-193), sphere by sphere: a tet is
// related to sphere i iff every neighbour's bisector leaves one of its
// corners on i's side.  A wavefront takes a part of the sphere's box
// (kPartTets): the lanes of a row (y, z), four of them for each of kRelRows
// rows, bound the x range that the pushed planes leave of it; the tets of the
// ranges are then tested 64 at a time,
// their corners read contiguously, the planes read from LDS by all lanes at
// once, nearest first, until no lane is left.  Values within a plane's error
// bound leave a pair open, and relation_exact decides it.
//
// Bound by instruction issue (18 per plane and 64 tets).  One thread per tet
// over the spheres registered in its bin, in binary64, was bound by the
// divergence of 64 different lists and, on small meshes, by their length:
// 1.57 M tets, 18,000 sites: binning, counting and filling 2.6 ms, this
// with the pair lists 0.64 ms; 16 instances of 2,000 to 200,000 tets with up
// to 20,000 sites (bin lists past 128, tested twice) 11.7 -> 0.57 ms; 6,000
// tets 0.55 -> 0.03 ms.
//
// Related pairs are counted per tet (nothing waits for these atomics) and go
// to an unordered list.  A wavefront takes list entries in chunks (one atomic
// at one address for 64 pairs took 2.0 ms of 2.5 at 3.5 M pairs) and marks
// what it leaves of its last one.
constexpr int kRelPl = 128;
__global__ __launch_bounds__(64) void k_rel_pairs(
    DevMesh M, DevSites S, MeshBins B, const InstInfo* inst,
    const int32_t* site_inst, const double* bbox, const float4* rel_pl,
    const float2* rel_aux, const int64_t* part_off, const int32_t* part_rows,
    unsigned long long* tet_count, int2* pairs, uint32_t* n_pairs,
    uint32_t chunk, int64_t cap, unsigned long long* work) {
  __shared__ float4 s_pl[kRelPl];
  __shared__ float2 s_aux[kRelPl];
  __shared__ int32_t s_first[kRelRows];
  __shared__ int32_t s_pref[kRelRows + 1];
  const int lane = threadIdx.x;
  const int n_site = S.n_site;
  const int64_t n_parts = part_off[n_site];
  uint32_t pos = 0, end = 0;  // the rest of this wavefront's chunk
  for (int64_t part = blockIdx.x; part < n_parts; part += gridDim.x) {
    // the sphere: part_off[i] <= part < part_off[i + 1]
    int i = 0, hi = n_site;
    while (hi - i > 1) {
      const int step = (hi - i + 63) / 64;
      const int at = i + lane * step;
      const uint64_t le = ballot(at < hi && part_off[at] <= part);
      i += (63 - __clzll((long long)le)) * step;  // lane 0 always holds
      hi = min(hi, i + step);
    }
    const InstInfo& I = inst[site_inst[i]];
    const BinGrid& g = I.g;
    const int64_t k0 = S.knn_off[i];
    const int deg = (int)(S.knn_off[i + 1] - k0);
    const int np = min(deg, kRelPl);
    wsync();
    for (int k = lane; k < ((np + 3) & ~3); k += 64) {
      s_pl[k] = k < np ? rel_pl[k0 + k] : make_float4(0, 0, 0, 1);
      s_aux[k] = k < np ? rel_aux[k0 + k] : make_float2(0, 0);
    }
    wsync();
    int r[6];
    bin_range(bbox + 6 * (int64_t)i, g, r);
#pragma unroll
    for (int a = 0; a < 6; ++a) r[a] = __builtin_amdgcn_readfirstlane(r[a]);
    int rows = (r[4] - r[1] + 1) * (r[5] - r[2] + 1);
    const int per = __builtin_amdgcn_readfirstlane(part_rows[i]);
    int row0 = __builtin_amdgcn_readfirstlane((int)(part - part_off[i]));
    uint32_t acc = 0, t0 = 0;  // by count: before row0, before the part
    if (per > 0) {
      row0 *= per;
      rows = min(rows, row0 + per);
    } else {  // the row that holds t0
      t0 = (uint32_t)row0 * kPartTets;
      row0 = 0;
      while (t0 > 0 && row0 < rows) {
        int f0;
        uint32_t n = 0;
        if (row0 + lane < rows)
          n = max(kRowTets,
                  row_tets(B.first, I.bin_base, g, r, row0 + lane, f0));
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const uint32_t v = __shfl_up(n, off);
          if (lane >= off) n += v;
        }
        const int skip = __popcll(ballot(acc + n <= t0));
        if (skip > 0) acc += lane_value(n, skip - 1);
        row0 += skip;
        if (skip < 64) break;
      }
    }
    uint32_t tests = 0, tested = 0;
    for (; row0 < rows && acc < t0 + kPartTets; row0 += kRelRows) {
      const int row = row0 + (lane & (kRelRows - 1));
      int len = 0, f_lo = 0, p_lo = 0, p_hi = row < rows ? 0x7fffffff : 0;
      if (per == 0) {  // the part's share of the row: positions [p_lo, p_hi)
        uint32_t pre = 0;  // count up to this row
        if (row < rows) {
          p_hi = row_tets(B.first, I.bin_base, g, r, row, p_lo);
          pre = max(kRowTets, p_hi);
        }
        const uint32_t w_row = pre;
#pragma unroll
        for (int off = 1; off < kRelRows; off <<= 1) {
          const uint32_t v = __shfl_up(pre, off);
          if ((lane & (kRelRows - 1)) >= off) pre += v;
        }
        const int at = (int)(t0 - (acc + pre - w_row));
        p_hi = p_lo + min(p_hi, at + kPartTets);
        p_lo += max(0, at);
        acc += lane_value(pre, kRelRows - 1);
      }
      if (p_lo < p_hi) {
        const int ny = r[4] - r[1] + 1;
        const int y = r[1] + row % ny, z = r[2] + row / ny;
        // the row's box about the domain centre (the last bin of a capped
        // grid reaches to the end of the domain), 1e-6 of a bin wider
        const double bs = 1.0 / g.inv_bs;
        double o[3];
        for (int a = 0; a < 3; ++a)
          o[a] = g.org[a] - 0.5 * (I.gdom[a] + I.gdom[3 + a]);
        const float ylo = (float)(o[1] + (y - 1e-6) * bs);
        const float yhi = (float)(y == g.dim[1] - 1
                                      ? 0.500001 * (I.gdom[4] - I.gdom[1]) +
                                            1e-6 * bs
                                      : o[1] + (y + 1 + 1e-6) * bs);
        const float zlo = (float)(o[2] + (z - 1e-6) * bs);
        const float zhi = (float)(z == g.dim[2] - 1
                                      ? 0.500001 * (I.gdom[5] - I.gdom[2]) +
                                            1e-6 * bs
                                      : o[2] + (z + 1 + 1e-6) * bs);
        float xlo = -INFINITY, xhi = INFINITY;
        for (int k = lane / kRelRows; k < np; k += 64 / kRelRows) {
          const float4 p = s_pl[k];
          const float2 q = s_aux[k];
          // p.x x + t >= 0 for some point of the row, or no tet there relates
          const float t = (p.w + q.y + q.x) + fmaxf(p.y * ylo, p.y * yhi) +
                          fmaxf(p.z * zlo, p.z * zhi) + q.x;
          const float x = -t / p.x;
          if (p.x > 0)
            xlo = fmaxf(xlo, x);
          else if (p.x < 0)
            xhi = fminf(xhi, x);
          else if (t < 0)
            xhi = -INFINITY;
        }
  #pragma unroll
        for (int off = kRelRows; off < 64; off <<= 1) {
          xlo = fmaxf(xlo, __shfl_xor(xlo, off));
          xhi = fminf(xhi, __shfl_xor(xhi, off));
        }
        // bins of [xlo, xhi], with 1e-3 of a bin for the rounding
        const float inv = (float)g.inv_bs, ox = (float)o[0];
        const float flo = (xlo - ox) * inv - 1e-3f;
        const float fhi = (xhi - ox) * inv + 1e-3f;
        // (a bound that is not a number narrows nothing)
        const float last = (float)(g.dim[0] - 1);
        const int a =
            flo > 0.f ? max(r[0], (int)fminf(floorf(flo), last)) : r[0];
        const int b =
            fhi < last ? min(r[3], (int)fmaxf(floorf(fhi), -1.f)) : r[3];
        if (a <= b) {
          const int64_t base =
              I.bin_base + (int64_t)g.dim[0] * (y + (int64_t)g.dim[1] * z);
          f_lo = max(p_lo, B.first[base + a]);
          len = max(0, min(p_hi, B.first[base + b + 1]) - f_lo);
        }
      }
      // tets to test before each row of the part
      wsync();
      if (lane < kRelRows) s_first[lane] = f_lo;
      int pre = len;
  #pragma unroll
      for (int off = 1; off < kRelRows; off <<= 1) {
        const int v = __shfl_up(pre, off);
        if ((lane & (kRelRows - 1)) >= off) pre += v;
      }
      if (lane < kRelRows) s_pref[lane + 1] = pre;
      if (lane == 0) s_pref[0] = 0;
      wsync();
      const int total = s_pref[kRelRows];
      tested += total;
      for (int f0 = 0; f0 < total; f0 += 64) {
        const int f = f0 + lane;
        int q = 0;  // the row: s_pref[q] <= f < s_pref[q + 1]
  #pragma unroll
        for (int w = kRelRows / 2; w > 0; w >>= 1)
          if (s_pref[q + w] <= f) q += w;
        bool in = f < total, open = deg > kRelPl;
        const int at = in ? s_first[q] + (f - s_pref[q]) : 0;
        float4 c0 = make_float4(0, 0, 0, 0), c1 = c0, c2 = c0;
        int t = 0;
        if (in) {
          t = B.tet[at];
          c0 = B.c0[at];
          c1 = B.c1[at];
          c2 = B.c2[at];
        }
        int k = 0;
        auto plane = [&](const float4& p, float eps) {
          auto at = [&](float x, float y, float z) {
            return fmaf(p.z, z, fmaf(p.y, y, fmaf(p.x, x, p.w)));
          };
          const float v0 = at(c0.x, c0.y, c0.z), v1 = at(c0.w, c1.x, c1.y);
          const float v2 = at(c1.z, c1.w, c2.x), v3 = at(c2.y, c2.z, c2.w);
          const float v = fmaxf(fmaxf(v0, v1), fmaxf(v2, v3));
          in = in && !(v < -eps);
          open = open || !(v > eps);
        };
        // four planes between two looks at the lanes left (their LDS reads
        // overlap); the list is padded with planes that every point passes
        for (; k < np && ballot(in) != 0; k += 4) {
          const float4 p0 = s_pl[k], p1 = s_pl[k + 1], p2 = s_pl[k + 2],
                       p3 = s_pl[k + 3];
          const float e0 = s_aux[k].x, e1 = s_aux[k + 1].x, e2 = s_aux[k + 2].x,
                      e3 = s_aux[k + 3].x;
          plane(p0, e0);
          plane(p1, e1);
          plane(p2, e2);
          plane(p3, e3);
        }
        tests += k;
        if (ballot(in && open) != 0)
          if (in && open) in = relation_exact(M, S, t, i);
        const uint64_t m = ballot(in);
        if (m != 0) {
          const uint32_t n = (uint32_t)__popcll(m), rest = end - pos;
          uint32_t next = 0;  // a new chunk for what the old one can't hold
          if (n > rest) {
            if (lane == 0) next = atomicAdd(n_pairs, chunk);
            next = lane_value(next, 0);
          }
          if (in) {
            const uint32_t w = (uint32_t)lanes_below(m, lane);
            const int64_t at = w < rest ? pos + w : next + (w - rest);
            atomicAdd(tet_count + t, 1ull);
            if (at < cap) pairs[at] = make_int2(t, i);
          }
          if (n > rest) {
            pos = next + (n - rest);
            end = next + chunk;
          } else {
            pos += n;
          }
        }
      }
    }
    if (work && lane == 0) {  // pairs tested, plane tests (count_work)
      unsigned long long* w = work + 4 * (blockIdx.x & 63);
      atomicAdd(w + 0, (unsigned long long)tested);
      atomicAdd(w + 1, (unsigned long long)tests * 64);
    }
    wsync();
  }
  for (int64_t q = (int64_t)pos + lane; q < end; q += 64)
    if (q < cap) pairs[q] = make_int2(-1, -1);
}

// A captured run whose pairs do not fit their list: no pairs at all, and
// the overflow flag (no later kernel may read an entry that was not written)
__global__ __launch_bounds__(256) void k_rel_guard(int32_t n_tet,
                                                   const uint32_t* n_pairs,
                                                   int64_t cap,
                                                   unsigned long long* count,
                                                   int32_t* overflow) {
  // (the list's room past the captured candidates is the chunks' slack, so
  // more candidates than captured can fit it: the host sees their count)
  if ((int64_t)*n_pairs <= cap) return;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n_tet) count[t] = 0;
  if (t == 0) overflow[0] = 1;
}

// pairs to their tet's segment, in the order of the atomics (k_pair_rank
// sorts it away)
__global__ __launch_bounds__(256) void k_pair_place(
    int64_t room, int64_t cap, const uint32_t* n_pairs, const int2* pairs,
    const int64_t* tet_off, int32_t* tet_fill, int2* seg) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t n = (int64_t)*n_pairs;
  if (n > room || q >= n) return;
  const int2 p = pairs[q];
  if (p.x < 0) return;
  const int64_t at = tet_off[p.x] + atomicAdd(tet_fill + p.x, 1);
  if (at < cap) seg[at] = p;
}

// candidates in tet order, ascending sites: each pair's place is the number
// of smaller sites in its segment
__global__ __launch_bounds__(256) void k_pair_rank(
    int64_t cap, int32_t n_tet, const int2* seg, const int64_t* tet_off,
    Cand* cand, int32_t* rel_ids) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= min(cap, tet_off[n_tet])) return;
  const int2 p = seg[q];
  const int64_t o0 = tet_off[p.x], o1 = min(cap, tet_off[p.x + 1]);
  int64_t at = o0;
  for (int64_t o = o0; o < o1; ++o) at += seg[o].y < p.y;
  Cand c;
  c.tet = p.x;
  c.seed = p.y;
  c.m0 = 0;
  c.m1 = 0;
  cand[at] = c;
  rel_ids[at] = p.y;
}

// the bisector table of the neighbour lists: one wavefront per site
__global__ __launch_bounds__(64) void k_knn_bis(DevSites S, double4* bis,
                                                float4* bisf) {
  const int i = blockIdx.x;
  const int64_t k0 = S.knn_off[i], k1 = S.knn_off[i + 1];
  const rpd_d4 si = ld4(S.site + i);
  for (int64_t q = k0 + threadIdx.x; q < k1; q += 64) {
    const int m = S.knn_ids[q];
    double4 e = make_double4(0, 0, 0, 0);
    if (m >= 0) {
      const rpd_d4 b = rpd_bisector(si, ld4(S.site + m));
      e = make_double4(b.x, b.y, b.z, b.w);
    }
    bis[q] = e;
    bisf[q] = make_float4(rpd_mask_coef(e.x), rpd_mask_coef(e.y),
                          rpd_mask_coef(e.z), rpd_mask_coef(e.w));
  }
}

// The tet's four corners as the clip kernel's initial vertices: homogeneous
// coordinates X and cofactor magnitudes Q of the dual triangles (1,3,2),
// (0,2,3), (0,3,1), (0,1,2) of its binary64 face planes; sQ = the sum of
// a corner's four magnitudes.
struct CornerFrames {
  rpd_d4 X[4];
  double sQ[4];
  // dot(e, X~) is certainly negative (no conflict) at all four corners, so
  // the plane e cannot cut any state of a cell of this tet (every vertex of
  // the cell lies in the convex hull of the corners); decided from the
  // binary32 table entry f of e (rpd_mask_negative), one 16-byte load per
  // plane.  The few planes it leaves undecided that a tighter test would
  // skip are only clipped without effect.
  __device__ __forceinline__ bool inactive(const float4& f) const {
    return rpd_mask_negative(f.x, f.y, f.z, f.w, X, sQ);
  }
};
__device__ __forceinline__ void corner_frames(const TetLoad& L,
                                              CornerFrames& F) {
  rpd_d4 pl[4], Q[4];
  tet_planes(L.V, pl);
  rpd_vertex_homog(pl[1], pl[3], pl[2], F.X[0], Q[0]);
  rpd_vertex_homog(pl[0], pl[2], pl[3], F.X[1], Q[1]);
  rpd_vertex_homog(pl[0], pl[3], pl[1], F.X[2], Q[2]);
  rpd_vertex_homog(pl[0], pl[1], pl[2], F.X[3], Q[3]);
#pragma unroll
  for (int k = 0; k < 4; ++k) F.sQ[k] = ((Q[k].x + Q[k].y) + Q[k].z) + Q[k].w;
}
// a cell's number of clip steps: mask bits, plus the list positions past
// 128 (always clipped), saturated to a byte
__device__ __forceinline__ uint8_t clip_steps(uint64_t m0, uint64_t m1,
                                              int deg) {
  const int n = __popcll(m0) + __popcll(m1) + (deg > 128 ? deg - 128 : 0);
  return (uint8_t)(n < 255 ? n : 255);
}

// One thread per candidate cell: bit k of the mask is set unless the k-th
// neighbour's bisector is certainly positive at all four corners of the
// tet cell (then it cannot cut any state of the cell: every cell vertex
// lies in the convex hull of the corners).
// With trips != nullptr it also writes each cell's number of clip steps
// (mask bits below the degree, plus the positions past 128) and its index
// c0 + c for the step-count ordering of the clip launch.
__global__ __launch_bounds__(256) void k_cand_mask(DevMesh M, DevSites S,
                                                   int64_t n_cand,
                                                   Cand* cand,
                                                   uint8_t* trips,
                                                   int32_t* trip_ids,
                                                   int64_t c0,
                                                   const int64_t* n_dev) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n_cand) return;
  if (n_dev && c >= dev_count(n_cand, n_dev, c0)) {
    if (trips) {  // past the count: sorts after every cell
      trips[c] = 0;
      trip_ids[c] = (int32_t)(c0 + c);
    }
    return;
  }
  const int t = cand[c].tet, i = cand[c].seed;
  TetLoad L;
  load_tet(M, t, L);
  CornerFrames F;
  corner_frames(L, F);
  const int64_t k0 = S.knn_off[i];
  const int deg = (int)(S.knn_off[i + 1] - k0);
  uint64_t m0 = 0, m1 = 0;
  const int lim = deg < 128 ? deg : 128;
  // the next plane's load is issued before this plane's test (the test's
  // corner branches keep the compiler from hoisting it)
  float4 nxt = lim > 0 ? S.knn_bisf[k0] : make_float4(0, 0, 0, 0);
  for (int k = 0; k < lim; ++k) {
    const float4 f = nxt;
    if (k + 1 < lim) nxt = S.knn_bisf[k0 + k + 1];
    if (!F.inactive(f)) {
      if (k < 64)
        m0 |= 1ull << k;
      else
        m1 |= 1ull << (k - 64);
    }
  }
  cand[c].m0 = m0;
  cand[c].m1 = m1;
  if (trips) {
    trips[c] = clip_steps(m0, m1, deg);
    trip_ids[c] = (int32_t)(c0 + c);
  }
}

// ========================================================== compaction
// per cell: location of its final slot; tier 0 small (index = cell),
// tier 1 large / 2 exact (index = re-run position)
__global__ __launch_bounds__(256) void k_mark_rerun(const int32_t* list,
                                                    int32_t r0, int32_t r1,
                                                    int32_t tier,
                                                    int32_t* loc,
                                                    const int32_t* r1_dev) {
  const int r = r0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= (r1_dev ? min(r1, *r1_dev) : r1)) return;
  loc[list[r]] = (tier << 28) | r;
}

struct Sizes3 {
  int64_t cells, words, areas;
};
struct Sizes3Sum {
  __host__ __device__ Sizes3 operator()(const Sizes3& a,
                                        const Sizes3& b) const {
    return Sizes3{a.cells + b.cells, a.words + b.words, a.areas + b.areas};
  }
};

struct TierViews {
  SlotView t[4];  // small, full capacity, exact, middle
};

// Compaction in blocks of kCB consecutive output positions r (cell
// perm[r], or r when perm is null).  A cell's sizes pack into one u64
// (cells in bits 0-15, areas 16-35, words 36-63), so one integer sum
// scans all three: a block holds at most 256 cells, 256 x 64 areas and
// 256 x 312 words.
constexpr int kCB = 256;

struct CellRef {
  int tier;
  int64_t idx;
  uint32_t hdr;
};

__device__ __forceinline__ CellRef cell_ref(int64_t r, const int32_t* perm,
                                            const int32_t* loc,
                                            const TierViews& tv) {
  const int64_t c = perm ? perm[r] : r;
  const int32_t l = loc[c];
  CellRef x;
  x.tier = l >> 28;
  x.idx = x.tier ? (l & ((1 << 28) - 1)) : c;
  x.hdr = tv.t[x.tier].hdr[x.idx];
  return x;
}

__device__ __forceinline__ uint64_t packed_size(uint32_t hd) {
  if ((hd >> 24) != RPD_SUCCESS) return 0;
  const uint64_t nv = hd & 255, np = (hd >> 8) & 255, ne = (hd >> 16) & 255;
  return 1ull | (np << 16) | ((nv + np + ne) << 36);
}

// per block: totals of its cells (bsum[b]) and the dropped cells by status
// per-status counts of the cells not emitted, spread over kDropSlots copies
// of the 9 counters (a block adds to copy blockIdx % kDropSlots) so that
// the blocks' atomics do not all meet at one address
constexpr int kDropSlots = 64;
__global__ __launch_bounds__(kCB) void k_block_sizes(int64_t n_cells,
                                                     const int32_t* perm,
                                                     const int32_t* loc,
                                                     TierViews tv,
                                                     Sizes3* bsum,
                                                     int64_t* drops,
                                                     const int64_t* n_dev) {
  typedef hipcub::BlockReduce<uint64_t, kCB> Red;
  n_cells = dev_count(n_cells, n_dev);
  __shared__ typename Red::TempStorage tmp;
  __shared__ int32_t h[9];
  if (threadIdx.x < 9) h[threadIdx.x] = 0;
  __syncthreads();
  const int64_t r = (int64_t)blockIdx.x * kCB + threadIdx.x;
  uint64_t z = 0;
  if (r < n_cells) {
    const CellRef x = cell_ref(r, perm, loc, tv);
    const uint32_t st = x.hdr >> 24;
    z = packed_size(x.hdr);
    if (st != RPD_SUCCESS && st < 9) atomicAdd(&h[st], 1);
  }
  const uint64_t tot = Red(tmp).Sum(z);
  if (threadIdx.x == 0)
    bsum[blockIdx.x] = Sizes3{(int64_t)(tot & 0xffff),
                              (int64_t)(tot >> 36),
                              (int64_t)((tot >> 16) & 0xfffff)};
  __syncthreads();
  if (threadIdx.x < 9 && h[threadIdx.x])
    atomicAdd((unsigned long long*)&drops[9 * (blockIdx.x % kDropSlots) +
                                          threadIdx.x],
              (unsigned long long)h[threadIdx.x]);
}

// block b writes its cells from boff[b] on: cell records and geometry one
// per thread, payload words and areas by the whole block over the block's
// contiguous output range (each output element finds its cell by binary
// search in the block's offsets), so every store is coalesced.
__global__ __launch_bounds__(kCB) void k_compact(
    int64_t n_cells, const int32_t* perm, const Cand* cand,
    const int32_t* loc, TierViews tv, const Sizes3* boff, rpd_cell* out_cells,
    uint32_t* out_words, double* out_geom, double* out_areas,
    int32_t geometry, const int64_t* n_dev, Sizes3 cap, int32_t* overflow) {
  typedef hipcub::BlockScan<uint64_t, kCB> Scan;
  __shared__ typename Scan::TempStorage tmp;
  __shared__ uint32_t s_w[kCB + 1];
  __shared__ uint32_t s_a[kCB + 1];
  __shared__ const uint32_t* s_wsrc[kCB];
  __shared__ const double* s_asrc[kCB];
  // a slot holds the edges at 0 and the vertices and plane sources after
  // them; the stream holds vertices, plane sources, edges
  __shared__ uint32_t s_lay[kCB];  // nb_v | nb_p << 8 | nb_e << 16
  const int i = threadIdx.x;
  const int64_t r = (int64_t)blockIdx.x * kCB + i;
  n_cells = dev_count(n_cells, n_dev);
  {  // a captured pipeline's output capacity: the block's whole range
    const Sizes3 B0 = boff[blockIdx.x], B1 = boff[blockIdx.x + 1];
    if (B1.cells > cap.cells || B1.words > cap.words ||
        B1.areas > cap.areas) {
      if (i == 0) overflow[0] = 1;
      return;
    }
    (void)B0;
  }
  CellRef x{0, 0, 0};
  int64_t c = 0;
  uint64_t z = 0;
  if (r < n_cells) {
    c = perm ? perm[r] : r;
    x = cell_ref(r, perm, loc, tv);
    z = packed_size(x.hdr);
  }
  uint64_t off, tot;
  Scan(tmp).ExclusiveSum(z, off, tot);
  const Sizes3 B = boff[blockIdx.x];
  const uint32_t w_off = (uint32_t)(off >> 36);
  const uint32_t a_off = (uint32_t)((off >> 16) & 0xfffff);
  const int64_t c_off = B.cells + (int64_t)(off & 0xffff);
  s_w[i] = w_off;
  s_a[i] = a_off;
  if (i == 0) {
    s_w[kCB] = (uint32_t)(tot >> 36);
    s_a[kCB] = (uint32_t)((tot >> 16) & 0xfffff);
  }
  const SlotView& sv = tv.t[x.tier];
  s_wsrc[i] = sv.words + x.idx * sv.stride_words;
  s_asrc[i] = sv.areas + x.idx * sv.stride_areas;
  s_lay[i] = x.hdr & 0xffffffu;
  if (z) {
    rpd_cell rc;
    rc.tet_id = cand[c].tet;
    rc.seed = cand[c].seed;
    rc.nb_v = (uint8_t)(x.hdr & 255);
    rc.nb_p = (uint8_t)((x.hdr >> 8) & 255);
    rc.nb_e = (uint8_t)((x.hdr >> 16) & 255);
    rc.status = RPD_SUCCESS;
    rc.reserved = 0;
    rc.word_off = (uint64_t)(B.words + w_off);
    rc.area_off = (uint64_t)(B.areas + a_off);
    out_cells[c_off] = rc;
    if (geometry) {
      const double* gs = sv.geom + 4 * x.idx;
      double* gd = out_geom + 4 * c_off;
      gd[0] = gs[0];
      gd[1] = gs[1];
      gd[2] = gs[2];
      gd[3] = gs[3];
    }
  }
  __syncthreads();
  // the cell holding element e: the last k with s[k] <= e (cells without
  // output have s[k] == s[k + 1] and are skipped by "last")
  auto owner = [](const uint32_t* sa, uint32_t e) {
    int lo = 0, hi = kCB;  // sa[lo] <= e < sa[hi]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (sa[mid] <= e)
        lo = mid;
      else
        hi = mid;
    }
    return lo;
  };
  // Each wavefront copies a contiguous quarter of the block's elements, 64
  // consecutive ones per step (coalesced stores); a lane finds the cell of
  // its first element by binary search and then walks forward, past about
  // 64 / (elements per cell) cells a step.  kU steps at a time: their
  // sources first, then their loads together, then their stores.
  constexpr int kU = 4;
  const int wv = i >> 6, ln = i & 63;
  auto range = [&](uint32_t n, uint32_t* q0, uint32_t* q1) {
    *q0 = (uint32_t)((uint64_t)n * wv / (kCB / 64));
    *q1 = (uint32_t)((uint64_t)n * (wv + 1) / (kCB / 64));
  };
  const uint32_t W = s_w[kCB];
  uint32_t* wd = out_words + B.words;
  {
    uint32_t q0, q1;
    range(W, &q0, &q1);
    int k = q0 + ln < q1 ? owner(s_w, q0 + ln) : 0;
    for (uint32_t e0 = q0 + ln; e0 < q1; e0 += 64 * kU) {
      const uint32_t* src[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const uint32_t e = e0 + 64 * u;
        src[u] = nullptr;
        if (e < q1) {
          while (s_w[k + 1] <= e) ++k;
          const uint32_t w = e - s_w[k], lay = s_lay[k];
          const uint32_t nvp = (lay & 255) + ((lay >> 8) & 255);
          src[u] = s_wsrc[k] + (w < nvp ? (lay >> 16) + w : w - nvp);
        }
      }
      uint32_t v[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) v[u] = src[u] ? *src[u] : 0u;
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (src[u]) wd[e0 + 64 * u] = v[u];
    }
  }
  if (geometry) {
    const uint32_t A = s_a[kCB];
    double* ad = out_areas + B.areas;
    uint32_t q0, q1;
    range(A, &q0, &q1);
    int k = q0 + ln < q1 ? owner(s_a, q0 + ln) : 0;
    for (uint32_t e0 = q0 + ln; e0 < q1; e0 += 64 * kU) {
      const double* src[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const uint32_t e = e0 + 64 * u;
        src[u] = nullptr;
        if (e < q1) {
          while (s_a[k + 1] <= e) ++k;
          src[u] = s_asrc[k] + (e - s_a[k]);
        }
      }
      double v[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) v[u] = src[u] ? *src[u] : 0.0;
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (src[u]) ad[e0 + 64 * u] = v[u];
    }
  }
}

// active-plane statistics of the candidate masks
__global__ __launch_bounds__(256) void k_mask_stats(int64_t n, const Cand* cand,
                                                    DevSites S,
                                                    unsigned long long* acc) {
  __shared__ unsigned long long s_a, s_b;
  if (threadIdx.x == 0) s_a = s_b = 0;
  __syncthreads();
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c < n) {
    const Cand cd = cand[c];
    const int64_t deg = S.knn_off[cd.seed + 1] - S.knn_off[cd.seed];
    int64_t act = __popcll(cd.m0) + __popcll(cd.m1);
    if (deg > 128) act += deg - 128;
    atomicAdd(&s_a, (unsigned long long)act);
    atomicAdd(&s_b, (unsigned long long)deg);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    atomicAdd(&acc[0], s_a);
    atomicAdd(&acc[1], s_b);
  }
}

}  // namespace rpd
