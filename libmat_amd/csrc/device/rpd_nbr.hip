// Regular-triangulation neighbours of a sphere set on the device: the
// power cell of every sphere inside the domain box, clipped by the power
// bisectors of the spheres that can reach it, with exact signs (filtered
// dot product of the plane with the vertex's homogeneous coordinates, exact
// expansion fallback).  A sphere is valid (not hidden) iff its cell is not
// empty; its neighbours are the spheres whose bisector carries a face of
// the cell.  This is the restatement of the reference's CGAL regular
// triangulation step (triangulation.cxx:62-144, get_RT_neighbors_given_
// spheres :396-438) that the host builder rpd_power_neighbors computes.
// Lists that are their own symmetric closure (k_nbr_check) are packed on the
// device; where bisectors meet in one point they may not be, and the host
// closes them (rpd_nbr_from_lists).
//
// Candidates come from weight-class grids (rpd_classgrid.h): class by
// class, shells of grid cells at Chebyshev distance r around the sphere's
// cell, until no sphere of the class can reach the cell: a sphere j cuts
// the cell of i only if d_ij < R + sqrt(max(0, R^2 - w_i + w_j)), R the
// cell's largest vertex distance from c_i.

namespace rpd {

constexpr int kNbP = 192;   // planes of one cell (6 box planes + bisectors)
constexpr int kNbV = 256;   // vertices of one cell
constexpr int kNbOut = 160;  // neighbours written per sphere

struct NbGrid {
  double org[3];
  double cs;
  double wmax;
  int32_t dim[3];
  int32_t used;
  int64_t cell_base;  // into start (cells + 1 entries)
};
struct NbGrids {
  NbGrid g[8];
};

// k / d for 0 <= k and 0 < d, by a reciprocal below 2^21 (there the
// product's error, at most (k + 0.5) / d * 2^-22, stays under 0.5 / d)
__device__ __forceinline__ int quot(int k, int d) {
  return k < (1 << 21)
             ? (int)(((float)k + 0.5f) * __builtin_amdgcn_rcpf((float)d))
             : k / d;
}

// cell of Chebyshev shell r (k in [0, shell size)) around the origin
__device__ __forceinline__ void shell_cell(int r, int k, int& dx, int& dy,
                                           int& dz) {
  const int side = 2 * r + 1, face = side * side;
  if (k < 2 * face) {  // the two z faces
    dz = k < face ? -r : r;
    const int q = k < face ? k : k - face;
    const int row = quot(q, side);
    dy = row - r;
    dx = q - row * side - r;
    return;
  }
  const int q = k - 2 * face;  // rings of the slabs between them
  const int per = 8 * r;
  const int slab = quot(q, per);
  dz = -r + 1 + slab;
  const int p = q - slab * per;
  if (p < side) {
    dy = -r;
    dx = -r + p;
  } else if (p < 2 * side) {
    dy = r;
    dx = -r + (p - side);
  } else {
    const int p2 = p - 2 * side;  // 0 .. 4r-3: the two columns
    dx = (p2 & 1) ? r : -r;
    dy = -r + 1 + (p2 >> 1);
  }
}

__device__ __noinline__ int nb_exact_w(rpd_d4 p1, rpd_d4 p2, rpd_d4 p3) {
  return rpd_exact_w_sign(p1, p2, p3);
}
// The builder's unit of length, a power of two near the box's largest
// coordinate (1 for the unit cube): filter bounds and binary32 positions are
// taken in it, so neither depends on the scale of the spheres.
struct NbUnit {
  double len, inv;  // and its reciprocal
};

// dot(e, X) and the filter bound of its sign: rpd_filtered_sign4 with
// sum |e_r| Q_r replaced by the larger me * sq, me = max(|e_xyz|, |e_w| / len)
// and sq = Q_x + Q_y + Q_z + len Q_w (the sum and the product fall short by
// at most 4u relative, which the 8 % slack of the constant over gamma_10
// covers; products may fuse into the sums, no monomial then passing through
// more roundings).  e_w and Q_xyz carry one length more than e_xyz and Q_w:
// without the unit the bound is too wide by the scale or its reciprocal, and
// from 1e12 on every sign was open (6,000 spheres 10 -> 2,500 ms).  An
// unrepresentable bound is infinite: nothing is decided.
__device__ __forceinline__ void nb_dot(const rpd_d4& e, double me,
                                       const rpd_d4& X, double sq, double& s,
                                       double& eps) {
#pragma clang fp contract(fast)
  s = e.x * X.x + e.y * X.y + e.z * X.z + e.w * X.w;
  const double b = me * sq;
  eps = b < RPD_FILTER_MAX ? RPD_FILTER_C * b + RPD_FILTER_ABS : INFINITY;
}

// Reductions over a wavefront: within rows of 16 lanes by DPP rotations, the
// four rows by reads of their first lanes (no LDS-routed shuffle).
template <int C>
__device__ __forceinline__ float row_ror(float v) {
  return __int_as_float(
      __builtin_amdgcn_mov_dpp(__float_as_int(v), 0x120 + C, 0xF, 0xF, false));
}
template <class Op>
__device__ __forceinline__ float wave_reduce(float v, Op op) {
  v = op(v, row_ror<8>(v));
  v = op(v, row_ror<4>(v));
  v = op(v, row_ror<2>(v));
  v = op(v, row_ror<1>(v));
  return op(op(lane_value(v, 0), lane_value(v, 16)),
            op(lane_value(v, 32), lane_value(v, 48)));
}
__device__ __forceinline__ float wave_max(float v) {
  return wave_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float wave_min(float v) {
  return wave_reduce(v, [](float a, float b) { return fminf(a, b); });
}
__device__ __forceinline__ float wave_add(float v) {
  return wave_reduce(v, [](float a, float b) { return a + b; });
}

// One wavefront per sphere.  The cell's vertices live in registers, vertex
// slot 64 q + lane in slot q of a lane: homogeneous coordinates X with
// X.w > 0 (the plane triple is ordered for it), the sum of its cofactor
// permanents, the triple.  Only the planes are in LDS.
//
// What bounds it is the chain of clips per sphere (each a few dependent LDS
// and lane exchanges), so a clip is kept short and unneeded ones are not
// started: candidates are taken 64 at a time, one per lane, in the order of
// the search (class, shell, 64 cells of it, member number, cell: it decides
// which of several bisectors through one point carries a face), and each
// lane first tests its bisector against every vertex of the cell as it is
// now; a bisector certainly positive everywhere cannot cut the cell or any
// later state of it.  The rest are clipped one after the other.  In a clip
// the edges that the plane cuts are the pairs (removed, kept) of vertices
// that share two planes: for each removed vertex every lane compares its
// own triple.  New vertices take the free slots.
//
// kVS = 1 (64 vertices, 64 planes) holds nearly every cell; a sphere whose
// cell outgrows it is listed and done again from the start with kVS = 4
// (256 vertices, 192 planes), whose launch reads the list's length on the
// device.  50,000 spheres of the boundary rule: one kernel of 256-vertex
// cells in LDS (42 KB a wavefront, every candidate clipped, the cut edges
// found by one lane per removed vertex scanning all vertices) took
// 203 ms, this one 8.8 ms with the larger cells (5,003 uniform spheres: 2.3
// and 0.54 ms).  The grid search is half of it there: 96 chunks of 64 grid
// cells a sphere, 161 before rows and faces outside the reach of every
// vertex were left out (11.9 -> 7.8 ms without the larger cells, together
// with reductions by DPP, binary32 corners and 32-bit cell numbers).  The
// small tier at 2, 3 and 4 wavefronts per SIMD (the register limit), before
// that: 14.7, 11.8 and 15.0 ms (4 spills).
//
// valid[i]: 1 valid, 0 hidden, -1 capacity or topology failure; counts[i] /
// lists[i * kNbOut ..]: neighbour ids, ascending.
template <int kVS, int kP>
__device__ __forceinline__ void power_cell(
    int i, const double4* __restrict__ sph, const double* box,
    const NbGrids& G, const NbUnit& unit, const int64_t* __restrict__ start,
    const int32_t* __restrict__ ids, int32_t* valid, int32_t* counts,
    int32_t* lists, int32_t* rerun, int32_t* n_rerun, double4* s_pl,
    int32_t* s_src, uint32_t* s_new, int32_t* s_q, uint8_t* s_used,
    uint8_t* s_map, const float* __restrict__ cell_w) {
  constexpr bool kSmall = kP < kNbP;
  const int lane = threadIdx.x;
  const double4 sd = sph[i];
  const rpd_d4 si{sd.x, sd.y, sd.z, sd.w};
  // the centre in units
  const double cx = si.x * unit.inv, cy = si.y * unit.inv, cz = si.z * unit.inv;
  rpd_d4 X[kVS];
  double sq[kVS];
  uint32_t tr[kVS];     // planes a | b << 8 | c << 16, bit 31: X.w is 0
  uint64_t alive[kVS];  // slots in use
  float ux[kVS], uy[kVS], uz[kVS];  // position less the centre, in units
#pragma unroll
  for (int q = 0; q < kVS; ++q) {
    X[q] = rpd_d4{0, 0, 0, 1};
    sq[q] = 0;
    tr[q] = 0;
    ux[q] = uy[q] = uz[q] = 0;
    alive[q] = q == 0 ? 0xffull : 0;
  }
  int nv = 8, np = 6;
  bool empty = false, fail = false;
  bool lost = false;  // small tier: a sign this lane could not decide

  // vertex of the planes a, b, c as this lane's slot q
  auto set_vertex = [&](rpd_d4& Xq, double& sqq, uint32_t& trq, float& uxq,
                        float& uyq, float& uzq, uint32_t a, uint32_t b,
                        uint32_t c) {
    const rpd_d4 pa = ld4(&s_pl[a]), pb = ld4(&s_pl[b]), pc = ld4(&s_pl[c]);
    rpd_d4 Y, Q;
    rpd_vertex_homog(pa, pb, pc, Y, Q);
    int sw = rpd_filtered_sign_w(Y, Q);
    if constexpr (kSmall)
      lost = lost || sw == 0;
    else if (sw == 0)
      sw = nb_exact_w(pa, pb, pc);
    if (sw < 0) {
      Y = rpd_d4{-Y.x, -Y.y, -Y.z, -Y.w};
      trq = b | (a << 8) | (c << 16);
    } else {
      trq = a | (b << 8) | (c << 16) | (sw == 0 ? 0x80000000u : 0u);
    }
    Xq = Y;
    sqq = fma(Q.w, unit.len, (Q.x + Q.y) + Q.z);
    const double iw = rcp64(Y.w) * unit.inv;
    uxq = (float)fma(Y.x, iw, -cx);
    uyq = (float)fma(Y.y, iw, -cy);
    uzq = (float)fma(Y.z, iw, -cz);
  };

  // the domain box: x >= x0, x <= x1, y >= y0, y <= y1, z >= z0, z <= z1
  wsync();
  if (lane < 6) {
    const int a = lane >> 1;
    double4 p = make_double4(0, 0, 0, 0);
    double* pp = &p.x;
    if ((lane & 1) == 0) {
      pp[a] = 1.0;
      p.w = -box[a];
    } else {
      pp[a] = -1.0;
      p.w = box[3 + a];
    }
    s_pl[lane] = p;
    s_src[lane] = -1 - lane;
  }
  wsync();
  if (lane < 8)
    set_vertex(X[0], sq[0], tr[0], ux[0], uy[0], uz[0], lane & 1,
               2 + ((lane >> 1) & 1), 4 + ((lane >> 2) & 1));
  // bounds of the cell about the centre c, in binary32: R2 no less than
  // the largest |v - c|^2, and a ball (centre m, radius rm) that holds every
  // vertex; 1e-5 covers the rounding of the positions and sums
  float R2 = 0, mx = 0, my = 0, mz = 0, rm = 0;
  auto set_bounds = [&]() {
    float r2 = 0, sx = 0, sy = 0, sz = 0;
#pragma unroll
    for (int q = 0; q < kVS; ++q)
      if ((alive[q] >> lane) & 1) {
        r2 = fmaxf(r2, ux[q] * ux[q] + uy[q] * uy[q] + uz[q] * uz[q]);
        sx += ux[q];
        sy += uy[q];
        sz += uz[q];
      }
    r2 = wave_max(r2);
    const float inv = 1.0f / (float)nv;
    mx = wave_add(sx) * inv;
    my = wave_add(sy) * inv;
    mz = wave_add(sz) * inv;
    float d2 = 0;
#pragma unroll
    for (int q = 0; q < kVS; ++q)
      if ((alive[q] >> lane) & 1) {
        const float dx = ux[q] - mx, dy = uy[q] - my, dz = uz[q] - mz;
        d2 = fmaxf(d2, dx * dx + dy * dy + dz * dz);
      }
    d2 = wave_max(d2);
    R2 = r2 * 1.00001f;
    rm = sqrtf(d2) * 1.00001f + 1e-5f * sqrtf(r2);
  };
  set_bounds();

  // clip the cell by e, the bisector of sphere j (the same in every lane)
  auto clip = [&](int j, const rpd_d4& e, double me) {
    uint64_t out[kVS];
    int n_out = 0;
#pragma unroll
    for (int q = 0; q < kVS; ++q) {
      out[q] = 0;
      if (alive[q] == 0) continue;
      bool o = false;
      if (((alive[q] >> lane) & 1) && !(tr[q] >> 31)) {
        double s, eps;
        nb_dot(e, me, X[q], sq[q], s, eps);
        o = s < -eps;
        const bool open = !o && !(s > eps);
        if constexpr (kSmall)
          lost = lost || open;
        else if (open)
          o = conflict_exact(ld4(&s_pl[tr[q] & 255]),
                             ld4(&s_pl[(tr[q] >> 8) & 255]),
                             ld4(&s_pl[(tr[q] >> 16) & 255]), e) < 0;
      }
      out[q] = ballot(o);
      n_out += __popcll(out[q]);
    }
    if (kSmall && ballot(lost) != 0) {
      fail = true;
      return;
    }
    if (n_out == 0) return;
    if (n_out == nv) {
      empty = true;
      return;
    }
    if (np >= kP) {
      // planes no vertex uses any more are dropped and the rest renumbered
      // (box planes stay at 0..5)
      for (int q = lane; q < np; q += 64) s_used[q] = q < 6;
      wsync();
#pragma unroll
      for (int q = 0; q < kVS; ++q)
        if ((alive[q] >> lane) & 1) {
          s_used[tr[q] & 255] = 1;
          s_used[(tr[q] >> 8) & 255] = 1;
          s_used[(tr[q] >> 16) & 255] = 1;
        }
      wsync();
      int kept = 0;
      for (int q0 = 0; q0 < np; q0 += 64) {
        const int q = q0 + lane;
        const bool u = q < np && s_used[q];
        const uint64_t bm = ballot(u);
        const int to = kept + lanes_below(bm, lane);
        double4 pl = make_double4(0, 0, 0, 0);
        int32_t sr = 0;
        if (u) {
          pl = s_pl[q];
          sr = s_src[q];
          s_map[q] = (uint8_t)to;
        }
        wsync();
        if (u) {
          s_pl[to] = pl;
          s_src[to] = sr;
        }
        wsync();
        kept += __popcll(bm);
      }
#pragma unroll
      for (int q = 0; q < kVS; ++q)
        if ((alive[q] >> lane) & 1)
          tr[q] = (uint32_t)s_map[tr[q] & 255] |
                  ((uint32_t)s_map[(tr[q] >> 8) & 255] << 8) |
                  ((uint32_t)s_map[(tr[q] >> 16) & 255] << 16) |
                  (tr[q] & 0x80000000u);
      wsync();
      np = kept;
      if (np >= kP) {
        fail = true;
        return;
      }
    }
    const uint32_t p = (uint32_t)np;
    if (lane == 0) {
      s_pl[p] = make_double4(e.x, e.y, e.z, e.w);
      s_src[p] = j;
    }
    int n_new, n_edge;
    cut_edges<kVS>(tr, alive, out, lane, s_new, n_new, n_edge);
    // every removed vertex has three edges
    if (n_edge != 3 * n_out || nv - n_out + n_new > 64 * kVS) {
      fail = true;
      return;
    }
    wsync();
    int base = 0;  // the new vertices take the free slots
#pragma unroll
    for (int q = 0; q < kVS; ++q) {
      alive[q] &= ~out[q];
      const uint64_t fr = ~alive[q];
      const int at = base + lanes_below(fr, lane);
      const bool take = ((fr >> lane) & 1) && at < n_new;
      if (take) {
        const uint32_t ab = s_new[at];
        set_vertex(X[q], sq[q], tr[q], ux[q], uy[q], uz[q], ab & 255, ab >> 8,
                   p);
      }
      base += __popcll(fr);
      alive[q] |= ballot(take);
      if (base >= n_new) {
#pragma unroll
        for (int u = q + 1; u < kVS; ++u) alive[u] &= ~out[u];
        break;
      }
    }
    wsync();
    nv += n_new - n_out;
    np = (int)p + 1;
  };

  // the first cnt spheres of s_q, one per lane
  auto flush = [&](int cnt) {
    const int j = lane < cnt ? s_q[lane] : -1;
    rpd_d4 e{0, 0, 0, 0};
    double me = 0;
    bool may = false;
    if (j >= 0) {
      const double4 sj = sph[j];
      const double dx = sj.x - si.x, dy = sj.y - si.y, dz = sj.z - si.z;
      const double d = sqrt(dx * dx + dy * dy + dz * dz);
      const double Rc = sqrt((double)R2) * unit.len * (1 + 1e-9) + 1e-12;
      const double bj = Rc + sqrt(fmax(0.0, Rc * Rc - si.w + sj.w));
      may = !(d > bj * (1 + 1e-9) + 1e-12);
      e = rpd_bisector(si, rpd_d4{sj.x, sj.y, sj.z, sj.w});
      me = fmax(fmax(fabs(e.x), fabs(e.y)),
                fmax(fabs(e.z), fabs(e.w) * unit.inv));
    }
    const uint64_t reach = ballot(may);
    if (reach == 0) return;
    bool cuts = false;
    uint64_t todo = 0;
#pragma unroll
    for (int q = 0; q < kVS; ++q) {
      uint64_t v = alive[q];
      while (v) {
        const int l = __ffsll((long long)v) - 1;
        v &= v - 1;
        const rpd_d4 Y{lane_value(X[q].x, l), lane_value(X[q].y, l),
                       lane_value(X[q].z, l), lane_value(X[q].w, l)};
        double s, eps;
        nb_dot(e, me, Y, lane_value(sq[q], l), s, eps);
        cuts = cuts || !(s > eps);
        todo = ballot(may && cuts);
        if (todo == reach) break;
      }
      if (todo == reach) break;
    }
    if (todo == 0) return;
    while (todo && !empty && !fail) {
      const int l = __ffsll((long long)todo) - 1;
      todo &= todo - 1;
      const rpd_d4 ej{lane_value(e.x, l), lane_value(e.y, l),
                      lane_value(e.z, l), lane_value(e.w, l)};
      clip((int)lane_value((uint32_t)j, l), ej, lane_value(me, l));
    }
    if (!empty && !fail) set_bounds();
  };

  for (int c = 0; c < 8 && !empty && !fail; ++c) {
    const NbGrid& g = G.g[c];
    if (!g.used) continue;
    int64_t q0[3], rmin = 0, rmax = 0;
    int g_lo[3], g_hi[3];  // the grid's cells, relative to q0
    float off[3];          // corner of cell q0 less the centre
    for (int a = 0; a < 3; ++a) {
      q0[a] = (int64_t)floor(((&si.x)[a] - g.org[a]) / g.cs);
      const int64_t lo = q0[a], hi = q0[a] - (g.dim[a] - 1);
      const int64_t d1 = lo < 0 ? -lo : lo, d2 = hi < 0 ? -hi : hi;
      if (d1 > rmax) rmax = d1;
      if (d2 > rmax) rmax = d2;
      if (-lo > rmin) rmin = -lo;  // rings before the grid: none
      if (hi > rmin) rmin = hi;
      g_lo[a] = (int)max(-lo, (int64_t)-0x7fffffff);
      g_hi[a] = (int)max(min(-hi, (int64_t)0x7fffffff), (int64_t)-0x7fffffff);
      off[a] = (float)((g.org[a] + (double)q0[a] * g.cs - (&si.x)[a]) *
                       unit.inv);
    }
    const int64_t cell0 =
        g.cell_base + q0[0] +
        (int64_t)g.dim[0] * (q0[1] + (int64_t)g.dim[1] * q0[2]);
    const float csf = (float)(g.cs * unit.inv);
    const float wi = (float)(si.w * unit.inv * unit.inv);
    const float wm = (float)(g.wmax * unit.inv * unit.inv) * 1.00001f;
    const float ics = 1.0f / csf;
    // A sphere of weight up to wl in a cell's box cuts a vertex off only if
    // d2 <= vv - w_i + wl (d2: squared distance of the vertex to the box,
    // vv: to the centre), here with 1e-5 of every term for the rounding:
    // not (d2' > vertex_side + wl'), primes for the factors 1 -+ 1e-5
    auto vertex_side = [&](float x, float y, float z) {
      return 1.00001f * (x * x + y * y + z * z) - wi + 1e-5f * fabsf(wi);
    };
    auto box_side = [&](float x, float y, float z, float wl) {
      return 0.99999f * (x * x + y * y + z * z) - wl;
    };
    int qn = 0;  // spheres waiting in s_q
    bool done = false;
    for (int64_t r = rmin; !done && !empty && !fail; ++r) {
      const double R = sqrt((double)R2) * unit.len * (1 + 1e-9) + 1e-12;
      {
        const double bound = R + sqrt(fmax(0.0, R * R - si.w + g.wmax));
        done = r > rmax ||
               (r >= 1 && (double)(r - 1) * g.cs > bound * (1 + 1e-9) + 1e-12);
      }
      const int ri = (int)r;
      int d_lo[3] = {g_lo[0], g_lo[1], g_lo[2]};  // cells worth a look
      int d_hi[3] = {g_hi[0], g_hi[1], g_hi[2]};
      // From the third shell on (four chunks and more; the box costs about
      // one) also those that meet the bounding box of the balls in which a sphere of the class would
      // have to lie to cut a vertex off: the cell of a sphere near a
      // boundary reaches far on one side only, and R counts for all.
      if (!done && r >= 3) {
        float lx = INFINITY, ly = INFINITY, lz = INFINITY;
        float hx = -INFINITY, hy = -INFINITY, hz = -INFINITY;
#pragma unroll
        for (int q = 0; q < kVS; ++q)
          if ((alive[q] >> lane) & 1) {
            const float vv = ux[q] * ux[q] + uy[q] * uy[q] + uz[q] * uz[q];
            const float t = vv - wi + wm + 1e-5f * (vv + fabsf(wi) + wm);
            if (!(t < 0)) {
              const float rad =
                  t < 1e30f ? __builtin_amdgcn_sqrtf(t) * 1.0001f : INFINITY;
              lx = fminf(lx, ux[q] - rad);
              ly = fminf(ly, uy[q] - rad);
              lz = fminf(lz, uz[q] - rad);
              hx = fmaxf(hx, ux[q] + rad);
              hy = fmaxf(hy, uy[q] + rad);
              hz = fmaxf(hz, uz[q] + rad);
            }
          }
        const float l[3] = {wave_min(lx), wave_min(ly), wave_min(lz)};
        const float h[3] = {wave_max(hx), wave_max(hy), wave_max(hz)};
        bool inside = true;  // nothing of this shell or a later one
        for (int a = 0; a < 3; ++a) {
          // (cell d covers off + d cs .. off + (d + 1) cs)
          const float fl = (l[a] - off[a]) * ics, fh = (h[a] - off[a]) * ics;
          const int cl = (int)fminf(
              fmaxf(floorf(fl - 1e-5f * fabsf(fl) - 0.01f), -1e9f), 1e9f);
          const int ch = (int)fmaxf(
              fminf(floorf(fh + 1e-5f * fabsf(fh) + 0.01f), 1e9f), -1e9f);
          d_lo[a] = max(d_lo[a], cl);
          d_hi[a] = min(d_hi[a], ch);
          inside = inside && d_lo[a] > -ri && d_hi[a] < ri;
        }
        done = inside || d_lo[0] > d_hi[0] || d_lo[1] > d_hi[1] ||
               d_lo[2] > d_hi[2];
      }
      // the shell's cells in [k_lo[u], k_hi[u]): the rows of its two z
      // faces and the slabs between them that hold cells worth a look
      int k_lo[3] = {0, 0, 0}, k_hi[3] = {0, 0, 0};
      if (!done) {
        const int side = 2 * ri + 1, face = side * side;
        const int y0 = max(d_lo[1], -ri) + ri, y1 = min(d_hi[1], ri) + ri;
        if (y0 <= y1 && d_lo[2] <= -ri && d_hi[2] >= -ri) {
          k_lo[0] = y0 * side;
          k_hi[0] = (y1 + 1) * side;
        }
        if (y0 <= y1 && ri > 0 && d_lo[2] <= ri && d_hi[2] >= ri) {
          k_lo[1] = face + y0 * side;
          k_hi[1] = face + (y1 + 1) * side;
        }
        const int s0 = max(d_lo[2], 1 - ri) + ri - 1;
        const int s1 = min(d_hi[2], ri - 1) + ri - 1;
        if (s0 <= s1 && (d_lo[0] <= -ri || d_hi[0] >= ri || d_lo[1] <= -ri ||
                         d_hi[1] >= ri)) {
          k_lo[2] = 2 * face + s0 * 8 * ri;
          k_hi[2] = 2 * face + (s1 + 1) * 8 * ri;
        }
      }
      // margin of a cell's box: 1e-5 of a cell, and the rounding of its
      // corner in binary32 (off + d cs)
      const float mg = (1e-5f + 2e-7f * (float)(ri + 1)) * csf;
      const float wd = csf + 2 * mg;
      // the next chunk of 64 cells (from a multiple of 64) at or after k
      // that meets one of the ranges; INT_MAX: none
      auto chunk_from = [&](int k) {
        int best = 0x7fffffff;
        for (int u = 0; u < 3; ++u)
          if (k < k_hi[u])
            best = min(best, max(k, k_lo[u] & ~63));
        return best;
      };
      int k0 = chunk_from(0);
      for (;;) {
        // this lane's cell of the shell and its member range, if a sphere
        // of the cell may cut the polytope: a sphere j of its box cuts a
        // vertex v off only if dist(v, box)^2 - max w_j < |v - c|^2 - w.
        // First with the ball about m and R2 for every vertex, then vertex
        // by vertex (binary32 about the centre c, 1e-5 of every term for
        // its rounding): lanes take the cells and the vertices are
        // broadcast, or the other way round, whichever loop is shorter
        int64_t a0 = 0, a1 = 0, cell = 0;
        const int k = k0 + lane;
        float lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0}, wc = 0;
        bool near = false;
        if (k0 != 0x7fffffff &&
            ((k >= k_lo[0] && k < k_hi[0]) || (k >= k_lo[1] && k < k_hi[1]) ||
             (k >= k_lo[2] && k < k_hi[2]))) {
          int dx, dy, dz;
          shell_cell(ri, k, dx, dy, dz);
          if (dx >= d_lo[0] && dx <= d_hi[0] && dy >= d_lo[1] &&
              dy <= d_hi[1] && dz >= d_lo[2] && dz <= d_hi[2]) {
            cell = cell0 + dx + (int64_t)g.dim[0] * (dy + g.dim[1] * dz);
            wc = cell_w[cell];  // below 0: no member
            lo[0] = fmaf((float)dx, csf, off[0]) - mg;
            lo[1] = fmaf((float)dy, csf, off[1]) - mg;
            lo[2] = fmaf((float)dz, csf, off[2]) - mg;
            for (int a = 0; a < 3; ++a) hi[a] = lo[a] + wd;
            const float ex = fmaxf(0.f, fmaxf(lo[0] - mx, mx - hi[0]));
            const float ey = fmaxf(0.f, fmaxf(lo[1] - my, my - hi[1]));
            const float ez = fmaxf(0.f, fmaxf(lo[2] - mz, mz - hi[2]));
            const float far =
                __builtin_amdgcn_sqrtf(ex * ex + ey * ey + ez * ez) * 0.99999f;
            const float sl = R2 - wi + wc + 1e-5f * (R2 + fabsf(wi) + wc);
            near = wc >= 0 && !(far > rm && (far - rm) * (far - rm) > sl);
          }
        }
        uint64_t nearm = ballot(near);
        if (nearm != 0) {
          const float wl = 1.00001f * wc;
          if (__popcll(nearm) < nv) {
            uint64_t todo = nearm;
            while (todo) {
              const int l = __ffsll((long long)todo) - 1;
              todo &= todo - 1;
              const float x0 = lane_value(lo[0], l), y0 = lane_value(lo[1], l),
                          z0 = lane_value(lo[2], l), wv = lane_value(wl, l);
              bool cuts = false;
#pragma unroll
              for (int q = 0; q < kVS; ++q) {
                const float ex =
                    ux[q] - __builtin_amdgcn_fmed3f(ux[q], x0, x0 + wd);
                const float ey =
                    uy[q] - __builtin_amdgcn_fmed3f(uy[q], y0, y0 + wd);
                const float ez =
                    uz[q] - __builtin_amdgcn_fmed3f(uz[q], z0, z0 + wd);
                cuts = cuts || (((alive[q] >> lane) & 1) &&
                                !(box_side(ex, ey, ez, wv) >
                                  vertex_side(ux[q], uy[q], uz[q])));
              }
              if (ballot(cuts) == 0) nearm &= ~(1ull << l);
            }
          } else {
            bool cuts = false;
            uint64_t cm = 0;
#pragma unroll
            for (int q = 0; q < kVS; ++q) {
              const float vs = vertex_side(ux[q], uy[q], uz[q]);
              uint64_t v = alive[q];
              while (v && cm != nearm) {
                const int l = __ffsll((long long)v) - 1;
                v &= v - 1;
                const float vx = lane_value(ux[q], l),
                            vy = lane_value(uy[q], l),
                            vz = lane_value(uz[q], l);
                const float ex = vx - __builtin_amdgcn_fmed3f(vx, lo[0], hi[0]);
                const float ey = vy - __builtin_amdgcn_fmed3f(vy, lo[1], hi[1]);
                const float ez = vz - __builtin_amdgcn_fmed3f(vz, lo[2], hi[2]);
                cuts = cuts ||
                       !(box_side(ex, ey, ez, wl) > lane_value(vs, l));
                cm = ballot(near && cuts);
              }
            }
            nearm = cm;
          }
          near = (nearm >> lane) & 1;
        }
        if (near) {
          a0 = start[cell];
          a1 = start[cell + 1];
        }
        const int kn = k0 == 0x7fffffff ? k0 : chunk_from(k0 + 64);
        // waiting spheres are clipped when 64 are there, at the end of the
        // first shells (whose spheres shrink the cell) and of the class
        const bool last = kn == 0x7fffffff && (done || (r > 0 && r < rmin + 4));
        for (int m = 0; !empty && !fail; ++m) {
          const bool more = ballot(a0 + m < a1) != 0;
          if (more) {
            const int j = a0 + m < a1 ? ids[a0 + m] : i;
            const uint64_t bm = ballot(j != i);
            if (j != i) s_q[qn + lanes_below(bm, lane)] = j;
            qn += __popcll(bm);
            wsync();
          }
          if (qn >= 64 || (!more && last && qn > 0)) {
            const int cnt = min(qn, 64);
            flush(cnt);
            const int rest = lane < qn - cnt ? s_q[64 + lane] : 0;
            wsync();
            if (lane < qn - cnt) s_q[lane] = rest;
            qn -= cnt;
            wsync();
          }
          if (!more && !(last && qn > 0)) break;
        }
        k0 = kn;
        if (k0 == 0x7fffffff || empty || fail) break;
      }
    }
  }
  if (kSmall && (fail || ballot(lost) != 0)) {
    if (lane == 0) rerun[atomicAdd(n_rerun, 1)] = i;
    return;
  }
  if (fail || empty || nv == 0) {
    if (lane == 0) {
      valid[i] = fail ? -1 : 0;
      counts[i] = 0;
    }
    return;
  }
  // neighbours: the bisectors that carry a vertex of the cell, ascending
  wsync();
  for (int p = lane; p < np; p += 64) s_used[p] = 0;
  wsync();
#pragma unroll
  for (int q = 0; q < kVS; ++q)
    if ((alive[q] >> lane) & 1) {
      s_used[tr[q] & 255] = 1;
      s_used[(tr[q] >> 8) & 255] = 1;
      s_used[(tr[q] >> 16) & 255] = 1;
    }
  wsync();
  int cnt = 0;
  for (int p = 6; p < np; ++p) cnt += s_used[p];
  for (int p = 6 + lane; p < np; p += 64) {
    if (!s_used[p]) continue;
    const int j = s_src[p];
    int pos = 0;  // a sphere may carry two planes only if it came twice
    for (int u = 6; u < np; ++u) pos += s_used[u] && s_src[u] < j;
    if (pos < kNbOut) lists[(int64_t)i * kNbOut + pos] = j;
  }
  if (lane == 0) {
    valid[i] = cnt > kNbOut ? -1 : 1;
    counts[i] = min(cnt, kNbOut);
  }
}

template <int kVS, int kP>
__global__ __launch_bounds__(64, (kVS == 1 ? 3 : 1)) void k_power_nbrs(
    int32_t n, const int32_t* items, const int32_t* n_items,
    const double4* __restrict__ sph, const double* box, NbGrids G,
    NbUnit unit, const int64_t* __restrict__ start,
    const int32_t* __restrict__ ids, const float* __restrict__ cell_w, int32_t* valid, int32_t* counts,
    int32_t* lists, int32_t* rerun, int32_t* n_rerun) {
  __shared__ double4 s_pl[kP];
  __shared__ int32_t s_src[kP];
  __shared__ uint32_t s_new[64 * kVS];
  __shared__ int32_t s_q[128];
  __shared__ uint8_t s_used[kP];
  __shared__ uint8_t s_map[kP];
  const int32_t m = items ? min(n, *n_items) : n;
  for (int32_t q = blockIdx.x; q < m; q += gridDim.x)
    power_cell<kVS, kP>(items ? items[q] : q, sph, box, G, unit, start, ids,
                        valid, counts, lists, rerun, n_rerun, s_pl, s_src,
                        s_new, s_q, s_used, s_map, cell_w);
}

// One thread per list entry (i, k): every entry's sphere must be valid and
// name i back; *n_odd counts the entries where it does not (bisectors
// through one point) -- then the host closes the lists
// (rpd_nbr_from_lists) -- and the spheres that failed.
__global__ __launch_bounds__(256) void k_nbr_check(int32_t n,
                                                   const int32_t* valid,
                                                   const int32_t* counts,
                                                   const int32_t* lists,
                                                   int64_t* cnt64,
                                                   int32_t* n_odd) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t i = q / 32;
  if (i > n) return;
  const int c = i < n ? counts[i] : 0;
  if (q % 32 == 0) cnt64[i] = c;
  if (i == n) return;
  bool odd = valid[i] < 0;
  for (int k = (int)(q % 32); k < c; k += 32) {
    const int64_t j = lists[i * kNbOut + k];
    const int cj = counts[j];
    int lo = 0, hi = cj;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (lists[j * kNbOut + mid] < (int32_t)i)
        lo = mid + 1;
      else
        hi = mid;
    }
    odd = odd || !(lo < cj && lists[j * kNbOut + lo] == (int32_t)i);
  }
  if (odd) atomicAdd(n_odd, 1);
}
__global__ __launch_bounds__(256) void k_nbr_pack(int32_t n,
                                                  const int32_t* lists,
                                                  const int64_t* off,
                                                  int32_t* ids) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t i = q / 32;
  if (i >= n) return;
  const int64_t o = off[i];
  const int c = (int)(off[i + 1] - o);
  for (int k = (int)(q % 32); k < c; k += 32) ids[o + k] = lists[i * kNbOut + k];
}

}  // namespace rpd
