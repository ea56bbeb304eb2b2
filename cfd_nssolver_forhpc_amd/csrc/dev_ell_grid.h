// The assembled ELL operator over planes: its entries formed from the axis
// coefficients (ell_grid_value), its rows two a lane.  What it cannot do
// without is x, y and the dot's vector (16 or 24 B/row); at 512x256x64 inside
// an iteration it takes 49.6 us with one dot and 43.4 with two (reading the
// stored entries 138 and 133), 31 us as a plain product from a warm cache
// (131).  It is bound by the loads of the four y and z neighbours, which hit
// the L1 but go through its pipe (58 and 43 -> 45 and 32 us without them, one
// row a lane): hence two rows a lane, which halves them.  The division is
// hidden (73.6 -> 73.5 us without it), an XCD-contiguous block order is 5%
// slower, one row a lane over four planes a thread without the march took 68.5
// and 53.
#pragma once
#include <algorithm>
#include <initializer_list>

#include "dev_common.h"
#include "dev_spmv.h"
#include "pred_tiled.h"

namespace cfd {
namespace {

typedef double double2v __attribute__((ext_vector_type(2)));

__device__ inline double2v at_bytes2(const double *base, uint32_t off) {
  return *reinterpret_cast<const double2v *>(reinterpret_cast<const char *>(base) + off);
}

// wave_sum of the 64 rows that half a wave holds, two a lane (rows 2 l and
// 2 l + 1 in lane l): wave_sum adds neighbouring lanes, then neighbouring
// pairs, and so on; here its first step is the lane's own sum.  Lanes 31 and
// 63 hold the totals of the two halves.
__device__ inline double half_wave_sum(double v0, double v1) {
  double v = v0 + v1;
  v += dpp_move<0xb1>(v);   // quad_perm [1,0,3,2]
  v += dpp_move<0x4e>(v);   // quad_perm [2,3,0,1]
  v += dpp_move<0x124>(v);  // row_ror:4
  v += dpp_move<0x128>(v);  // row_ror:8
  v += dpp_move<0x142>(v);  // row_bcast:15
  return v;
}

// Planes first .. first + np - 1 at the rows at, at + 1 of a plane (at even,
// nzc even: one line), plane by plane: fn(m, their row values, x's own
// entries, w's).  An entry of x is loaded once for its plane's diagonal and
// the x neighbours of the planes beside it, and the rows are each other's z
// neighbours.  What a plane needs is loaded GRID_RING - 1 planes ahead (its
// coefficients too), into the registers of the plane just left, without a
// branch around a load (clamped indexes past the grid instead), so that the
// loads stay in flight; 104 registers, four waves a SIMD (a plane more ahead
// takes 134, three waves, and 50.0 / 41.8 us).  first and np are the same in the whole block,
// np <= nxc - first; x and w are 16-byte aligned.
constexpr int GRID_RING = 2;

struct EllGridPair {
  int j, k;                        // of the first row
  uint32_t oc, oym, oyp, oa, ob;   // byte offsets in a plane: the pair, its y neighbours, the z neighbours at its ends
  bool hym, hyp, ha, hb;
};

// wrap: the z faces are joined
__device__ inline EllGridPair ell_grid_pair(const OpArgs &a, uint32_t at, bool wrap) {
  EllGridPair c;
  const uint32_t line = (uint32_t)a.nzc, seam = line - 1;
  c.j = (int)fastdiv(at, a.div_nz);
  c.k = (int)(at - (uint32_t)c.j * line);
  c.hym = c.j != 0;
  c.hyp = c.j != a.nyc - 1;
  const bool first = c.k == 0, last = c.k == a.nzc - 2;
  c.ha = wrap || !first;
  c.hb = wrap || !last;
  c.oc = at * 8u;
  c.oym = (c.hym ? at - line : at) * 8u;
  c.oyp = (c.hyp ? at + line : at) * 8u;
  c.oa = (!first ? at - 1 : c.ha ? at + seam : at) * 8u;
  c.ob = (!last ? at + 2 : c.hb ? at + 1 - seam : at) * 8u;
  return c;
}

struct SpeCoef {
  double ym, yp, zm, zp, sym, syp, szm, szp;  // s: what a closed face takes off the diagonal
};

// spe_row from the coefficients, 1 / jp summed in spe_jp_kernel's order
template <bool YW, bool ZW>
__device__ inline double spe_grid_value(const EllGridPlane &e, bool hym, bool hyp, bool hzm, bool hzp, const SpeCoef &q,
                                        double sxm, double sxp, double xc, double vxm, double vxp, double vym,
                                        double vyp, double vzm, double vzp) {
  double d = e.xm + q.ym;
  d = d + q.zm;
  d = d + e.xp;
  d = d + q.yp;
  d = d + q.zp;
  d = d - sxm;
  d = d - sxp;
  if (!YW) {
    d = d - q.sym;
    d = d - q.syp;
  }
  if (!ZW) {
    d = d - q.szm;
    d = d - q.szp;
  }
  const double J = 1.0 / d;
  double sum = 0.0, t = fma(-e.xm * J, vxm, sum);
  sum = e.hxm ? t : sum;
  t = fma(-q.ym * J, vym, sum);
  sum = YW || hym ? t : sum;
  t = fma(-q.zm * J, vzm, sum);
  sum = ZW || hzm ? t : sum;
  sum += xc;
  t = fma(-q.zp * J, vzp, sum);
  sum = ZW || hzp ? t : sum;
  t = fma(-q.yp * J, vyp, sum);
  sum = YW || hyp ? t : sum;
  t = fma(-e.xp * J, vxp, sum);
  return e.hxp ? t : sum;
}

template <bool SPE, bool YW, bool ZW, bool W, typename F>
__device__ __attribute__((always_inline)) inline void ell_grid_march(const OpArgs &a, const EllGridPair &c, int first,
                                                                     int np, const double *__restrict__ x,
                                                                     const double *__restrict__ w, F fn) {
  constexpr int R = GRID_RING;
  const int64_t plane = (int64_t)a.nyc * a.nzc;
  double2v below, here, above, vym[R], vyp[R], wv[R];  // x of planes i - 1, i, i + 1; the rest of plane i by i % R
  double va[R], vb[R], pxm[R], pxp[R];
  auto fetch = [&](int s, int i) __attribute__((always_inline)) {
    const int ic = min(i, a.nxc - 1);
    const int64_t o = ic * plane;
    vym[s] = at_bytes2(x + o, c.oym);
    vyp[s] = at_bytes2(x + o, c.oyp);
    va[s] = at_bytes(x + o, c.oa);
    vb[s] = at_bytes(x + o, c.ob);
    if (W) wv[s] = at_bytes2(w + o, c.oc);
    pxm[s] = (SPE ? a.coef : a.ecoef)[ic];
    pxp[s] = (SPE ? a.coef : a.ecoef)[a.nxc + ic];
  };
  below = at_bytes2(x + max(first - 1, 0) * plane, c.oc);
  here = at_bytes2(x + first * plane, c.oc);
  above = at_bytes2(x + min(first + 1, a.nxc - 1) * plane, c.oc);
#pragma unroll
  for (int s = 0; s < R - 1; ++s) fetch(s, first + s);
  const double xlast = x[a.N - 1];
  // the line's coefficients, whose loads stay behind those of x, which come from farther away
  __builtin_amdgcn_sched_barrier(0);
  int jl = c.j, kl = c.k;
  asm volatile("" : "+v"(jl), "+v"(kl));
  EllGridPlace c0, c1;
  c0.j = c1.j = jl;
  c0.k = kl;
  c1.k = kl + 1;
  c0.hym = c1.hym = c.hym;
  c0.hyp = c1.hyp = c.hyp;
  const bool first_z = c.k == 0;  // the first row's +z neighbour has the slot before its -z one
  c0.hz1 = first_z || c.ha;
  c0.hz2 = first_z ? c.ha : true;
  c1.hz1 = true;
  c1.hz2 = c.hb;
  EllGridCoef q0, q1;
  SpeCoef w0, w1;
  if (SPE) {
    const double *ym = a.coef + 2 * a.nxc, *yp = ym + a.nyc, *zm = yp + a.nyc, *zp = zm + a.nzc;
    w0.ym = w1.ym = ym[jl];
    w0.yp = w1.yp = yp[jl];
    w0.zm = zm[kl];
    w0.zp = zp[kl];
    w1.zm = zm[kl + 1];
    w1.zp = zp[kl + 1];
    w0.sym = w1.sym = jl == 0 && !a.spd[2] ? w0.ym : 0.0;
    w0.syp = w1.syp = jl == a.nyc - 1 && !a.spd[3] ? w0.yp : 0.0;
    w0.szm = kl == 0 && !a.spd[4] && !a.swrapz ? w0.zm : 0.0;
    w1.szp = kl + 1 == a.nzc - 1 && !a.spd[5] && !a.swrapz ? w1.zp : 0.0;
    w0.szp = w1.szm = 0.0;
  } else {
    q0 = ell_grid_coef(a, c0);
    q1 = ell_grid_coef(a, c1);
    q1.z1 = q1.zm;
    q1.z2 = q1.zp;
  }
#pragma unroll 1
  for (int m = 0; m < np; m += R) {
#pragma unroll
    for (int s = 0; s < R; ++s) {
      if (m + s >= np) return;
      const int i = first + m + s;
      EllGridPlane e;
      e.xm = pxm[s];
      e.xp = pxp[s];
      e.hxm = i != 0;
      e.hxp = i != a.nxc - 1;
      double2v y;
      if (SPE) {
        const double sxm = !e.hxm && !a.spd[0] ? e.xm : 0.0, sxp = !e.hxp && !a.spd[1] ? e.xp : 0.0;
        y.x = spe_grid_value<YW, ZW>(e, c.hym, c.hyp, c.ha, true, w0, sxm, sxp, here.x, below.x, above.x, vym[s].x,
                                     vyp[s].x, va[s], here.y);
        y.y = spe_grid_value<YW, ZW>(e, c.hym, c.hyp, true, c.hb, w1, sxm, sxp, here.y, below.y, above.y, vym[s].y,
                                     vyp[s].y, here.x, vb[s]);
      } else {
        e.aa = 0.0;
        if (!e.hxm && !a.epd[0]) e.aa = -e.xm;
        if (!e.hxp && !a.epd[1]) e.aa = -e.xp;
        const double z1 = first_z ? here.y : va[s], z2 = first_z ? va[s] : here.y;
        y.x = ell_grid_value<YW, ZW>(e, c0, q0, here.x, below.x, above.x, vym[s].x, vyp[s].x, z1, z2, xlast);
        y.y = ell_grid_value<YW, ZW>(e, c1, q1, here.y, below.y, above.y, vym[s].y, vyp[s].y, here.x, vb[s], xlast);
      }
      fn(m + s, y, here, wv[s]);
      __builtin_amdgcn_sched_barrier(0);
      below = here;
      here = above;
      above = at_bytes2(x + min(i + 2, a.nxc - 1) * plane, c.oc);
      fetch((s + R - 1) % R, i + R - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// y = A x with the dots that follow it (DOTS: 0 none; 1 y . w; 2 (y . x,
// y . y); 3 (y . w, y . y)).  A block of BT / 2 threads owns BT consecutive
// rows of a plane (nyc nzc a multiple of BT) and walks M planes of a period of
// planes, PP = gridDim of the row-wise kernel x BT / (nyc nzc) (all of them
// while a row a thread is enough for it).  With more than one period (MULTI)
// it walks the same planes of each in turn, so that a row position's sum is
// the one of the row-wise kernel's thread, and the partial of each BT rows is
// that kernel's bit for bit.
// Planes a block walks: up to sixteen, as long as 1024 blocks remain, four of
// 256 threads a CU (512x256x64: 49.6 / 43.4 us at 16 planes, 52.4 / 38.6 at
// 4; 256x128x32 with 16 planes and an eighth of the CUs 13 us, with 2 planes 7).
constexpr int GRID_BLOCKS = 1024;
constexpr int GRID_WALK = 16, GRID_WALK_MULTI = 4;

template <int BT, int DOTS, bool MULTI>
__global__ void __launch_bounds__(BT / 2, 4) ell_grid_kernel(OpArgs a, int PP, int M, const KrylovScalars *__restrict__ ks,
                                                          const double *__restrict__ x, double *__restrict__ y,
                                                          const double *__restrict__ w, double *part) {
  if (DOTS && ks->done) return;
  constexpr int NV = DOTS < 2 ? 1 : 2;
  __shared__ double red[GRID_WALK][NV][BT / 64];
  __shared__ double2v own[MULTI ? GRID_WALK_MULTI * NV : 1][MULTI ? BT / 2 : 1];  // a row position's sums over the periods
  const int nynz = a.nyc * a.nzc, ntile = nynz / BT;
  const int blk = (int)blockIdx.x;
  const int tile = blk % ntile, i0 = blk / ntile * M;
  const int tid = (int)threadIdx.x, half = tid >> 5;
  const EllGridPair c = ell_grid_pair(a, (uint32_t)(tile * BT + 2 * tid), a.ewrapz);
  const int np0 = min(M, min(PP, a.nxc) - i0);
  if (MULTI) {
    for (int u = 0; u < M * NV; ++u) own[u][tid] = double2v{0.0, 0.0};
  }
  for (int first = i0; first < a.nxc; first += PP) {
    const int np = min(np0, a.nxc - first);
    double *yi = y + (int64_t)first * nynz;
    auto rows = [&](int m, double2v v, double2v xc, double2v wv) __attribute__((always_inline)) {
      ntstore(v, reinterpret_cast<double2v *>(reinterpret_cast<char *>(yi + (int64_t)m * nynz) + c.oc));
      const double2v d = DOTS == 2 ? xc : wv;
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const double2v f = u ? v : d;
        if (MULTI) {
          double2v s = own[m * NV + u][tid];
          s.x += v.x * f.x;
          s.y += v.y * f.y;
          own[m * NV + u][tid] = s;
        } else if (DOTS) {
          const double s = half_wave_sum(fma(v.x, f.x, 0.0), fma(v.y, f.y, 0.0));
          if ((tid & 31) == 31) red[m][u][half] = s;
        }
      }
    };
    const bool yw = __all(c.hym && c.hyp);  // most waves have no y face, and with joined z faces no z one
    if (yw && a.ewrapz)
      ell_grid_march<false, true, true, (DOTS & 1) != 0>(a, c, first, np, x, w, rows);
    else if (yw)
      ell_grid_march<false, true, false, (DOTS & 1) != 0>(a, c, first, np, x, w, rows);
    else
      ell_grid_march<false, false, false, (DOTS & 1) != 0>(a, c, first, np, x, w, rows);
  }
  if (!DOTS) return;
  if (MULTI) {
    for (int u = 0; u < M * NV; ++u) {
      const double s = half_wave_sum(own[u][tid].x, own[u][tid].y);
      if ((tid & 31) == 31) red[u / NV][u % NV][half] = s;
    }
  }
  __syncthreads();
  if (tid < np0 * NV) {
    const int m = tid / NV, u = tid % NV;
    double s = red[m][u][0];
#pragma unroll
    for (int v = 1; v < BT / 64; ++v) s += red[m][u][v];
    part[u * RED_MAX_BLOCKS + (i0 + m) * ntile + tile] = s;
  }
}

// planes of a period for the row-wise kernel's nb blocks of bt threads; 0
// where its threads' rows are not whole planes apart, or a line or a vector
// does not start at a pair (row-wise then)
inline int ell_grid_period(const OpArgs &a, int64_t nb, int bt, std::initializer_list<const void *> vecs) {
  if (a.op != OP_ELL_GRID || a.nzc % 2 != 0) return 0;
  for (const void *p : vecs)
    if (reinterpret_cast<uintptr_t>(p) % 16 != 0) return 0;
  const int64_t nynz = (int64_t)a.nyc * a.nzc, rows = nb * bt;
  if (nynz % bt != 0) return 0;
  if (rows >= a.N) return a.nxc;
  return rows % nynz == 0 ? (int)(rows / nynz) : 0;
}

template <int BT, int DOTS>
void launch_ell_grid(const OpArgs &a, int pp, const KrylovScalars *ks, const double *x, double *y, const double *w,
                     double *part, hipStream_t st) {
  const int ntile = a.nyc * a.nzc / BT;
  if (DOTS && pp < a.nxc) {
    const int m = GRID_WALK_MULTI;
    ell_grid_kernel<BT, DOTS, DOTS != 0><<<(pp + m - 1) / m * ntile, BT / 2, 0, st>>>(a, pp, m, ks, x, y, w, part);
  } else {
    const int m = std::min(GRID_WALK, std::max(2, (int)((int64_t)pp * ntile / GRID_BLOCKS)));
    ell_grid_kernel<BT, DOTS, false><<<(pp + m - 1) / m * ntile, BT / 2, 0, st>>>(a, pp, m, ks, x, y, w, part);
  }
}

// The SPE operator the same way, with the dots and partials of the kernels
// over plane columns (spe_column_rows): a tile is kb x jb columns (k, j) and
// SPE_PLANES planes, a thread of 128 has two columns beside each other in k,
// and a block walks G tiles above each other in i without loading their
// borders again.  jp, 8 B/row, is formed again too.
// us, K1 alone / an iteration, plane columns -> here: 512x256x64 46.5 / 273 ->
// 38.9 / 253, 256x128x64 15.4 / 79.7 -> 12.5 / 72.3, 190x210x40 15.0 / 70.3 ->
// 12.1 / 65.2 (1272 tiles), 200x104x40 10.3 / 44.0 -> 9.6 / 43.9 (650),
// 64x32x32 5.9 / 23.2 -> 6.0 / 26.0 (64): a tile's planes come one behind the
// other, so it takes SPE_TILES of them, four blocks a CU, to hide that.  Tiles
// are walked on (G) as long as SPE_BLOCKS blocks remain.
constexpr int SPE_WALK = 4, SPE_BLOCKS = 2048, SPE_TILES = 1024;

template <int DOTS>
__global__ void __launch_bounds__(128, 4) spe_walk_kernel(OpArgs a, SpeTiles T, int G,
                                                          const KrylovScalars *__restrict__ ks,
                                                          const double *__restrict__ x, double *__restrict__ y,
                                                          const double *__restrict__ w, double *part) {
  if (DOTS && ks->done) return;
  constexpr int NV = DOTS < 2 ? 1 : 2;
  __shared__ double red[SPE_WALK][NV][4];
  const int b = blockIdx.x, tk = b % T.nkt, rest = b / T.nkt, jt = rest % T.njt, ig = rest / T.njt * G;
  const int tid = (int)threadIdx.x;
  const int k = tk * T.kb + 2 * tid % T.kb, j = jt * T.jb + 2 * tid / T.kb;
  const bool ok = k < a.nzc && j < a.nyc;  // nzc is even: both columns or none
  const EllGridPair c = ell_grid_pair(a, (uint32_t)(min(j, a.nyc - 1) * a.nzc + min(k, a.nzc - 2)), a.wrapz);
  const int first = ig * SPE_PLANES, np = min(G * SPE_PLANES, a.nxc - first);
  const int64_t nynz = (int64_t)a.nyc * a.nzc;
  double *yi = y + first * nynz;
  double2v acc[NV];
#pragma unroll
  for (int u = 0; u < NV; ++u) acc[u] = double2v{0.0, 0.0};
  auto rows = [&](int m, double2v v, double2v xc, double2v wv) __attribute__((always_inline)) {
    const double2v d = DOTS == 2 ? xc : wv;
    if (ok) {
      ntstore(v, reinterpret_cast<double2v *>(reinterpret_cast<char *>(yi + m * nynz) + c.oc));
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const double2v f = u ? v : d;
        if (DOTS) {
          acc[u].x += v.x * f.x;
          acc[u].y += v.y * f.y;
        }
      }
    }
    if (DOTS && (m % SPE_PLANES == SPE_PLANES - 1 || m == np - 1)) {
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const double s = half_wave_sum(acc[u].x, acc[u].y);
        if ((tid & 31) == 31) red[m / SPE_PLANES][u][tid >> 5] = s;
        acc[u] = double2v{0.0, 0.0};
      }
    }
  };
  const bool yw = __all(c.hym && c.hyp);
  if (yw && a.wrapz && a.swrapz)
    ell_grid_march<true, true, true, (DOTS & 1) != 0>(a, c, first, np, x, w, rows);
  else if (yw)
    ell_grid_march<true, true, false, (DOTS & 1) != 0>(a, c, first, np, x, w, rows);
  else
    ell_grid_march<true, false, false, (DOTS & 1) != 0>(a, c, first, np, x, w, rows);
  if (!DOTS) return;
  __syncthreads();
  const int ng = (np + SPE_PLANES - 1) / SPE_PLANES;
  if (tid < ng * NV) {
    const int g = tid / NV, u = tid % NV;
    double s = red[g][u][0];
#pragma unroll
    for (int v = 1; v < 4; ++v) s += red[g][u][v];
    part[u * RED_MAX_BLOCKS + ((ig + g) * T.njt + jt) * T.nkt + tk] = s;
  }
}

// whether the operator's kernels walk pairs of columns
inline bool spe_pairs(const OpArgs &a, const SpeTiles &T, std::initializer_list<const void *> vecs) {
  for (const void *p : vecs)
    if (reinterpret_cast<uintptr_t>(p) % 16 != 0) return false;
  return a.op == CFD_OP_SPE && T.blocks >= SPE_TILES && a.nzc % 2 == 0 && (int64_t)a.nyc * a.nzc < (int64_t)1 << 29;
}

template <int DOTS>
void launch_spe_walk(const OpArgs &a, const SpeTiles &T, const KrylovScalars *ks, const double *x, double *y,
                     const double *w, double *part, hipStream_t st) {
  const int64_t col = (int64_t)T.nkt * T.njt;
  const int G = (int)std::min<int64_t>(SPE_WALK, std::max<int64_t>(1, T.blocks / SPE_BLOCKS));
  spe_walk_kernel<DOTS><<<(unsigned)(col * ((T.nig + G - 1) / G)), 128, 0, st>>>(a, T, G, ks, x, y, w, part);
}

}  // namespace
}  // namespace cfd
