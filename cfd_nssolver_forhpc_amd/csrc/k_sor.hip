// k_sor.hip -- red-black SOR on the ELL pressure operator.
//
// The reference's SOR (SorPipeLine_seq / _omp, inc/pressure/solver/) sweeps
// lexicographically in place, which is sequential (and racy under OpenMP).
// With the 7-point stencil a red-black colouring makes every colour's
// update independent: x_r += omega (b_r - (A x)_r) / a_rr for all rows of one
// colour, then the other.  Rows (and x, b) live in a colour-permuted copy so
// that each colour launch streams a contiguous half of the matrix; the FMA
// chain per row is in slot order, as in the SpMV.
#include <algorithm>
#include <cmath>

#include "dev_common.h"
#include "dev_exchange.h"
#include "dev_spmv.h"

namespace cfd {

namespace {

template <typename TV, typename TX>
__global__ void __launch_bounds__(256) sweep_kernel(int64_t N, int sliced, int64_t off, int64_t cnt,
                                                    const int32_t *__restrict__ colP, const TV *__restrict__ valP,
                                                    const TX *__restrict__ bP, TX *__restrict__ xP, double omega) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t st = ell_stride(N, sliced);
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < cnt; t += stride) {
    const int64_t q = off + t, b = ell_base(q, sliced);
    double acc = 0.0;
#pragma unroll
    for (int s = 0; s < KSLOTS; ++s) {
      const int32_t cidx = ntload(colP + b + s * st);
      acc = fma((double)ntload(valP + b + s * st), (double)xP[cidx], acc);
    }
    const double d = (double)valP[b];  // slot 0: the diagonal
    xP[q] = (TX)((double)xP[q] + omega * ((double)bP[q] - acc) / d);
  }
}

template <typename TV, typename TX>
__global__ void __launch_bounds__(256) resid_kernel(int64_t N, int sliced, const int32_t *__restrict__ colP,
                                                    const TV *__restrict__ valP, const TX *__restrict__ bP,
                                                    const TX *__restrict__ xP, double *part) {
  double acc[2] = {0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t st = ell_stride(N, sliced);
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < N; q += stride) {
    const int64_t b = ell_base(q, sliced);
    double ax = 0.0;
#pragma unroll
    for (int s = 0; s < KSLOTS; ++s) {
      const int32_t cidx = ntload(colP + b + s * st);
      ax = fma((double)ntload(valP + b + s * st), (double)xP[cidx], ax);
    }
    const double r = (double)bP[q] - ax;
    acc[0] += r * r;
    acc[1] += (double)bP[q] * (double)bP[q];
  }
  block_partials<2>(acc, part);
}

template <typename TI, typename TO>
__global__ void __launch_bounds__(256) permute_in_kernel(int64_t N, const int32_t *__restrict__ perm,
                                                         const TI *__restrict__ a, TO *__restrict__ aP) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r < N) aP[perm[r]] = (TO)a[r];
}

template <typename T>
__global__ void __launch_bounds__(256) permute_out_kernel(int64_t N, const int32_t *__restrict__ perm,
                                                          const T *__restrict__ aP, T *__restrict__ a) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r < N) a[r] = aP[perm[r]];
}

__global__ void __launch_bounds__(FIN_THREADS) finalize2(const double *part, int nblk, double *out) {
  double tot[2];
  combine_partials<2>(part, nblk, tot);
  if (threadIdx.x == 0) {
    out[0] = tot[0];
    out[1] = tot[1];
  }
}

template <typename TV, typename TX>
int rbsor_generic(Ctx &c, const TV *valP, const TX *bP, TX *xP, double omega, double tol, int maxit, int check,
                  int *iters, double *relres) {
  const int64_t N = c.g.N;
  const int nbr = blocks_for(N, 256, RED_MAX_BLOCKS);
  if (check < 1) check = 1;
  int it = 0;
  double rel = INFINITY;
  while (it < maxit) {
    const int chunk = std::min(check, maxit - it);
    for (int s = 0; s < chunk; ++s) {
      for (int colour = 0; colour < 2; ++colour) {
        const int64_t off = colour ? c.ncolour[0] : 0, cnt = c.ncolour[colour];
        sweep_kernel<TV, TX><<<blocks_for(cnt, 256, 1 << 30), 256, 0, c.stream>>>(N, c.ell_sliced, off, cnt, c.colP,
                                                                                valP, bP, xP, omega);
      }
    }
    it += chunk;
    double *part = red_part_host(c, RS_NORM);
    resid_kernel<TV, TX><<<nbr, 256, 0, c.stream>>>(N, c.ell_sliced, c.colP, valP, bP, xP, part);
    finalize2<<<1, FIN_THREADS, 0, c.stream>>>(part, nbr, c.red.out + RS_NORM * 4);
    CFD_HIP(hipGetLastError());
    CFD_HIP(hipMemcpyAsync(c.hred, c.red.out + RS_NORM * 4, 2 * sizeof(double), hipMemcpyDeviceToHost, c.stream));
    CFD_HIP(hipStreamSynchronize(c.stream));
    rel = std::sqrt(c.hred[0]) / std::sqrt(c.hred[1]);
    if (rel < tol) break;
  }
  *iters = it;
  *relres = rel;
  return CFD_OK;
}

}  // namespace

int rbsor_solve(Ctx &c, const double *b, double *x, double omega, double tol, int maxit, int check_every, int *iters,
                double *relres) {
  if (!c.ell_ready || !c.colP) return fail(CFD_ERR_STATE, "ELL operator not assembled");
  const int64_t N = c.g.N;
  const int nb = blocks_for(N, 256, 1 << 30);
  permute_in_kernel<double, double><<<nb, 256, 0, c.stream>>>(N, c.perm, b, c.bP);
  permute_in_kernel<double, double><<<nb, 256, 0, c.stream>>>(N, c.perm, x, c.xP);
  CFD_HIP(hipGetLastError());
  int rc = rbsor_generic<double, double>(c, c.valP, c.bP, c.xP, omega, tol, maxit, check_every, iters, relres);
  if (rc != CFD_OK) return rc;
  permute_out_kernel<double><<<nb, 256, 0, c.stream>>>(N, c.perm, c.xP, x);
  CFD_HIP(hipGetLastError());
  return CFD_OK;
}

int rbsor_solve_f32(Ctx &c, const float *b, float *x, double omega, double tol, int maxit, int check_every,
                    int *iters, double *relres) {
  if (!c.ell_ready || !c.valP32) return fail(CFD_ERR_STATE, "FP32 ELL operator not assembled");
  const int64_t N = c.g.N;
  const int nb = blocks_for(N, 256, 1 << 30);
  permute_in_kernel<float, float><<<nb, 256, 0, c.stream>>>(N, c.perm, b, c.bP32);
  permute_in_kernel<float, float><<<nb, 256, 0, c.stream>>>(N, c.perm, x, c.xP32);
  CFD_HIP(hipGetLastError());
  int rc = rbsor_generic<float, float>(c, c.valP32, c.bP32, c.xP32, omega, tol, maxit, check_every, iters, relres);
  if (rc != CFD_OK) return rc;
  permute_out_kernel<float><<<nb, 256, 0, c.stream>>>(N, c.perm, c.xP32, x);
  CFD_HIP(hipGetLastError());
  return CFD_OK;
}

hipError_t launch_rbsor_sweep(Ctx &c, double omega) {
  const int64_t N = c.g.N;
  for (int colour = 0; colour < 2; ++colour) {
    const int64_t off = colour ? c.ncolour[0] : 0, cnt = c.ncolour[colour];
    sweep_kernel<double, double><<<blocks_for(cnt, 256, 1 << 30), 256, 0, c.stream>>>(N, c.ell_sliced, off, cnt,
                                                                                    c.colP, c.valP, c.bP, c.xP, omega);
  }
  return hipGetLastError();
}

}  // namespace cfd

// ---------------------------------------------------------------------------
// SorPipeLine (inc/pressure/solver/SorPipeLine.seq.hpp:4-122): the
// reference's own SOR, in its volume-weighted form on the ghosted pressure,
// in place.  Per interior cell, with the face coefficients of the seq
// version (cf0..cf5 = face area / centre distance, cf7 = -1 / grid::coef,
// cf6 = mChange / dt from the predicted velocity):
//   pNEW = (-p[i+1] cf0 - p[i-1] cf1 - p[j+1] cf2 - p[j-1] cf3
//           - p[k+1] cf4 - p[k-1] cf5 + cf6) cf7
//   p += omega (pNEW - p)
// boundary neighbours read the ghost pressure as the last BC left it.  The
// sweep stops when max |pNEW - p| over the sweep is at most p_criteria
// (SOR_ERROR_MAXVAL, SorPipeLine.top.hpp:7) or after itmax sweeps, and
// reports sweeps - 1 and that maximum (simu.iters, simu.error).
//
// The reference sweeps lexicographically; here the cells go in red-black
// order ((i + j + k) even first), each colour one launch in which every
// cell reads only the other colour, so the sweep is race-free and the same
// on every run.  It converges to the same fixed point.  cf0..cf7 are not
// stored (the reference keeps 8 doubles a cell): each sweep forms them from
// the 1-D metrics in the reference's operation order, with contraction off,
// so every cell's update is the oracle's red-black restatement bit for bit.
// ---------------------------------------------------------------------------
namespace cfd {
namespace {

__global__ void __launch_bounds__(256) sorp_rhs_kernel(DevGrid g, double rdt, const double *__restrict__ u1,
                                                       const double *__restrict__ v1, const double *__restrict__ w1,
                                                       double *__restrict__ cf6) {
#pragma clang fp contract(off)
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= g.N) return;
  const int64_t nyz = (int64_t)g.nyc * g.nzc;
  const int i = (int)(t / nyz) + GC, j = (int)((t / g.nzc) % g.nyc) + GC, k = (int)(t % g.nzc) + GC;
  const int64_t ic = icel(g, i, j, k), sx = (int64_t)g.ny * g.nz, sy = g.nz;
  const double mChange = (u1[ic] - u1[ic - sx]) * g.Dy[j] * g.Dz[k] + (v1[ic] - v1[ic - sy]) * g.Dx[i] * g.Dz[k] +
                         (w1[ic] - w1[ic - 1]) * g.Dx[i] * g.Dy[j];
  cf6[t] = mChange * rdt;
}

__global__ void sorp_setup_kernel(KrylovScalars *ks, double crit, int itmax) {
  ks->tol = crit;
  ks->maxit = itmax;
  ks->iters = 0;
  ks->done = 0;
  ks->relres = 0.0;
}

// the do-while test of SorPipeLine_seq after a sweep of maximum `residual`
__device__ inline bool sorp_stops(const KrylovScalars *ks, double residual) {
  return !(residual > ks->tol) || ks->iters + 1 >= ks->maxit;
}
__device__ inline void sorp_advance(const KrylovScalars *in, KrylovScalars *out, double residual) {
  const bool was = in->done != 0, stops = sorp_stops(in, residual);
  const int iters = in->iters;
  const double relres = in->relres;
  out->tol = in->tol;
  out->maxit = in->maxit;
  out->relres = was ? relres : residual;
  out->iters = was ? iters : iters + 1;
  out->done = was || stops;
}

// A sweep is two dependent launches of a few microseconds on a small grid, and
// was three: the one-block kernel that combines the maxima takes as long as a
// colour (3.6 us beside 2 x 4.3).  With at most SORP_FOLD blocks the next
// sweep's first colour combines them in every block instead (a maximum does
// not depend on the order), so the launch is gone: 12.1 -> 9.9 us a sweep at
// 8x8x1100.  The state then has two copies, read from one and written to the
// other.
constexpr int SORP_FOLD = 1024;

// one colour of a sweep; partial max |pNEW - p| per block
// wrapz: periodic z, the z neighbours of the first and last planes are the
// live pressure across the seam (not ghosts), which keeps the red-black
// colouring valid for an even nz
// FOLD: the sweep before this one left its maxima in prev[0 .. 2 RED_MAX_BLOCKS);
// ks is the state before it, next (block 0's) the state after it
template <bool FOLD>
__global__ void __launch_bounds__(256) sorp_sweep_kernel(DevGrid g, int colour, double omega, int wrapz,
                                                         const double *__restrict__ cf6, double *__restrict__ p,
                                                         const KrylovScalars *__restrict__ ks, double *part,
                                                         const double *__restrict__ prev, KrylovScalars *next) {
#pragma clang fp contract(off)
  if (FOLD) {
    __shared__ double lds[4];
    double m = 0.0;  // the maxima are not negative
    if (!ks->done) {
#pragma unroll
      for (int u = 0; u < SORP_FOLD / 256; ++u) {
        const int b = min((int)threadIdx.x + u * 256, (int)gridDim.x - 1);
        m = fmax(m, fmax(prev[b], prev[RED_MAX_BLOCKS + b]));
      }
    }
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = m;
    __syncthreads();
    const double residual = fmax(fmax(lds[0], lds[1]), fmax(lds[2], lds[3]));
    if (blockIdx.x == 0 && threadIdx.x == 0) sorp_advance(ks, next, residual);
    if (ks->done || sorp_stops(ks, residual)) return;
  } else if (ks->done) {
    return;
  }
  double mx[1] = {0.0};
  const int nzh = (g.nzc + 1) / 2;
  const int64_t cnt = (int64_t)g.nxc * g.nyc * nzh;
  const int64_t sx = (int64_t)g.ny * g.nz, sy = g.nz;
  const double *__restrict__ Dx = g.Dx, *__restrict__ Dy = g.Dy, *__restrict__ Dz = g.Dz;
  const double *__restrict__ Dxs = g.Dxs, *__restrict__ Dys = g.Dys, *__restrict__ Dzs = g.Dzs;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < cnt; t += stride) {
    const int kh = (int)(t % nzh);
    const int64_t rest = t / nzh;
    const int jc = (int)(rest % g.nyc), ic_ = (int)(rest / g.nyc);
    const int kc = 2 * kh + ((ic_ + jc + colour) & 1);
    if (kc >= g.nzc) continue;
    const int i = ic_ + GC, j = jc + GC, k = kc + GC;
    const int64_t ic = icel(g, i, j, k);
    const double cf0 = Dy[j] * Dz[k] / Dxs[i], cf1 = Dy[j] * Dz[k] / Dxs[i - 1];
    const double cf2 = Dx[i] * Dz[k] / Dys[j], cf3 = Dx[i] * Dz[k] / Dys[j - 1];
    const double cf4 = Dx[i] * Dy[j] / Dzs[k], cf5 = Dx[i] * Dy[j] / Dzs[k - 1];
    // grid::coef (inc/grid/structureGrid.hpp:278-287), summed in its order
    const double coef = Dy[j] * Dz[k] / Dxs[i] + Dy[j] * Dz[k] / Dxs[i - 1] + Dx[i] * Dz[k] / Dys[j] +
                        Dx[i] * Dz[k] / Dys[j - 1] + Dx[i] * Dy[j] / Dzs[k] + Dx[i] * Dy[j] / Dzs[k - 1];
    const double cf7 = -1.0 / coef;
    const int64_t izp = (wrapz && k == g.nz - 3) ? ic - (g.nzc - 1) : ic + 1;
    const int64_t izm = (wrapz && k == GC) ? ic + (g.nzc - 1) : ic - 1;
    const double pxp = p[ic + sx], pxm = p[ic - sx], pyp = p[ic + sy], pym = p[ic - sy], pzp = p[izp],
                 pzm = p[izm], pc = p[ic];
    const int64_t row = ((int64_t)ic_ * g.nyc + jc) * g.nzc + kc;
    const double pNEW = (-pxp * cf0 - pxm * cf1 - pyp * cf2 - pym * cf3 - pzp * cf4 - pzm * cf5 + cf6[row]) * cf7;
    mx[0] = fmax(mx[0], fabs(pNEW - pc));
    p[ic] = pc + omega * (pNEW - pc);
  }
  block_partials<1, true>(mx, part);
}

// the sweep's maximum over both colours
__global__ void __launch_bounds__(FIN_THREADS) sorp_finalize_kernel(const double *part, int nblk,
                                                                    const KrylovScalars *in, KrylovScalars *out) {
  double a[1], b[1];
  combine_partials<1, true>(part, nblk, a);
  combine_partials<1, true>(part + RED_MAX_BLOCKS, nblk, b);
  if (threadIdx.x == 0) sorp_advance(in, out, fmax(a[0], b[0]));
}

// ---- all the sweeps of a small grid in one launch ---------------------------
// A colour of a small grid is a launch of 4.3 us whatever its size, most of it
// launch, drain and the thirteen divisions of its coefficients.  Here every
// workgroup keeps its cells for all the sweeps: a thread owns the two cells
// of a pair in z (one of each colour), their coefficients in registers, their
// pressure in LDS beside that of the halo and of the ghosts, which do
// not change.  After a colour a workgroup leaves its new values for the others
// and waits for those of its halo (dev_exchange.h).  The sweep's maximum
// travels while the next sweep's first colour runs; if it ends the solve, that
// colour is dropped.  Every cell's update is sorp_sweep_kernel's, operation for
// operation, and a maximum has no order, so the results are the same bits.
// A value is rewritten two colours later, after the neighbours' values of the
// colour between, which they leave after their reads; a maximum two sweeps
// later, after every workgroup's next one, left after its reads.
// Bound by the two exchanges a sweep.  us a sweep, launches -> here: 512 cells
// 11.2 -> 1.0 (one workgroup), 4096 11.8 -> 2.5, 110592 12.7 -> 4.4, 262144
// 13.3 -> 5.8.  Two pairs a thread reach 524288 cells, but take 17.9 us there
// against the launches' 15.7.
constexpr int SORR_THREADS = 512, SORR_BLOCKS = 256;  // one workgroup a CU, all resident

struct SorLds {
  static constexpr int OWN = SORR_THREADS;      // pairs
  static constexpr int HALO = OWN * 2 + 512;    // cells of a colour: x neighbours of every pair, two z lines and more
  static constexpr int GHOST = 3072;
  double p[2 * OWN + 2 * HALO + GHOST];         // own cells (parity of k), halo (colour), ghosts
  int32_t hrow[2][HALO];
  double wmax[SORR_THREADS / 64], tot[SORR_BLOCKS / 64];
  int nhalo[2], nghost, state, stuck;
};

struct SorArgs {
  uint64_t *ll0, *ll1;  // the two words of each cell
  uint64_t *mx;         // maxima: [sweep parity][word][workgroup]
  double *keep;         // the cells' pressure before the solve
  KrylovScalars *ks;    // pad0: arrivals, pad1: RES_* state
  int nblk, chunk;      // chunk: sweeps this launch runs at most
  ResBounds bounds;
};

__global__ void __launch_bounds__(SORR_THREADS) sorp_resident_kernel(DevGrid g, double omega, int wrapz,
                                                                     const double *__restrict__ cf6,
                                                                     double *__restrict__ p, SorArgs a) {
#pragma clang fp contract(off)
  __shared__ SorLds L;
  constexpr int OWN = SorLds::OWN, HALO = SorLds::HALO, GHOST = SorLds::GHOST;
  const int tid = threadIdx.x, blk = blockIdx.x;
  const int nxc = g.nxc, nyc = g.nyc, nzc = g.nzc, nzh = (nzc + 1) / 2;
  const int npair = nxc * nyc * nzh;
  if (a.ks->done) return;  // uniform over the grid
  const double tol = a.ks->tol;
  const int maxit = a.ks->maxit;
  int iters = a.ks->iters;
  if (tid < 2) L.nhalo[tid] = 0;
  if (tid == 2) L.nghost = L.stuck = 0;
  __syncthreads();
  const double *__restrict__ Dx = g.Dx, *__restrict__ Dy = g.Dy, *__restrict__ Dz = g.Dz;
  const double *__restrict__ Dxs = g.Dxs, *__restrict__ Dys = g.Dys, *__restrict__ Dzs = g.Dzs;
  double cf[2][6], rhs[2], cf7[2], cur[2];
  unsigned pos[2][3], row[2], at[2];
  bool own[2];
  int fits = 1;
  {
    const int t = blk * OWN + tid, kh = t % nzh, rest = t / nzh, j0 = rest % nyc, i0 = rest / nyc;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int k0 = 2 * kh + ((i0 + j0 + c) & 1);
      own[c] = t < npair && k0 < nzc;
      const int ic_ = own[c] ? i0 : 0, jc = own[c] ? j0 : 0, kc = own[c] ? k0 : 0;
      const int i = ic_ + GC, j = jc + GC, k = kc + GC;
      const double cf0 = Dy[j] * Dz[k] / Dxs[i], cf1 = Dy[j] * Dz[k] / Dxs[i - 1];
      const double cf2 = Dx[i] * Dz[k] / Dys[j], cf3 = Dx[i] * Dz[k] / Dys[j - 1];
      const double cf4 = Dx[i] * Dy[j] / Dzs[k], cf5 = Dx[i] * Dy[j] / Dzs[k - 1];
      const double coef = Dy[j] * Dz[k] / Dxs[i] + Dy[j] * Dz[k] / Dxs[i - 1] + Dx[i] * Dz[k] / Dys[j] +
                          Dx[i] * Dz[k] / Dys[j - 1] + Dx[i] * Dy[j] / Dzs[k] + Dx[i] * Dy[j] / Dzs[k - 1];
      cf[c][0] = cf0, cf[c][1] = cf1, cf[c][2] = cf2, cf[c][3] = cf3, cf[c][4] = cf4, cf[c][5] = cf5;
      cf7[c] = -1.0 / coef;
      row[c] = (unsigned)((ic_ * nyc + jc) * nzc + kc);
      rhs[c] = cf6[row[c]];
      cur[c] = p[icel(g, i, j, k)];
      at[c] = (unsigned)((kc & 1) * OWN + tid);
      if (own[c]) L.p[at[c]] = cur[c];
      unsigned ps[6];
#pragma unroll
      for (int d = 0; d < 6; ++d) {  // +x, -x, +y, -y, +z, -z
        int in = ic_, jn = jc, kn = kc;
        if (d < 2) in += d == 0 ? 1 : -1;
        else if (d < 4) jn += d == 2 ? 1 : -1;
        else kn += d == 4 ? 1 : -1;
        if (wrapz) kn = kn == nzc ? 0 : kn < 0 ? nzc - 1 : kn;
        unsigned at_n = 0;
        if (own[c]) {
          const double v = p[icel(g, in + GC, jn + GC, kn + GC)];
          if (in < 0 || in >= nxc || jn < 0 || jn >= nyc || kn < 0 || kn >= nzc) {
            const int e = atomicAdd(&L.nghost, 1);
            at_n = 2 * OWN + 2 * HALO + min(e, GHOST - 1);
            if (e >= GHOST) fits = 0;
            else L.p[at_n] = v;
          } else {
            const int tn = (in * nyc + jn) * nzh + (kn >> 1);
            if (tn / OWN == blk) {
              at_n = (kn & 1) * OWN + tn % OWN;
            } else {
              const int e = atomicAdd(&L.nhalo[1 - c], 1);
              at_n = 2 * OWN + (1 - c) * HALO + min(e, HALO - 1);
              if (e >= HALO) {
                fits = 0;
              } else {
                L.hrow[1 - c][e] = (in * nyc + jn) * nzc + kn;
                L.p[at_n] = v;
              }
            }
          }
        }
        ps[d] = at_n;
      }
#pragma unroll
      for (int d = 0; d < 3; ++d) pos[c][d] = ps[2 * d] | ps[2 * d + 1] << 16;
    }
  }
  fits = __syncthreads_and(fits);
  if (resident_arrive(a.ks, a.nblk, &L.state, fits, a.bounds.arrive) != RES_GO) return;

  double mx = 0.0, old = 0.0;
  // colour c of the sweep with exchange number epoch (1, 2, 3, ..)
  auto colour = [&](auto cc, unsigned epoch) __attribute__((always_inline)) {
#pragma clang fp contract(off)
    constexpr int c = decltype(cc)::value;
    {
      double n[6];
#pragma unroll
      for (int d = 0; d < 6; ++d) n[d] = L.p[(d & 1) ? pos[c][d >> 1] >> 16 : pos[c][d >> 1] & 0xffffu];
      const double *f = cf[c];
      const double pc = cur[c];
      const double pNEW = (-n[0] * f[0] - n[1] * f[1] - n[2] * f[2] - n[3] * f[3] - n[4] * f[4] - n[5] * f[5] +
                           rhs[c]) * cf7[c];
      if (c == 0) old = pc;
      if (own[c]) {
        mx = fmax(mx, fabs(pNEW - pc));
        cur[c] = pc + omega * (pNEW - pc);
        L.p[at[c]] = cur[c];
        if (a.nblk > 1) ll_store(at32(a.ll0, row[c]), at32(a.ll1, row[c]), cur[c], epoch);
      }
    }
  };
  // the halo's cells of colour c with that number, by the threads from `busy` on
  auto halo = [&](int c, unsigned epoch, int busy) __attribute__((always_inline)) {
    const int nh = L.nhalo[c], step = SORR_THREADS - busy;
    if (tid < busy) return;
    for (int e0 = tid - busy; e0 < nh; e0 += 4 * step) {
      const bool ok = ll_fetch<4>(
          a.ll0, a.ll1, epoch, res_spin<true>(a.bounds), L.stuck,
          [&](int u) { return e0 + u * step < nh ? (unsigned)L.hrow[c][e0 + u * step] : RES_NONE; },
          [&](int u, bool have, double v) {
            if (have) L.p[2 * OWN + c * HALO + e0 + u * step] = v;
          });
      if (!ok) L.stuck = 1;
    }
  };
  const int busy = (a.nblk + 63) / 64 * 64;  // threads that wait for the maxima, at most half
  double residual = a.ks->relres;
  int done = 0;
  for (int s = 0;; ++s) {
    const unsigned h = 2u * (unsigned)s;
    if (s > 0) halo(1, h, 0);
    __syncthreads();
    colour(std::integral_constant<int, 0>(), h + 1);
    __syncthreads();  // every wave has issued its words (RES_SPIN)
    if (a.nblk > 1) {
      if (s > 0 && tid < busy) {
        double v = 0.0;
        const uint64_t *w = a.mx + ((s - 1) & 1) * 2 * SORR_BLOCKS;
        const bool ok = ll_fetch<1>(
            w, w + SORR_BLOCKS, (unsigned)s, res_spin<true>(a.bounds), L.stuck,
            [&](int) { return tid < a.nblk ? (unsigned)tid : RES_NONE; },
            [&](int, bool have, double x) { v = have ? x : 0.0; });
        if (!ok) L.stuck = 1;
        v = wave_max(v);
        if ((tid & 63) == 0) L.tot[tid >> 6] = v;
      }
      halo(0, h + 1, s > 0 ? busy : 0);
    } else if (s > 0 && tid == 0) {
      double v = L.wmax[0];
      for (int w = 1; w < SORR_THREADS / 64; ++w) v = fmax(v, L.wmax[w]);
      L.tot[0] = v;
    }
    __syncthreads();
    if (L.stuck) {  // a wait reached its bound
      if (tid == 0) __hip_atomic_store(&a.ks->pad1, (int)RES_STUCK, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    if (s > 0) {
      residual = L.tot[0];
      for (int w = 1; w < busy / 64; ++w) residual = fmax(residual, L.tot[w]);
      iters += 1;
      done = !(residual > tol) || iters >= maxit;
      if (done || s >= a.chunk) {  // without the colour just done
        cur[0] = old;
        break;
      }
    }
    colour(std::integral_constant<int, 1>(), h + 2);
    const double m = wave_max(mx);
    mx = 0.0;
    if ((tid & 63) == 0) L.wmax[tid >> 6] = m;
    __syncthreads();
    if (tid == 0 && a.nblk > 1) {
      double v = L.wmax[0];
#pragma unroll
      for (int w = 1; w < SORR_THREADS / 64; ++w) v = fmax(v, L.wmax[w]);
      uint64_t *w = a.mx + (s & 1) * 2 * SORR_BLOCKS + blk;
      ll_store(w, w + SORR_BLOCKS, v, (unsigned)s + 1);
    }
  }
#pragma unroll
  for (int c = 0; c < 2; ++c)
    if (own[c]) {
      const int r = (int)row[c], kc = r % nzc, rest = r / nzc;
      p[icel(g, rest / nyc + GC, rest % nyc + GC, kc + GC)] = cur[c];
    }
  if (blk == 0 && tid == 0) {
    a.ks->relres = residual;
    a.ks->iters = iters;
    a.ks->done = done;
  }
}

// the ghosted position of cell q
__device__ inline int64_t sorp_cell(const DevGrid &g, int64_t q) {
  const int r = (int)q, kc = r % g.nzc, rest = r / g.nzc;
  return icel(g, rest / g.nyc + GC, rest % g.nyc + GC, kc + GC);
}

__global__ void __launch_bounds__(256) sorp_clear_kernel(DevGrid g, const double *__restrict__ p, SorArgs a,
                                                         bool first) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, n = g.N;
  if (first && q < n) a.keep[q] = p[sorp_cell(g, q)];
  if (q < n) a.ll0[q] = a.ll1[q] = 0;
  if (q < 4 * SORR_BLOCKS) a.mx[q] = 0;
  if (q == 0) a.ks->pad0 = a.ks->pad1 = 0;
}

__global__ void __launch_bounds__(256) sorp_restore_kernel(DevGrid g, double *__restrict__ p, SorArgs a) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < g.N) p[sorp_cell(g, q)] = a.keep[q];
}

// *solved is false when the launches have to do it: more cells than the
// workgroups hold (262144 at an even nz), a halo or ghosts that LDS does not
// hold, or CUs that are taken.  *lost: they start again, from the pressure that
// is back in place (a wait reached its bound).
int sorp_resident(Ctx &c, double omega, const double *cf6, bool *solved, bool *lost) {
  *solved = *lost = false;
  const DevGrid &g = c.g;
  const int64_t npair = (int64_t)g.nxc * g.nyc * ((g.nzc + 1) / 2);
  if (npair > SORR_THREADS * SORR_BLOCKS) return CFD_OK;
  SorArgs a;
  a.ll0 = reinterpret_cast<uint64_t *>(c.s1);  // the Krylov solver's vectors
  a.ll1 = reinterpret_cast<uint64_t *>(c.ap);
  a.mx = reinterpret_cast<uint64_t *>(red_part_host(c, RS_SPMV_DOT));
  a.keep = c.as;
  a.ks = c.ks;
  a.nblk = (int)((npair + SORR_THREADS - 1) / SORR_THREADS);
  a.chunk = 4096;  // bounds one launch to some tens of milliseconds
  a.bounds = res_bounds(c.one);
  ResidentSlots slots;
  if (!c.one.due()) return CFD_OK;
  if (!slots.take(c.device, a.nblk)) {
    c.one.handed_back++;
    return CFD_OK;
  }
  const int nbc = blocks_for(std::max<int64_t>(g.N, 4 * SORR_BLOCKS), 256, 1 << 30);
  for (bool first = true;; first = false) {
    sorp_clear_kernel<<<nbc, 256, 0, c.stream>>>(g, c.f[CFD_P], a, first);
    sorp_resident_kernel<<<a.nblk, SORR_THREADS, 0, c.stream>>>(g, omega, c.prm.periodic_z, cf6, c.f[CFD_P], a);
    CFD_HIP(hipGetLastError());
    CFD_HIP(hipMemcpyAsync(c.hks, c.ks, sizeof(KrylovScalars), hipMemcpyDeviceToHost, c.stream));
    CFD_HIP(hipStreamSynchronize(c.stream));
    if (c.hks->pad1 != RES_GO) {
      if (c.hks->pad1 == RES_STUCK) {
        sorp_restore_kernel<<<nbc, 256, 0, c.stream>>>(g, c.f[CFD_P], a);
        CFD_HIP(hipGetLastError());
        *lost = true;
      }
      c.one.gave_up();
      return CFD_OK;
    }
    if (c.hks->done) break;
  }
  c.one.finish();
  *solved = true;
  return CFD_OK;
}

}  // namespace

int sor_pipeline_solve(Ctx &c, double omega, double crit, int itmax, int *iters, double *error) {
  const DevGrid &g = c.g;
  if (itmax < 1) return fail(CFD_ERR_ARG, "SorPipeLine: p_sor_iter_max must be >= 1");
  double *cf6 = c.f[CFD_RHS];
  sorp_rhs_kernel<<<blocks_for(g.N, 256, 1 << 30), 256, 0, c.stream>>>(g, 1.0 / c.prm.dt, c.f[CFD_T1_U],
                                                                      c.f[CFD_T1_V], c.f[CFD_T1_W], cf6);
  sorp_setup_kernel<<<1, 1, 0, c.stream>>>(c.ks, crit, itmax);
  CFD_HIP(hipGetLastError());
  bool solved = false, lost = false;
  if (int rc = sorp_resident(c, omega, cf6, &solved, &lost)) return rc;
  if (lost) sorp_setup_kernel<<<1, 1, 0, c.stream>>>(c.ks, crit, itmax);
  if (solved) {
    *iters = c.hks->iters - 1;
    *error = c.hks->relres;
    return CFD_OK;
  }
  const int64_t cnt = (int64_t)g.nxc * g.nyc * ((g.nzc + 1) / 2);
  const int nb = blocks_for(cnt, 256, RED_MAX_BLOCKS);
  // a sweep's maxima, the first colour's and the second's; sweeps take turns (a
  // block may still read the last one's)
  double *part[2] = {red_part_host(c, RS_SPMV_DOT), red_part_host(c, RS_SPMV_DOT2)};
  const bool fold = nb <= SORP_FOLD;
  int batch = 4, done_sweeps = 0;
  double prev = -1.0;
  int prev_it = 0;
  for (;;) {
    KrylovScalars *st = c.ks;  // the state before the sweep, once it is known
    for (int s = 0; s < batch; ++s) {
      double *mx = part[s & 1];
      if (s > 0 && fold) {
        KrylovScalars *before = st;
        st = before == c.ks ? c.ks + 1 : c.ks;
        sorp_sweep_kernel<true><<<nb, 256, 0, c.stream>>>(g, 0, omega, c.prm.periodic_z, cf6, c.f[CFD_P], before, mx,
                                                          part[(s - 1) & 1], st);
      } else {
        sorp_sweep_kernel<false><<<nb, 256, 0, c.stream>>>(g, 0, omega, c.prm.periodic_z, cf6, c.f[CFD_P], st, mx,
                                                           nullptr, nullptr);
      }
      sorp_sweep_kernel<false><<<nb, 256, 0, c.stream>>>(g, 1, omega, c.prm.periodic_z, cf6, c.f[CFD_P], st,
                                                         mx + RED_MAX_BLOCKS, nullptr, nullptr);
      if (!fold || s == batch - 1)
        sorp_finalize_kernel<<<1, FIN_THREADS, 0, c.stream>>>(mx, nb, st, c.ks);
    }
    CFD_HIP(hipGetLastError());
    CFD_HIP(hipMemcpyAsync(c.hks, c.ks, sizeof(KrylovScalars), hipMemcpyDeviceToHost, c.stream));
    CFD_HIP(hipStreamSynchronize(c.stream));
    const KrylovScalars h = *c.hks;
    done_sweeps = h.iters;
    if (h.done) break;
    // the sweeps still needed, from the last batch's contraction rate
    int next = batch * 2;
    if (prev > 0.0 && h.relres > 0.0 && h.relres < prev && h.iters > prev_it) {
      const double rate = std::log(h.relres / prev) / (double)(h.iters - prev_it);
      const double need = std::log(crit / h.relres) / rate;
      if (need > 0.0 && std::isfinite(need)) next = (int)std::ceil(need * 1.05) + 1;
    }
    prev = h.relres;
    prev_it = h.iters;
    batch = std::max(1, std::min(next, std::min(512, itmax - h.iters)));
  }
  *iters = done_sweeps - 1;  // SorPipeLine_seq's --simu.iters
  *error = c.hks->relres;
  return CFD_OK;
}

}  // namespace cfd

// ---------------------------------------------------------------------------
// Red-black SOR on the CSR operator (grid::createPressureMatrixCSR, the
// operator of P_SOLVER_BICG_CSR): rows in natural order, the cells of one
// colour per launch, x_r += omega (b_r - (A x)_r) / a_rr with the row's
// products summed in stored order (csr_row) and a_rr the entry whose column
// is r.  Same colouring and update as the ELL form.
// ---------------------------------------------------------------------------
namespace cfd {
namespace {

__global__ void __launch_bounds__(256) csr_sweep_kernel(int nxc, int nyc, int nzc, int colour,
                                                        const int32_t *__restrict__ ptr,
                                                        const int32_t *__restrict__ col,
                                                        const double *__restrict__ val, const double *__restrict__ b,
                                                        double *__restrict__ x, double omega) {
  const int nzh = (nzc + 1) / 2;
  const int64_t cnt = (int64_t)nxc * nyc * nzh;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < cnt; t += stride) {
    const int kh = (int)(t % nzh);
    const int64_t rest = t / nzh;
    const int jc = (int)(rest % nyc), ic = (int)(rest / nyc);
    const int kc = 2 * kh + ((ic + jc + colour) & 1);
    if (kc >= nzc) continue;
    const int64_t r = ((int64_t)ic * nyc + jc) * nzc + kc;
    double acc = 0.0, diag = 0.0;
    const int32_t e1 = ptr[r + 1];
    for (int32_t e = ptr[r]; e < e1; ++e) {
      const int32_t cc = col[e];
      const double v = val[e];
      acc = fma(v, x[cc], acc);
      if (cc == r) diag = v;
    }
    x[r] = x[r] + omega * (b[r] - acc) / diag;
  }
}

__global__ void __launch_bounds__(256) csr_resid_kernel(int64_t N, const int32_t *__restrict__ ptr,
                                                        const int32_t *__restrict__ col,
                                                        const double *__restrict__ val, const double *__restrict__ b,
                                                        const double *__restrict__ x, double *part) {
  double acc[2] = {0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += stride) {
    const double res = b[r] - csr_row(ptr, col, val, r, x);
    acc[0] += res * res;
    acc[1] += b[r] * b[r];
  }
  block_partials<2>(acc, part);
}

}  // namespace

int rbsor_csr_solve(Ctx &c, const double *b, double *x, double omega, double tol, int maxit, int check_every,
                    int *iters, double *relres) {
  if (!c.csr_ready) return fail(CFD_ERR_STATE, "CSR operator not assembled");
  const DevGrid &g = c.g;
  const int64_t N = g.N;
  const int64_t cnt = (int64_t)g.nxc * g.nyc * ((g.nzc + 1) / 2);
  const int nbs = blocks_for(cnt, 256, 1 << 30);
  const int nbr = blocks_for(N, 256, RED_MAX_BLOCKS);
  const int check = check_every < 1 ? 1 : check_every;
  int it = 0;
  double rel = INFINITY;
  while (it < maxit) {
    const int chunk = std::min(check, maxit - it);
    for (int s = 0; s < chunk; ++s)
      for (int colour = 0; colour < 2; ++colour)
        csr_sweep_kernel<<<nbs, 256, 0, c.stream>>>(g.nxc, g.nyc, g.nzc, colour, c.csr_ptr, c.csr_col, c.csr_val, b,
                                                    x, omega);
    it += chunk;
    double *part = red_part_host(c, RS_NORM);
    csr_resid_kernel<<<nbr, 256, 0, c.stream>>>(N, c.csr_ptr, c.csr_col, c.csr_val, b, x, part);
    finalize2<<<1, FIN_THREADS, 0, c.stream>>>(part, nbr, c.red.out + RS_NORM * 4);
    CFD_HIP(hipGetLastError());
    CFD_HIP(hipMemcpyAsync(c.hred, c.red.out + RS_NORM * 4, 2 * sizeof(double), hipMemcpyDeviceToHost, c.stream));
    CFD_HIP(hipStreamSynchronize(c.stream));
    rel = std::sqrt(c.hred[0]) / std::sqrt(c.hred[1]);
    if (rel < tol) break;
  }
  *iters = it;
  *relres = rel;
  return CFD_OK;
}

}  // namespace cfd
