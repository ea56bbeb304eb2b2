// k_krylov.hip -- restarted BiCGSTAB (solver::bicgstabRe2,
// inc/solver/bicgstabRe2.hpp:91-189) and FP32-inner / FP64-outer defect
// correction on gfx950.
//
// One iteration is five streaming kernels, each fusing the reference's
// BLAS-1 work with the reduction that follows it:
//   K1  ap = A p,               partial (ap . r0)           -> F1: alpha
//   K2  s  = r - alpha ap
//   K3  as = A s,               partials (as . s), (as . as) -> F2: omega
//   K4  x += alpha p + omega s; r = s - omega as;
//                               partials (r . r), (r . r0)   -> F3: stop test, beta, restart rule
//   K5  p  = r + beta (p - omega ap)   (or r0 = p = r on restart)
// F1-F3 are one-block kernels combining the per-block partials in a fixed
// order (deterministic results) and updating the solver's scalars in device
// memory, or parts of K2, K4 and K5 in small systems (fold_of); every kernel returns at once when the device-side `done` flag is
// set, so the host launches iterations in batches and reads the flag once per
// batch instead of once per dot product.  FP64 dots are kept for every
// scalar, also when the vectors are FP32.  FP64 systems of up to half a million
// ELL rows run their iterations in one kernel instead (dev_resident.h).
#include <algorithm>
#include <atomic>
#include <cstdio>
#include <mutex>
#include <string>
#include <type_traits>
#include <cmath>

#include "dev_common.h"
#include "dev_resident.h"
#include "dev_spmv.h"
#include "dev_ell_grid.h"

namespace cfd {

namespace {

template <typename T>
__device__ inline T op_apply(const OpArgs &a, int64_t r, const T *__restrict__ x);
template <>
__device__ inline double op_apply<double>(const OpArgs &a, int64_t r, const double *__restrict__ x) {
  return op_row(a, r, x);
}
template <>
__device__ inline float op_apply<float>(const OpArgs &a, int64_t r, const float *__restrict__ x) {
  return op_row32(a, r, x);
}

// (A x)[base + threadIdx.x] for the block of rows starting at base (0 past
// the last row); every thread of the block calls it with the same base
template <typename T>
__device__ inline T op_apply_block(const OpArgs &a, int64_t base, const T *__restrict__ x);
template <>
__device__ inline double op_apply_block<double>(const OpArgs &a, int64_t base, const double *__restrict__ x) {
  return op_row_block(a, base, x);
}
template <>
__device__ inline float op_apply_block<float>(const OpArgs &a, int64_t base, const float *__restrict__ x) {
  const int64_t r = base + threadIdx.x;
  return r < a.N ? op_row32(a, r, x) : 0.0f;
}

__global__ void ks_setup_kernel(KrylovScalars *ks, double tol, double restart_tol, int maxit, int timestep) {
  ks->tol = tol;
  ks->restart_tol = restart_tol;
  ks->maxit = maxit;
  ks->timestep = timestep;
  ks->done = 0;
  ks->hit_maxit = 0;
  ks->iters = 0;
  ks->restart = 0;
}

// r0 = b - A x; r1 = p1 = r0; px2 = px1; px1 = x; partials (b.b), (r0.r0)
template <typename T>
__global__ void __launch_bounds__(256) init_kernel(OpArgs a, const T *__restrict__ b, const T *__restrict__ x,
                                                   T *__restrict__ r0, T *__restrict__ r1, T *__restrict__ p1,
                                                   double *__restrict__ px1, double *__restrict__ px2,
                                                   double *part) {
  double acc[2] = {0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < a.N; base += stride) {
    const T ax = op_apply_block<T>(a, base, x);
    const int64_t r = base + threadIdx.x;
    if (r >= a.N) continue;
    const T br = b[r];
    const T rr = br - ax;
    r0[r] = rr;
    r1[r] = rr;
    p1[r] = rr;
    if (px1) {  // px2: NULL for a solver without history (its px2 is all zero)
      if (px2) px2[r] = px1[r];
      px1[r] = (double)x[r];
    }
    acc[0] += (double)br * (double)br;
    acc[1] += (double)rr * (double)rr;
  }
  block_partials<2>(acc, part);
}

__global__ void __launch_bounds__(FIN_THREADS) init_finalize(const double *part, int nblk, KrylovScalars *ks) {
  double tot[2];
  combine_partials<2>(part, nblk, tot);
  if (threadIdx.x == 0) {
    ks->norm0 = sqrt(tot[0]);
    ks->rho = tot[1];
    ks->relres = sqrt(tot[1]) / ks->norm0;
  }
}

// BT threads a block: 256 for the CSR operator (op_apply_block stages 256
// rows), SPMV_DOT_THREADS for the others
template <typename T, int BT = 256>
__global__ void __launch_bounds__(BT) spmv_dot_kernel(OpArgs a, const KrylovScalars *__restrict__ ks,
                                                      const T *__restrict__ p1, T *__restrict__ ap,
                                                      const T *__restrict__ r0, double *part) {
  if (ks->done) return;
  double acc[1] = {0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < a.N; base += stride) {
    const T y = op_apply_block<T>(a, base, p1);
    const int64_t r = base + threadIdx.x;
    if (r >= a.N) continue;
    ntstore(y, ap + r);
    acc[0] += (double)y * (double)r0[r];
  }
  block_partials<1, false, BT>(acc, part);
}

// spmv_dot and spmv_dot2 for the SPE operator over plane columns
// (spe_column_rows): the same rows, a third of the loads; the partials of a
// block sum its columns' planes, so the dot products are ordered differently
// from the row-wise kernels (deterministically)
__global__ void __launch_bounds__(256) spe_spmv_dot_kernel(OpArgs a, SpeTiles T, const KrylovScalars *__restrict__ ks,
                                                           const double *__restrict__ p1, double *__restrict__ ap,
                                                           const double *__restrict__ r0, double *part) {
  if (ks->done) return;
  double acc[1] = {0.0};
  const SpeColumn c = spe_column(a, T);
  if (c.ok) {
    const int64_t nynz = (int64_t)a.nyc * a.nzc, col = (int64_t)c.j * a.nzc + c.k;
    double w[SPE_PLANES];
    spe_plane_values(a, c, r0, w);
    double y[SPE_PLANES], xc[SPE_PLANES];
    const int np = spe_column_rows(a, c, p1, y, xc);
#pragma unroll
    for (int p = 0; p < SPE_PLANES; ++p)
      if (p < np) {
        const int64_t r = (int64_t)(c.i0 + p) * nynz + col;
        ntstore(y[p], ap + r);
        acc[0] += y[p] * w[p];
      }
  }
  block_partials<1>(acc, part);
}

__global__ void __launch_bounds__(256) spe_spmv_dot2_kernel(OpArgs a, SpeTiles T, const KrylovScalars *__restrict__ ks,
                                                            const double *__restrict__ s1, double *__restrict__ as,
                                                            double *part) {
  if (ks->done) return;
  double acc[2] = {0.0, 0.0};
  const SpeColumn c = spe_column(a, T);
  if (c.ok) {
    double y[SPE_PLANES], xc[SPE_PLANES];
    const int np = spe_column_rows(a, c, s1, y, xc);
    const int64_t nynz = (int64_t)a.nyc * a.nzc, col = (int64_t)c.j * a.nzc + c.k;
#pragma unroll
    for (int p = 0; p < SPE_PLANES; ++p)
      if (p < np) {
        ntstore(y[p], as + (int64_t)(c.i0 + p) * nynz + col);
        acc[0] += y[p] * xc[p];
        acc[1] += y[p] * y[p];
      }
  }
  block_partials<2>(acc, part);
}

// combine_partials of nblk <= C FIN_THREADS partials by a block of BT threads:
// thread t stands in for threads t, t + BT, .. of the finalize block, whose
// sums over its slots, waves and block are formed in the same order.  (In the
// finalize kernels too: with 2 of the 16 slots that combine_partials loads at a
// time, 5.7 -> 3.7 us.)
template <int BT, int C, int NV>
__device__ inline void combine_folded(const double *part, int nblk, double (&tot)[NV]) {
  constexpr int G = FIN_THREADS / BT;
  static_assert(C == 1 || C == 2 || C == 4, "the tree below");
  __shared__ double lds[NV][FIN_THREADS / 64];
  double s[NV][G][C];
#pragma unroll
  for (int q = 0; q < NV; ++q)
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int u = 0; u < C; ++u) {
        const int b = (int)threadIdx.x + g * BT + u * FIN_THREADS;
        s[q][g][u] = part[q * RED_MAX_BLOCKS + min(b, nblk - 1)];
      }
#pragma unroll
  for (int q = 0; q < NV; ++q)
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
      for (int u = 0; u < C; ++u) {
        const int b = (int)threadIdx.x + g * BT + u * FIN_THREADS;
        s[q][g][u] = b < nblk ? s[q][g][u] : 0.0;
      }
      double v = s[q][g][0];
      if (C > 1) v += s[q][g][C > 1 ? 1 : 0];
      if (C > 2) v += s[q][g][C > 2 ? 2 : 0] + s[q][g][C > 2 ? 3 : 0];
      v = wave_sum(v + 0.0);
      if ((threadIdx.x & 63) == 0) lds[q][g * (BT / 64) + (threadIdx.x >> 6)] = v;
    }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    double v = lds[q][0];
#pragma unroll
    for (int w = 1; w < FIN_THREADS / 64; ++w) v += lds[q][w];
    tot[q] = v;
  }
}

// f(slots a finalize thread takes; 0: combine_partials' chunks of sixteen)
template <typename F>
void with_slots(int nblk, F f) {
  if (nblk <= FIN_THREADS) f(std::integral_constant<int, 1>());
  else if (nblk <= 2 * FIN_THREADS) f(std::integral_constant<int, 2>());
  else if (nblk <= 4 * FIN_THREADS) f(std::integral_constant<int, 4>());
  else f(std::integral_constant<int, 0>());
}

template <int C, int NV>
__device__ inline void combine_slots(const double *part, int nblk, double (&tot)[NV]) {
  if constexpr (C > 0) combine_folded<FIN_THREADS, C>(part, nblk, tot);
  else combine_partials<NV>(part, nblk, tot);
}

// The finalize kernels read the scalars they use before the partials, so
// that those reads share the partials' round trip to memory instead of
// preceding it; with `done` set the totals are combined and dropped.
template <int C>
__global__ void __launch_bounds__(FIN_THREADS) alpha_finalize(const double *part, int nblk, KrylovScalars *ks) {
  const int done = ks->done;
  const double rho = ks->rho;
  asm volatile("" ::: "memory");  // issue both loads here, not after the combine
  double tot[1];
  combine_slots<C>(part, nblk, tot);
  if (done) return;
  if (threadIdx.x == 0) ks->alpha = rho / tot[0];
}

template <typename T>
__global__ void __launch_bounds__(256) s_update_kernel(int64_t N, const KrylovScalars *__restrict__ ks,
                                                       const T *__restrict__ r1, const T *__restrict__ ap,
                                                       T *__restrict__ s1) {
  if (ks->done) return;
  const double alpha = ks->alpha;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += stride)
    s1[r] = (T)((double)r1[r] - alpha * (double)ap[r]);
}

template <typename T, int BT = 256>
__global__ void __launch_bounds__(BT) spmv_dot2_kernel(OpArgs a, const KrylovScalars *__restrict__ ks,
                                                       const T *__restrict__ s1, T *__restrict__ as, double *part) {
  if (ks->done) return;
  double acc[2] = {0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < a.N; base += stride) {
    const T y = op_apply_block<T>(a, base, s1);
    const int64_t r = base + threadIdx.x;
    if (r >= a.N) continue;
    ntstore(y, as + r);
    acc[0] += (double)y * (double)s1[r];
    acc[1] += (double)y * (double)y;
  }
  block_partials<2, false, BT>(acc, part);
}

template <int C>
__global__ void __launch_bounds__(FIN_THREADS) omega_finalize(const double *part, int nblk, KrylovScalars *ks) {
  const int done = ks->done;
  asm volatile("" ::: "memory");
  double tot[2];
  combine_slots<C>(part, nblk, tot);
  if (done) return;
  if (threadIdx.x == 0) ks->omega = tot[0] / tot[1];
}

template <typename T>
__global__ void __launch_bounds__(256) xr_update_kernel(int64_t N, const KrylovScalars *__restrict__ ks,
                                                        T *__restrict__ x, const T *__restrict__ p1,
                                                        const T *__restrict__ s1, const T *__restrict__ as,
                                                        T *__restrict__ r1, const T *__restrict__ r0, double *part) {
  if (ks->done) return;
  const double alpha = ks->alpha, omega = ks->omega;
  double acc[2] = {0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += stride) {
    const double s = (double)s1[r];
    ntstore((T)((double)x[r] + fma(omega, s, alpha * (double)p1[r])), x + r);
    const T rn = (T)(s - omega * (double)as[r]);
    ntstore(rn, r1 + r);
    acc[0] += (double)rn * (double)rn;
    acc[1] += (double)rn * (double)r0[r];
  }
  block_partials<2>(acc, part);
}

// stop test, beta and the restart rule (bicgstabRe2.hpp:137-183)
// The scalars after an iteration with (r . r) = rr, (r . r0) = rho, from those
// within it (`in`) into those between iterations (`out`, the same or another
// copy, whose constants are there).  Field by field: a copy of the structure
// lands in scratch memory.
struct ConvNext {
  double rnorm, relres, beta;
  int stop, hit, restart;  // stop: done after this iteration
};
__device__ inline ConvNext conv_next(const KrylovScalars *in, double rr, double rho) {
  ConvNext n;
  const double pre_rho = in->rho;
  n.rnorm = sqrt(rr);
  n.relres = n.rnorm / in->norm0;
  const bool converged = n.relres < in->tol;
  n.hit = !converged && in->iters >= in->maxit;
  n.stop = converged || n.hit;
  n.beta = (in->alpha / in->omega) * (rho / pre_rho);
  n.restart = (in->timestep < 10 || fabs(pre_rho) > in->restart_tol) ? 0 : 1;
  return n;
}
__device__ inline void conv_store(const KrylovScalars *in, KrylovScalars *out, const ConvNext &n, double rho) {
  const double pre_rho = in->rho, alpha = in->alpha, omega = in->omega;
  const int iters = in->iters, restarts = in->restarts;
  out->alpha = alpha;
  out->omega = omega;
  out->rnorm = n.rnorm;
  out->relres = n.relres;
  if (n.stop) {
    out->done = 1;
    if (n.hit) out->hit_maxit = 1;
  } else {
    out->pre_rho = pre_rho;
    out->rho = rho;
    out->beta = n.beta;
    out->restart = n.restart;
    out->restarts = restarts + n.restart;
    out->iters = iters + 1;
  }
}
// K2's copy of the scalars between iterations (in) for those within (out)
__device__ inline void begin_iteration(const KrylovScalars *in, KrylovScalars *out, double alpha) {
  const int done = in->done;
  out->rho = in->rho;
  out->norm0 = in->norm0;
  out->tol = in->tol;
  out->restart_tol = in->restart_tol;
  out->iters = in->iters;
  out->maxit = in->maxit;
  out->timestep = in->timestep;
  out->restarts = in->restarts;
  out->done = done;
  if (!done) out->alpha = alpha;
}

template <int C>
__global__ void __launch_bounds__(FIN_THREADS) conv_finalize(const double *part, int nblk, const KrylovScalars *in,
                                                             KrylovScalars *out) {
  const int done = in->done;
  asm volatile("" ::: "memory");
  double tot[2];
  combine_slots<C>(part, nblk, tot);
  if (done) return;
  if (threadIdx.x == 0) conv_store(in, out, conv_next(in, tot[0], tot[1]), tot[1]);
}

void launch_alpha_finalize(const double *part, int nblk, KrylovScalars *ks, hipStream_t st) {
  with_slots(nblk, [&](auto c) { alpha_finalize<decltype(c)::value><<<1, FIN_THREADS, 0, st>>>(part, nblk, ks); });
}
void launch_omega_finalize(const double *part, int nblk, KrylovScalars *ks, hipStream_t st) {
  with_slots(nblk, [&](auto c) { omega_finalize<decltype(c)::value><<<1, FIN_THREADS, 0, st>>>(part, nblk, ks); });
}
void launch_conv_finalize(const double *part, int nblk, const KrylovScalars *in, KrylovScalars *out, hipStream_t st) {
  with_slots(nblk, [&](auto c) { conv_finalize<decltype(c)::value><<<1, FIN_THREADS, 0, st>>>(part, nblk, in, out); });
}


template <typename T>
__global__ void __launch_bounds__(256) p_update_kernel(int64_t N, const KrylovScalars *__restrict__ ks,
                                                       const T *__restrict__ r1, T *__restrict__ p1,
                                                       const T *__restrict__ ap, T *__restrict__ r0) {
  if (ks->done) return;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  if (ks->restart) {
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += stride) {
      r0[r] = r1[r];
      p1[r] = r1[r];
    }
    return;
  }
  const double beta = ks->beta, omega = ks->omega;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += stride)
    p1[r] = (T)((double)r1[r] + beta * ((double)p1[r] - omega * (double)ap[r]));
}

// right-preconditioned variant: t = A sh, partials (t . s), (t . t)
template <typename T>
__global__ void __launch_bounds__(256) spmv_dot2_pc_kernel(OpArgs a, const KrylovScalars *__restrict__ ks,
                                                           const T *__restrict__ sh, const T *__restrict__ s1,
                                                           T *__restrict__ tv, double *part) {
  if (ks->done) return;
  double acc[2] = {0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < a.N; base += stride) {
    const T y = op_apply_block<T>(a, base, sh);
    const int64_t r = base + threadIdx.x;
    if (r >= a.N) continue;
    ntstore(y, tv + r);
    acc[0] += (double)y * (double)s1[r];
    acc[1] += (double)y * (double)y;
  }
  block_partials<2>(acc, part);
}

// the same over SPE plane columns (FP64)
__global__ void __launch_bounds__(256) spe_spmv_dot2_pc_kernel(OpArgs a, SpeTiles T,
                                                               const KrylovScalars *__restrict__ ks,
                                                               const double *__restrict__ sh,
                                                               const double *__restrict__ s1, double *__restrict__ tv,
                                                               double *part) {
  if (ks->done) return;
  double acc[2] = {0.0, 0.0};
  const SpeColumn c = spe_column(a, T);
  if (c.ok) {
    const int64_t nynz = (int64_t)a.nyc * a.nzc, col = (int64_t)c.j * a.nzc + c.k;
    double w[SPE_PLANES];
    spe_plane_values(a, c, s1, w);
    double y[SPE_PLANES], xc[SPE_PLANES];
    const int np = spe_column_rows(a, c, sh, y, xc);
#pragma unroll
    for (int p = 0; p < SPE_PLANES; ++p)
      if (p < np) {
        const int64_t r = (int64_t)(c.i0 + p) * nynz + col;
        ntstore(y[p], tv + r);
        acc[0] += y[p] * w[p];
        acc[1] += y[p] * y[p];
      }
  }
  block_partials<2>(acc, part);
}

// x += alpha ph + omega sh; r = s - omega t; partials (r . r), (r . r0)
template <typename T>
__global__ void __launch_bounds__(256) xr_update_pc_kernel(int64_t N, const KrylovScalars *__restrict__ ks,
                                                           T *__restrict__ x, const T *__restrict__ ph,
                                                           const T *__restrict__ sh, const T *__restrict__ s1,
                                                           const T *__restrict__ tv, T *__restrict__ r1,
                                                           const T *__restrict__ r0, double *part) {
  if (ks->done) return;
  const double alpha = ks->alpha, omega = ks->omega;
  double acc[2] = {0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += stride) {
    ntstore((T)((double)x[r] + fma(alpha, (double)ph[r], omega * (double)sh[r])), x + r);
    const T rn = (T)((double)s1[r] - omega * (double)tv[r]);
    ntstore(rn, r1 + r);
    acc[0] += (double)rn * (double)rn;
    acc[1] += (double)rn * (double)r0[r];
  }
  block_partials<2>(acc, part);
}

// ---- the same updates with the reduction before them in each block ----------
// A finalize kernel is one block: 3 to 6 us, most of it a launch and two round
// trips to memory.  Small systems' updates combine the partials themselves, in
// every block, while their rows are on their way from memory.  The scalars
// then need two copies: ks[0] is read by K1 and written by K5, ks[1] is read
// by K3, K4 and K5 and written by K2 (all of it) and K4 (omega), so that no
// kernel writes what its blocks read.
// row r0 + u * step of a thread, clamped into the system (loads past it are not used)
__device__ inline int64_t fold_row(int64_t r0, int u, int64_t step, int64_t N) {
  const int64_t r = r0 + u * step;
  return r < N ? r : N - 1;
}

template <typename T, int BT, int ROWS, int C>
__global__ void __launch_bounds__(BT, BT == 1024 ? 8 : 4) s_fold_kernel(int64_t N, const double *part, int nblk,
                                                                    const KrylovScalars *__restrict__ ks0,
                                                                    KrylovScalars *ks1, const T *__restrict__ r1,
                                                                    const T *__restrict__ ap, T *__restrict__ s1) {
  const int64_t step = (int64_t)gridDim.x * BT, t = (int64_t)blockIdx.x * BT + threadIdx.x;
  T rv[ROWS], av[ROWS];
#pragma unroll
  for (int u = 0; u < ROWS; ++u) {
    const int64_t r = fold_row(t, u, step, N);
    rv[u] = r1[r];
    av[u] = ap[r];
  }
  double tot[1];
  combine_folded<BT, C>(part, nblk, tot);
  const int done = ks0->done;
  const double alpha = ks0->rho / tot[0];
  if (t == 0) begin_iteration(ks0, ks1, alpha);
  if (done) return;
#pragma unroll
  for (int u = 0; u < ROWS; ++u)
    if (t + u * step < N) s1[t + u * step] = (T)((double)rv[u] - alpha * (double)av[u]);
}

// xr_update_kernel (PC: xr_update_pc_kernel, with ph and sh in the places of
// p and s) of ROWS rows a thread, with that kernel's blocks and partials
template <typename T, bool PC, int ROWS>
__global__ void __launch_bounds__(256, 4)
    xr_fold_kernel(int64_t N, const double *dots, int nblk, KrylovScalars *ks1, T *__restrict__ x,
                   const T *__restrict__ ph, const T *__restrict__ sh, const T *__restrict__ s1,
                   const T *__restrict__ as, T *__restrict__ r1, const T *__restrict__ r0, double *part) {
  const int64_t step = (int64_t)gridDim.x * 256, t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  T xv[ROWS], pv[ROWS], hv[ROWS], sv[ROWS], av[ROWS], zv[ROWS];
#pragma unroll
  for (int u = 0; u < ROWS; ++u) {
    const int64_t r = fold_row(t, u, step, N);
    sv[u] = s1[r];
    av[u] = as[r];
    xv[u] = x[r];
    pv[u] = ph[r];
    hv[u] = PC ? sh[r] : T(0);
    zv[u] = r0[r];
  }
  double tot[2];
  combine_folded<256, 1>(dots, nblk, tot);
  if (ks1->done) return;
  const double alpha = ks1->alpha, omega = tot[0] / tot[1];
  if (blockIdx.x == 0 && threadIdx.x == 0) ks1->omega = omega;
  double acc[2] = {0.0, 0.0};
#pragma unroll
  for (int u = 0; u < ROWS; ++u) {
    const int64_t r = t + u * step;
    if (r < N) {
      const double s = (double)sv[u];
      const double d = PC ? fma(alpha, (double)pv[u], omega * (double)hv[u]) : fma(omega, s, alpha * (double)pv[u]);
      ntstore((T)((double)xv[u] + d), x + r);
      const T rn = (T)(s - omega * (double)av[u]);
      ntstore(rn, r1 + r);
      acc[0] += (double)rn * (double)rn;
      acc[1] += (double)rn * (double)zv[u];
    }
  }
  block_partials<2>(acc, part);
}

template <typename T, int ROWS>
__global__ void __launch_bounds__(256, 4) p_fold_kernel(int64_t N, const double *part, int nblk,
                                                                    const KrylovScalars *__restrict__ ks1,
                                                                    KrylovScalars *ks0, const T *__restrict__ r1,
                                                                    T *__restrict__ p1, const T *__restrict__ ap,
                                                                    T *__restrict__ r0) {
  const int64_t step = (int64_t)gridDim.x * 256, t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  T rv[ROWS], pv[ROWS], av[ROWS];
#pragma unroll
  for (int u = 0; u < ROWS; ++u) {
    const int64_t r = fold_row(t, u, step, N);
    rv[u] = r1[r];
    pv[u] = p1[r];
    av[u] = ap[r];
  }
  double tot[2];
  combine_folded<256, 1>(part, nblk, tot);
  if (ks1->done) return;
  const ConvNext n = conv_next(ks1, tot[0], tot[1]);
  const double omega = ks1->omega;
  if (t == 0) conv_store(ks1, ks0, n, tot[1]);
  if (n.stop) return;
#pragma unroll
  for (int u = 0; u < ROWS; ++u) {
    const int64_t r = t + u * step;
    if (r < N) {
      if (n.restart) {
        r0[r] = rv[u];
        p1[r] = rv[u];
      } else {
        p1[r] = (T)((double)rv[u] + n.beta * ((double)pv[u] - omega * (double)av[u]));
      }
    }
  }
}

// How an iteration's reductions run, for nd partials of each of the dots of
// K1 and K3 and nvb of K4's.  ALL: in K2, K4 and K5, up to 1024 partials each;
// K2: in K2 alone, by blocks of 1024 threads, up to 4096 partials; NONE.
// SPE iteration: 64x32x32 37 -> 23.5 us (ALL), 128x64x48 42 -> 29.5 (ALL),
// 200x104x40 60 -> 47.5 (ALL), 190x210x40 81 -> 70 (K2).  K4 and K5 folded at
// 190x210x40 take 22.7 + 14.8 us in blocks of 1024 threads that are all in
// flight at once, unfolded 3.7 + 17.0 + 4.3 + 11.5: the rows wait for the
// reduction, then all are stored at once.  The same holds K2 back where its
// blocks are more than the CUs take at once (two each, 4096 rows a block):
// 41.7 us at 512x256x64 with 4096 partials, 33 + 3.7 unfolded.  Past 4096
// partials every block would read more than 33 KB of them.
enum class Fold { NONE, K2, ALL };
constexpr int64_t FOLD_K2_ROWS = 512 * 4096;
Fold fold_of(int nd, int nvb, int64_t N) {
  if (nd <= FIN_THREADS && nvb <= FIN_THREADS) return Fold::ALL;
  return nd <= 4 * FIN_THREADS && N <= FOLD_K2_ROWS ? Fold::K2 : Fold::NONE;
}

template <typename T>
void launch_s_fold(Fold fold, int64_t N, const double *d1, int nd, KrylovScalars *ks, const T *r1, const T *ap, T *s1,
                   hipStream_t st) {
  auto blocks = [N](int rows) { return (unsigned)((N + rows - 1) / rows); };
  if (fold == Fold::K2)
    with_slots(nd, [&](auto c) {
      constexpr int C = decltype(c)::value > 0 ? decltype(c)::value : 4;
      s_fold_kernel<T, 1024, 4, C><<<blocks(4096), 1024, 0, st>>>(N, d1, nd, ks, ks + 1, r1, ap, s1);
    });
  else if (N <= 512 * 1024)
    s_fold_kernel<T, 256, 2, 1><<<blocks(512), 256, 0, st>>>(N, d1, nd, ks, ks + 1, r1, ap, s1);
  else
    s_fold_kernel<T, 256, 4, 1><<<blocks(1024), 256, 0, st>>>(N, d1, nd, ks, ks + 1, r1, ap, s1);
}

template <typename T>
void launch_p_fold(int64_t N, const double *part, int nvb, KrylovScalars *ks, const T *r1, T *p1, const T *ap, T *r0,
                   hipStream_t st) {
  if (N <= 512 * 1024)
    p_fold_kernel<T, 2><<<(unsigned)((N + 511) / 512), 256, 0, st>>>(N, part, nvb, ks + 1, ks, r1, p1, ap, r0);
  else
    p_fold_kernel<T, 4><<<(unsigned)((N + 1023) / 1024), 256, 0, st>>>(N, part, nvb, ks + 1, ks, r1, p1, ap, r0);
}

// NaN / Inf reset after iters_max (bicgstabRe2.hpp:143-163)
__global__ void __launch_bounds__(256) nan_reset_kernel(int64_t N, double *__restrict__ x,
                                                        const double *__restrict__ px1, double *part) {
  double acc[1] = {0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += stride) {
    const double v = x[r];
    if (isnan(v) || isinf(v)) {
      x[r] = px1[r];
      acc[0] += 1.0;
    }
  }
  block_partials<1>(acc, part);
}

template <int NV>
__global__ void __launch_bounds__(FIN_THREADS) sum_finalize(const double *part, int nblk, double *out) {
  double tot[NV];
  combine_partials<NV>(part, nblk, tot);
  if (threadIdx.x == 0)
    for (int q = 0; q < NV; ++q) out[q] = tot[q];
}

// defect correction: r = b - A64 x in FP64, r32 = (float) r, partials (r.r), (b.b)
__global__ void __launch_bounds__(256) dc_residual_kernel(OpArgs a, const double *__restrict__ b,
                                                          const double *__restrict__ x, float *__restrict__ r32,
                                                          double *part) {
  double acc[2] = {0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < a.N; base += stride) {
    const double ax = op_row_block(a, base, x);
    const int64_t r = base + threadIdx.x;
    if (r >= a.N) continue;
    const double br = b[r];
    const double rr = br - ax;
    r32[r] = (float)rr;
    acc[0] += rr * rr;
    acc[1] += br * br;
  }
  block_partials<2>(acc, part);
}

__global__ void __launch_bounds__(256) dc_update_kernel(int64_t N, double *__restrict__ x, float *__restrict__ d) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += stride) {
    x[r] += (double)d[r];
    d[r] = 0.0f;
  }
}

__global__ void __launch_bounds__(256) fill32_kernel(float *__restrict__ a, float v, int64_t n) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) a[t] = v;
}

template <typename T>
struct Vecs {
  T *x, *r0, *r1, *p1, *s1, *ap, *as;
  const T *b;
  double *px1, *px2;
};

// threads a block of the iteration's SpMV-dot kernels (ELL and SPE-as-rows
// operators): 512 halves the partials of 256-thread blocks at the same rows
// a thread
constexpr int SPMV_DOT_THREADS = 512;

template <typename T>
hipError_t launch_iters(Ctx &c, const OpArgs &a, const Vecs<T> &v, KrylovScalars *ks, int nit) {
  const int64_t N = c.g.N;
  // The SpMV-dots run SPMV_DOT_THREADS-thread blocks (256 on the CSR
  // operator) and the x / r update four rows a thread, which cuts the
  // partials their one-block finalize kernels combine; the s / p updates
  // take two rows a thread (3% faster streams).
  const bool wide = a.op != CFD_OP_CSR;
  const int nb = blocks_for(N, wide ? SPMV_DOT_THREADS : 256, RED_MAX_BLOCKS);
  const int nbu = blocks_for(N, 2 * 256, RED_MAX_BLOCKS), nbx = blocks_for(N, 4 * 256, RED_MAX_BLOCKS);
  double *p1 = red_part_host(c, RS_SPMV_DOT), *p2 = red_part_host(c, RS_SPMV_DOT2), *p3 = red_part_host(c, RS_XR);
  // the SPE operator's SpMV-dot kernels over plane columns (FP64)
  const SpeTiles tiles = spe_tiles(c.g.nxc, c.g.nyc, c.g.nzc);
  const bool spe = std::is_same<T, double>::value && a.op == CFD_OP_SPE && tiles.blocks <= RED_MAX_BLOCKS;
  const bool pairs = spe && spe_pairs(a, tiles, {v.p1, v.ap, v.r0, v.s1, v.as});
  const int nbs = spe ? (int)tiles.blocks : nb;
  const int pp = std::is_same<T, double>::value ? ell_grid_period(a, nb, SPMV_DOT_THREADS, {v.p1, v.ap, v.r0, v.s1, v.as}) : 0;
  const Fold fold = fold_of(nbs, nbx, N);
  KrylovScalars *ks3 = fold == Fold::NONE ? ks : ks + 1;  // from K2 to K4
  for (int it = 0; it < nit; ++it) {
    if (pp)
      launch_ell_grid<SPMV_DOT_THREADS, 1>(a, pp, ks, reinterpret_cast<const double *>(v.p1),
                                               reinterpret_cast<double *>(v.ap),
                                               reinterpret_cast<const double *>(v.r0), p1, c.stream);
    else if (pairs)
      launch_spe_walk<1>(a, tiles, ks, reinterpret_cast<const double *>(v.p1), reinterpret_cast<double *>(v.ap),
                         reinterpret_cast<const double *>(v.r0), p1, c.stream);
    else if (spe)
      spe_spmv_dot_kernel<<<nbs, 256, 0, c.stream>>>(a, tiles, ks, reinterpret_cast<const double *>(v.p1),
                                                     reinterpret_cast<double *>(v.ap),
                                                     reinterpret_cast<const double *>(v.r0), p1);
    else if (wide)
      spmv_dot_kernel<T, SPMV_DOT_THREADS><<<nb, SPMV_DOT_THREADS, 0, c.stream>>>(a, ks, v.p1, v.ap, v.r0, p1);
    else
      spmv_dot_kernel<T><<<nb, 256, op_lds_bytes(a), c.stream>>>(a, ks, v.p1, v.ap, v.r0, p1);
    if (fold != Fold::NONE) {
      launch_s_fold<T>(fold, N, p1, nbs, ks, v.r1, v.ap, v.s1, c.stream);
    } else {
      launch_alpha_finalize(p1, nbs, ks, c.stream);
      s_update_kernel<T><<<nbu, 256, 0, c.stream>>>(N, ks, v.r1, v.ap, v.s1);
    }
    if (pp)
      launch_ell_grid<SPMV_DOT_THREADS, 2>(a, pp, ks3, reinterpret_cast<const double *>(v.s1),
                                               reinterpret_cast<double *>(v.as), nullptr, p2, c.stream);
    else if (pairs)
      launch_spe_walk<2>(a, tiles, ks3, reinterpret_cast<const double *>(v.s1), reinterpret_cast<double *>(v.as),
                         nullptr, p2, c.stream);
    else if (spe)
      spe_spmv_dot2_kernel<<<nbs, 256, 0, c.stream>>>(a, tiles, ks3, reinterpret_cast<const double *>(v.s1),
                                                      reinterpret_cast<double *>(v.as), p2);
    else if (wide)
      spmv_dot2_kernel<T, SPMV_DOT_THREADS><<<nb, SPMV_DOT_THREADS, 0, c.stream>>>(a, ks3, v.s1, v.as, p2);
    else
      spmv_dot2_kernel<T><<<nb, 256, op_lds_bytes(a), c.stream>>>(a, ks3, v.s1, v.as, p2);
    if (fold == Fold::ALL) {
      xr_fold_kernel<T, false, 4><<<nbx, 256, 0, c.stream>>>(N, p2, nbs, ks3, v.x, v.p1, nullptr, v.s1, v.as, v.r1, v.r0,
                                                             p3);
      launch_p_fold<T>(N, p3, nbx, ks, v.r1, v.p1, v.ap, v.r0, c.stream);
      continue;
    }
    launch_omega_finalize(p2, nbs, ks3, c.stream);
    xr_update_kernel<T><<<nbx, 256, 0, c.stream>>>(N, ks3, v.x, v.p1, v.s1, v.as, v.r1, v.r0, p3);
    launch_conv_finalize(p3, nbx, ks3, ks, c.stream);
    p_update_kernel<T><<<nbu, 256, 0, c.stream>>>(N, ks, v.r1, v.p1, v.ap, v.r0);
  }
  return hipGetLastError();
}

// The iterations of an FP64 solve on the ELL operator in one launch
// (dev_resident.h) where its rows fit the chip's registers; the state after
// init_kernel is the launch path's and so is every result, bit for bit.
// *solved is false when the launch path has to go on from where the state is:
// the system is too large, a workgroup's halo does not fit, or the CUs are
// taken; *lost, when it has to start again, from the x that is back in place: a
// wait reached its bound.
// The limit is what the registers of 256 one-workgroup CUs hold (RES_MAX_N,
// 524288 rows); it is the faster path over that whole range (at the limit
// 21.0 us an iteration against 29.9, at one workgroup 4.6 against 20.0).
int solve_resident(Ctx &c, const OpArgs &a, const Vecs<double> &v, KrylovScalars *ks, bool *solved, bool *lost) {
  *solved = *lost = false;
  if ((a.op != CFD_OP_ELL && a.op != OP_ELL_GRID) || a.N > RES_MAX_N) return CFD_OK;
  ResArgs r;
  r.N = a.N;
  r.nbx = blocks_for(a.N, 4 * 256, RED_MAX_BLOCKS);
  r.S = (int64_t)r.nbx * 256;
  r.nblk = (int)((r.S + RES_THREADS - 1) / RES_THREADS);
  r.sliced = a.sliced;
  r.col = a.col;
  r.val = a.val;
  r.x = v.x;
  r.r0 = v.r0;
  r.r1 = v.r1;
  r.p1 = v.p1;
  // the launch path's s, A p and A s are its only users of these vectors
  r.ll0 = reinterpret_cast<uint64_t *>(v.s1);
  r.ll1 = reinterpret_cast<uint64_t *>(v.ap);
  r.keep = v.as;
  static_assert(2 * RES_RED_WORDS <= 3 * RED_MAX_BLOCKS, "an exchanged sum fits its site's partials");
  const int sites[3] = {RS_SPMV_DOT, RS_SPMV_DOT2, RS_XR};
  for (int q = 0; q < 3; ++q) r.red[q] = reinterpret_cast<uint64_t *>(red_part_host(c, sites[q]));
  r.ks = ks;
  r.chunk = 4096;  // bounds one launch to some tens of milliseconds
  r.bounds = res_bounds(c.one);
  ResidentSlots slots;
  if (!c.one.due()) return CFD_OK;
  if (!slots.take(c.device, r.nblk)) {
    c.one.handed_back++;
    return CFD_OK;
  }
  const int nbc = blocks_for(std::max<int64_t>(a.N, 2 * RES_RED_WORDS), 256, 1 << 30);
  for (bool first = true;; first = false) {
    resident_clear_kernel<<<nbc, 256, 0, c.stream>>>(r, first);
    if (r.bounds.set)
      bicg_resident_kernel<true><<<r.nblk, RES_THREADS, 0, c.stream>>>(r);
    else
      bicg_resident_kernel<false><<<r.nblk, RES_THREADS, 0, c.stream>>>(r);
    CFD_HIP(hipGetLastError());
    CFD_HIP(hipMemcpyAsync(c.hks, ks, sizeof(KrylovScalars), hipMemcpyDeviceToHost, c.stream));
    CFD_HIP(hipStreamSynchronize(c.stream));
    if (c.hks->pad1 != RES_GO) {
      if (c.hks->pad1 == RES_STUCK) {
        resident_restore_kernel<<<nbc, 256, 0, c.stream>>>(r);
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

// Generic driver: set up scalars, r0 = b - A x, then batches of iterations
// with one host read of the scalars per batch.  The batch length follows
// the observed convergence rate so that few no-op launches follow the
// converged iteration.
template <typename T>
int solve_bicg(Ctx &c, const OpArgs &a, const Vecs<T> &v, KrylovScalars *ks, int timestep, double tol, int maxit,
               int *iters, double *relres) {
  const int64_t N = c.g.N;
  const int nb = blocks_for(N, 256, RED_MAX_BLOCKS);
  auto init = [&](double *px1, double *px2) {
    ks_setup_kernel<<<1, 1, 0, c.stream>>>(ks, tol, 1e-7 * tol, maxit, timestep);
    init_kernel<T><<<nb, 256, op_lds_bytes(a), c.stream>>>(a, v.b, v.x, v.r0, v.r1, v.p1, px1, px2,
                                                        red_part_host(c, RS_INIT));
    init_finalize<<<1, FIN_THREADS, 0, c.stream>>>(red_part_host(c, RS_INIT), nb, ks);
    return hipGetLastError();
  };
  CFD_HIP(init(v.px1, v.px2));
  bool solved = false;
  if constexpr (std::is_same<T, double>::value) {
    bool lost = false;
    if (int rc = solve_resident(c, a, v, ks, &solved, &lost)) return rc;
    if (lost) CFD_HIP(init(nullptr, nullptr));  // the history has its entry
  }
  int batch = 2;
  double prev_rel = -1.0;
  int prev_it = 0;
  while (!solved) {
    CFD_HIP(launch_iters<T>(c, a, v, ks, batch));
    CFD_HIP(hipMemcpyAsync(c.hks, ks, sizeof(KrylovScalars), hipMemcpyDeviceToHost, c.stream));
    CFD_HIP(hipStreamSynchronize(c.stream));
    const KrylovScalars h = *c.hks;
    if (h.done) break;
    // predict the iterations still needed from the last batch's rate
    int next = batch * 2;
    if (prev_rel > 0.0 && h.relres > 0.0 && h.relres < prev_rel && h.iters > prev_it) {
      const double rate = std::log(h.relres / prev_rel) / (double)(h.iters - prev_it);
      const double need = std::log(h.tol / h.relres) / rate;
      if (need > 0.0 && std::isfinite(need)) next = (int)std::ceil(need * 1.05) + 1;
    }
    prev_rel = h.relres;
    prev_it = h.iters;
    next = std::max(1, std::min(next, 64));
    next = std::min(next, maxit - h.iters + 1);
    batch = std::max(next, 1);
  }
  const KrylovScalars h = *c.hks;
  if (h.hit_maxit && v.px1) {
    double *part = red_part_host(c, RS_MISC);
    nan_reset_kernel<<<nb, 256, 0, c.stream>>>(N, (double *)v.x, v.px1, part);
    sum_finalize<1><<<1, FIN_THREADS, 0, c.stream>>>(part, nb, c.red.out + RS_MISC * 4);
    CFD_HIP(hipMemcpyAsync(c.hred, c.red.out + RS_MISC * 4, sizeof(double), hipMemcpyDeviceToHost, c.stream));
    CFD_HIP(hipStreamSynchronize(c.stream));
    if (c.hred[0] > (double)N * 0.1) {
      if (v.px2) CFD_HIP(hipMemcpyAsync(v.x, v.px2, sizeof(double) * N, hipMemcpyDeviceToDevice, c.stream));
      else CFD_HIP(launch_fill(c, (double *)v.x, 0.0, N));
    }
    if (c.hred[0] > 0.0 && ks == c.ks) c.nan_resets++;
  }
  if (ks == c.ks) c.total_iters += h.iters;
  *iters = h.iters;
  *relres = h.relres;
  return CFD_OK;
}

// BiCGSTAB right-preconditioned by the multigrid V-cycle (an addition; the
// reference's bicgstabRe2 is Jacobi-scaled only):
//   ph = M p; v = A ph; alpha = rho / (v . r0); s = r - alpha v;
//   sh = M s; t = A sh; omega = (t . s) / (t . t);
//   x += alpha ph + omega sh; r = s - omega t; beta; p = r + beta (p - omega v)
// with the fused kernels and device-side scalars of the plain solve.
template <typename T>
struct PVecs {
  T *x, *r0, *r1, *p1, *s1, *v, *t, *ph, *sh;
  const T *b;
};

template <typename T>
int mg_apply_t(Ctx &c, const T *r, T *out, const KrylovScalars *ks);
template <>
int mg_apply_t<double>(Ctx &c, const double *r, double *out, const KrylovScalars *ks) {
  return mg_apply64(c, r, out, ks);
}
template <>
int mg_apply_t<float>(Ctx &c, const float *r, float *out, const KrylovScalars *ks) {
  return mg_apply32(c, r, out, ks);
}

// the preconditioner: the V-cycle in the vectors' precision, or (pc32, FP64
// vectors only) in FP32
template <typename T>
int precondition(Ctx &c, const T *r, T *out, const KrylovScalars *ks, bool pc32) {
  if constexpr (std::is_same<T, double>::value) {
    if (pc32) return mg_apply64_fp32cycle(c, r, out, ks);
  }
  return mg_apply_t<T>(c, r, out, ks);
}

template <typename T>
int launch_pc_iters(Ctx &c, const OpArgs &a, const PVecs<T> &v, KrylovScalars *ks, int nit, bool pc32) {
  const int64_t N = c.g.N;
  const int nb = blocks_for(N, 256, RED_MAX_BLOCKS);
  double *p1 = red_part_host(c, RS_SPMV_DOT), *p2 = red_part_host(c, RS_SPMV_DOT2), *p3 = red_part_host(c, RS_XR);
  const int nbu = blocks_for(N, 2 * 256, RED_MAX_BLOCKS);  // two rows a thread, as in launch_iters
  // the SPE operator's kernels over plane columns (FP64), as in launch_iters
  const SpeTiles tiles = spe_tiles(c.g.nxc, c.g.nyc, c.g.nzc);
  const bool spe = std::is_same<T, double>::value && a.op == CFD_OP_SPE && tiles.blocks <= RED_MAX_BLOCKS;
  const bool pairs = spe && spe_pairs(a, tiles, {v.ph, v.v, v.r0, v.sh, v.t, v.s1});
  const int nbs = spe ? (int)tiles.blocks : nb;
  const int pp = std::is_same<T, double>::value ? ell_grid_period(a, nb, 256, {v.ph, v.v, v.r0, v.sh, v.t, v.s1}) : 0;
  const Fold fold = fold_of(nbs, nbu, N);
  KrylovScalars *ks3 = fold == Fold::NONE ? ks : ks + 1;  // from K2 to K4
  for (int it = 0; it < nit; ++it) {
    int rc = precondition<T>(c, v.p1, v.ph, ks, pc32);
    if (rc) return rc;
    if (pp)
      launch_ell_grid<256, 1>(a, pp, ks, reinterpret_cast<const double *>(v.ph), reinterpret_cast<double *>(v.v),
                                  reinterpret_cast<const double *>(v.r0), p1, c.stream);
    else if (pairs)
      launch_spe_walk<1>(a, tiles, ks, reinterpret_cast<const double *>(v.ph), reinterpret_cast<double *>(v.v),
                         reinterpret_cast<const double *>(v.r0), p1, c.stream);
    else if (spe)
      spe_spmv_dot_kernel<<<nbs, 256, 0, c.stream>>>(a, tiles, ks, reinterpret_cast<const double *>(v.ph),
                                                     reinterpret_cast<double *>(v.v),
                                                     reinterpret_cast<const double *>(v.r0), p1);
    else
      spmv_dot_kernel<T><<<nb, 256, op_lds_bytes(a), c.stream>>>(a, ks, v.ph, v.v, v.r0, p1);
    if (fold != Fold::NONE) {
      launch_s_fold<T>(fold, N, p1, nbs, ks, v.r1, v.v, v.s1, c.stream);
    } else {
      launch_alpha_finalize(p1, nbs, ks, c.stream);
      s_update_kernel<T><<<nbu, 256, 0, c.stream>>>(N, ks, v.r1, v.v, v.s1);
    }
    if ((rc = precondition<T>(c, v.s1, v.sh, ks3, pc32))) return rc;
    if (pp)
      launch_ell_grid<256, 3>(a, pp, ks3, reinterpret_cast<const double *>(v.sh), reinterpret_cast<double *>(v.t),
                                  reinterpret_cast<const double *>(v.s1), p2, c.stream);
    else if (pairs)
      launch_spe_walk<3>(a, tiles, ks3, reinterpret_cast<const double *>(v.sh), reinterpret_cast<double *>(v.t),
                         reinterpret_cast<const double *>(v.s1), p2, c.stream);
    else if (spe)
      spe_spmv_dot2_pc_kernel<<<nbs, 256, 0, c.stream>>>(a, tiles, ks3, reinterpret_cast<const double *>(v.sh),
                                                         reinterpret_cast<const double *>(v.s1),
                                                         reinterpret_cast<double *>(v.t), p2);
    else
      spmv_dot2_pc_kernel<T><<<nb, 256, op_lds_bytes(a), c.stream>>>(a, ks3, v.sh, v.s1, v.t, p2);
    if (fold == Fold::ALL) {
      xr_fold_kernel<T, true, 2><<<nbu, 256, 0, c.stream>>>(N, p2, nbs, ks3, v.x, v.ph, v.sh, v.s1, v.t, v.r1, v.r0, p3);
      launch_p_fold<T>(N, p3, nbu, ks, v.r1, v.p1, v.v, v.r0, c.stream);
      CFD_HIP(hipGetLastError());
      continue;
    }
    launch_omega_finalize(p2, nbs, ks3, c.stream);
    xr_update_pc_kernel<T><<<nbu, 256, 0, c.stream>>>(N, ks3, v.x, v.ph, v.sh, v.s1, v.t, v.r1, v.r0, p3);
    launch_conv_finalize(p3, nbu, ks3, ks, c.stream);
    p_update_kernel<T><<<nbu, 256, 0, c.stream>>>(N, ks, v.r1, v.p1, v.v, v.r0);
    CFD_HIP(hipGetLastError());
  }
  return CFD_OK;
}

template <typename T>
int solve_pbicg(Ctx &c, const OpArgs &a, const PVecs<T> &v, KrylovScalars *ks, double tol, int maxit, int *iters,
                double *relres, bool pc32 = false) {
  const int64_t N = c.g.N;
  const int nb = blocks_for(N, 256, RED_MAX_BLOCKS);
  ks_setup_kernel<<<1, 1, 0, c.stream>>>(ks, tol, 0.0, maxit, 0);
  init_kernel<T><<<nb, 256, op_lds_bytes(a), c.stream>>>(a, v.b, v.x, v.r0, v.r1, v.p1, nullptr, nullptr,
                                                      red_part_host(c, RS_INIT));
  init_finalize<<<1, FIN_THREADS, 0, c.stream>>>(red_part_host(c, RS_INIT), nb, ks);
  CFD_HIP(hipGetLastError());
  CFD_HIP(hipMemcpyAsync(c.hks, ks, sizeof(KrylovScalars), hipMemcpyDeviceToHost, c.stream));
  CFD_HIP(hipStreamSynchronize(c.stream));
  if (!(c.hks->relres >= tol)) {  // already converged (or a zero right-hand side)
    *iters = 0;
    *relres = c.hks->norm0 > 0.0 ? c.hks->relres : 0.0;
    return CFD_OK;
  }
  // Each preconditioned iteration is ~100 launches, so the batch follows the
  // observed convergence rate: launches after the converged iteration are
  // no-ops but still cost their launch latency.
  int batch = 1;
  double prev_rel = c.hks->relres;
  int prev_it = 0;
  for (;;) {
    int rc = launch_pc_iters<T>(c, a, v, ks, batch, pc32);
    if (rc) return rc;
    CFD_HIP(hipMemcpyAsync(c.hks, ks, sizeof(KrylovScalars), hipMemcpyDeviceToHost, c.stream));
    CFD_HIP(hipStreamSynchronize(c.stream));
    const KrylovScalars h = *c.hks;
    if (h.done) break;
    int next = 1;
    if (h.relres > 0.0 && h.relres < prev_rel && h.iters > prev_it) {
      const double rate = std::log(h.relres / prev_rel) / (double)(h.iters - prev_it);
      const double need = std::log(h.tol / h.relres) / rate;
      if (need > 0.0 && std::isfinite(need)) next = (int)std::floor(need);
    }
    prev_rel = h.relres;
    prev_it = h.iters;
    batch = std::max(1, std::min(next, 8));
  }
  *iters = c.hks->iters;
  *relres = c.hks->relres;
  return CFD_OK;
}

}  // namespace

int pbicgstab_solve_aux(Ctx &c, const double *b, double *x, double tol, int maxit, bool pc32, int *iters,
                        double *relres) {
  if (!c.ell_ready) return fail(CFD_ERR_STATE, "ELL operator not assembled");
  int rc = mg_ensure(c, pc32);
  if (!rc && pc32) rc = mg_ensure(c, false);  // the FP64 preconditioned directions
  if (rc) return rc;
  PVecs<double> v{x, c.r0, c.r1, c.p1, c.s1, c.ap, c.as, c.ph64, c.sh64, b};
  // the configured operator (ELL, matrix-free SPE or CSR); the V-cycle
  // approximates its inverse from the grid metrics
  return solve_pbicg<double>(c, op_args(c, fp64_op(c)), v, c.ks, tol, maxit, iters, relres, pc32);
}

int pbicgstab_solve64(Ctx &c, const double *b, double *x, double tol, int maxit, bool pc32, int *iters,
                      double *relres) {
  c.solves++;
  return pbicgstab_solve_aux(c, b, x, tol, maxit, pc32, iters, relres);
}

int bicgstab_solve(Ctx &c, const double *b, double *x, double tol, int maxit, int *iters, double *relres) {
  if (int rc = op_ready(c, c.prm.op)) return rc;
  c.solves++;
  Vecs<double> v{x, c.r0, c.r1, c.p1, c.s1, c.ap, c.as, b, c.px1, c.px2};
  return solve_bicg<double>(c, op_args(c, c.prm.op), v, c.ks, c.solves, tol, maxit, iters, relres);
}

int bicgstab_solve_aux(Ctx &c, const double *b, double *x, double tol, int maxit, int timestep, int *iters,
                       double *relres) {
  if (!c.ell_ready) return fail(CFD_ERR_STATE, "ELL operator not assembled");
  Vecs<double> v{x, c.r0, c.r1, c.p1, c.s1, c.ap, c.as, b, nullptr, nullptr};
  return solve_bicg<double>(c, op_args(c, CFD_OP_ELL), v, c.ks, timestep, tol, maxit, iters, relres);
}

// FP64 defect correction around FP32 BiCGSTAB on the FP32 ELL copy:
// r = b - A x (FP64), solve A32 d = r32 to tol_inner, x += d, until
// ||b - A x|| / ||b|| < tol.
int defect_correction(Ctx &c, const double *b, double *x, double tol, double tol_inner, int max_outer, int *outer,
                      int *inner_total, double *relres) {
  if (!c.ell_ready || !c.val32) return fail(CFD_ERR_STATE, "FP32 ELL operator not assembled");
  const int64_t N = c.g.N;
  const int nb = blocks_for(N, 256, RED_MAX_BLOCKS);
  const OpArgs a64 = op_args(c, fp64_op(c));
  const OpArgs a32 = op_args(c, CFD_OP_ELL);
  float *r32 = c.q32[7], *d32 = c.q32[6];
  Vecs<float> v{d32, c.q32[0], c.q32[1], c.q32[2], c.q32[3], c.q32[4], c.q32[5], r32, nullptr, nullptr};
  fill32_kernel<<<blocks_for(N, 256, 1 << 30), 256, 0, c.stream>>>(d32, 0.0f, N);
  CFD_HIP(hipGetLastError());
  int k = 0, inner = 0;
  double rel = 0.0;
  c.solves++;
  for (;;) {
    double *part = red_part_host(c, RS_NORM);
    dc_residual_kernel<<<nb, 256, op_lds_bytes(a64), c.stream>>>(a64, b, x, r32, part);
    sum_finalize<2><<<1, FIN_THREADS, 0, c.stream>>>(part, nb, c.red.out + RS_NORM * 4);
    CFD_HIP(hipGetLastError());
    CFD_HIP(hipMemcpyAsync(c.hred, c.red.out + RS_NORM * 4, 2 * sizeof(double), hipMemcpyDeviceToHost, c.stream));
    CFD_HIP(hipStreamSynchronize(c.stream));
    rel = std::sqrt(c.hred[0]) / std::sqrt(c.hred[1]);
    if (!(rel >= tol) || k >= max_outer) break;
    int it = 0;
    double rin = 0.0;
    c.solves32++;
    if (c.prm.precond == CFD_PRECOND_MG && c.prm.solver == CFD_SOLVER_BICGSTAB) {
      int rc = mg_ensure(c, true);
      if (rc) return rc;
      PVecs<float> pv{d32, c.q32[0], c.q32[1], c.q32[2], c.q32[3], c.q32[4], c.q32[5], c.ph32, c.sh32, r32};
      rc = solve_pbicg<float>(c, a32, pv, c.ks32, tol_inner, c.prm.maxit, &it, &rin);
      if (rc != CFD_OK) return rc;
    } else if (c.prm.solver == CFD_SOLVER_RBSOR) {
      int rc = rbsor_solve_f32(c, r32, d32, c.prm.sor_omega, tol_inner, c.prm.maxit, c.prm.sor_check, &it, &rin);
      if (rc != CFD_OK) return rc;
    } else {
      int rc = solve_bicg<float>(c, a32, v, c.ks32, c.solves32, tol_inner, c.prm.maxit, &it, &rin);
      if (rc != CFD_OK) return rc;
    }
    inner += it + 1;
    dc_update_kernel<<<nb, 256, 0, c.stream>>>(N, x, d32);
    CFD_HIP(hipGetLastError());
    ++k;
  }
  *outer = k;
  *inner_total = inner;
  *relres = rel;
  return CFD_OK;
}

// Timing of one iteration: the solver runs on scratch vectors (x = VEC_B
// starting from 0) with the stop test disabled; the warm-start history of the
// real solver (px1, px2, X) is not touched.
hipError_t launch_bicg_iteration(Ctx &c) {
  Vecs<double> v{c.f[CFD_VEC_B], c.r0, c.r1, c.p1, c.s1, c.ap, c.as, c.f[CFD_RHS], nullptr, nullptr};
  return launch_iters<double>(c, op_args(c, c.prm.op), v, c.ks32, 1);
}

// Timing of the iteration's first kernel alone (K1: ap = A p with the
// partial dot ap . r0), the iteration's largest share, on the same scratch
// vectors and scalars as launch_bicg_iteration
hipError_t launch_spmv_dot(Ctx &c) {
  const OpArgs a = op_args(c, c.prm.op);
  const SpeTiles tiles = spe_tiles(c.g.nxc, c.g.nyc, c.g.nzc);
  double *part = red_part_host(c, RS_SPMV_DOT);
  if (const int pp = ell_grid_period(a, blocks_for(c.g.N, SPMV_DOT_THREADS, RED_MAX_BLOCKS), SPMV_DOT_THREADS,
                                      {c.p1, c.ap, c.r0}))
    launch_ell_grid<SPMV_DOT_THREADS, 1>(a, pp, c.ks32, c.p1, c.ap, c.r0, part, c.stream);
  else if (a.op == CFD_OP_SPE && tiles.blocks <= RED_MAX_BLOCKS && spe_pairs(a, tiles, {c.p1, c.ap, c.r0}))
    launch_spe_walk<1>(a, tiles, c.ks32, c.p1, c.ap, c.r0, part, c.stream);
  else if (a.op == CFD_OP_SPE && tiles.blocks <= RED_MAX_BLOCKS)
    spe_spmv_dot_kernel<<<(int)tiles.blocks, 256, 0, c.stream>>>(a, tiles, c.ks32, c.p1, c.ap, c.r0, part);
  else if (a.op != CFD_OP_CSR)  // launch_iters' launch
    spmv_dot_kernel<double, SPMV_DOT_THREADS>
        <<<blocks_for(c.g.N, SPMV_DOT_THREADS, RED_MAX_BLOCKS), SPMV_DOT_THREADS, 0, c.stream>>>(a, c.ks32, c.p1,
                                                                                               c.ap, c.r0, part);
  else
    spmv_dot_kernel<double><<<blocks_for(c.g.N, 256, RED_MAX_BLOCKS), 256, op_lds_bytes(a), c.stream>>>(
        a, c.ks32, c.p1, c.ap, c.r0, part);
  return hipGetLastError();
}

hipError_t launch_bicg_timing_setup(Ctx &c) {
  const int64_t N = c.g.N;
  const int nb = blocks_for(N, 256, RED_MAX_BLOCKS);
  hipError_t e = launch_fill(c, c.f[CFD_VEC_B], 0.0, N);
  if (e != hipSuccess) return e;
  ks_setup_kernel<<<1, 1, 0, c.stream>>>(c.ks32, 0.0, 0.0, 1 << 30, 100);
  const OpArgs a = op_args(c, c.prm.op);
  init_kernel<double><<<nb, 256, op_lds_bytes(a), c.stream>>>(a, c.f[CFD_RHS], c.f[CFD_VEC_B], c.r0, c.r1, c.p1,
                                                              nullptr, nullptr, red_part_host(c, RS_INIT));
  init_finalize<<<1, FIN_THREADS, 0, c.stream>>>(red_part_host(c, RS_INIT), nb, c.ks32);
  return hipGetLastError();
}

}  // namespace cfd

// ---------------------------------------------------------------------------
// Mixed precision by reliable updates: BiCGSTAB iterates in FP32 (FP32 ELL
// values and vectors, FP64 accumulation in the operator and in every dot);
// the FP32 iterate xl is folded into the FP64 solution x and the FP32
// residual is replaced by the FP64 true residual b - A64 x whenever the
// recurrence residual has fallen by `delta` since the last replacement, and
// at the end.  The search direction and shadow residual are kept across a
// replacement, so the Krylov space is not restarted; the stop test is on the
// FP64 true residual, the same criterion as the FP64 solve.
// ---------------------------------------------------------------------------
namespace cfd {
namespace {

__global__ void set_delta_kernel(KrylovScalars *ks, double delta) { ks->delta = delta; }

// r = b - A64 x (FP64); rv = r0 = p = (T) r; xl = 0; partials (b.b), (r.r), (rv.rv)
template <typename T>
__global__ void __launch_bounds__(256) mr_init_kernel(OpArgs a64, const double *__restrict__ b,
                                                      const double *__restrict__ x, T *__restrict__ r32,
                                                      T *__restrict__ r0, T *__restrict__ p, T *__restrict__ xl,
                                                      double *part) {
  double acc[3] = {0.0, 0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < a64.N; base += stride) {
    const double ax = op_row_block(a64, base, x);
    const int64_t r = base + threadIdx.x;
    if (r >= a64.N) continue;
    const double br = b[r];
    const double rr = br - ax;
    const T rf = (T)rr;
    r32[r] = rf;
    r0[r] = rf;
    p[r] = rf;
    if (xl) xl[r] = T(0);
    acc[0] += br * br;
    acc[1] += rr * rr;
    acc[2] += (double)rf * (double)rf;
  }
  block_partials<3>(acc, part);
}

__global__ void __launch_bounds__(FIN_THREADS) mr_init_finalize(const double *part, int nblk, KrylovScalars *ks) {
  double tot[3];
  combine_partials<3>(part, nblk, tot);
  if (threadIdx.x == 0) {
    ks->norm0 = sqrt(tot[0]);
    ks->rmax = sqrt(tot[1]);
    ks->relres = ks->rmax / ks->norm0;
    ks->rho = tot[2];
    ks->replace = 0;
    ks->replacements = 0;
    ks->breakdown = 0;
    if (!(ks->relres >= ks->tol)) ks->done = 1;
  }
}

__global__ void __launch_bounds__(FIN_THREADS) mr_alpha_finalize(const double *part, int nblk, KrylovScalars *ks) {
  if (ks->done) return;
  double tot[1];
  combine_partials<1>(part, nblk, tot);
  if (threadIdx.x == 0) {
    const double a = ks->rho / tot[0];
    if (!isfinite(a)) {  // breakdown: fold what has been gained and re-anchor on the true residual
      ks->breakdown += 1;
      ks->replace = 1;
      ks->alpha = 0.0;
    } else {
      ks->alpha = a;
    }
  }
}

__global__ void __launch_bounds__(FIN_THREADS) mr_omega_finalize(const double *part, int nblk, KrylovScalars *ks) {
  if (ks->done || ks->replace) return;
  double tot[2];
  combine_partials<2>(part, nblk, tot);
  if (threadIdx.x == 0) {
    const double w = tot[0] / tot[1];
    ks->omega = isfinite(w) ? w : 0.0;
    if (!isfinite(w)) {
      ks->breakdown += 1;
      ks->replace = 1;
    }
  }
}

// recurrence residual test: trigger a replacement on a `delta` drop, on the
// stop criterion, or at the iteration cap; otherwise beta and the restart rule
__global__ void __launch_bounds__(FIN_THREADS) mr_conv_finalize(const double *part, int nblk, KrylovScalars *ks) {
  if (ks->done || ks->replace) return;
  double tot[2];
  combine_partials<2>(part, nblk, tot);
  if (threadIdx.x == 0) {
    const double rn = sqrt(tot[0]);
    ks->rnorm = rn;
    if (ks->iters >= ks->maxit) ks->hit_maxit = 1;
    if (rn < ks->delta * ks->rmax || rn / ks->norm0 < ks->tol || ks->hit_maxit || !isfinite(rn)) {
      ks->replace = 1;
    } else {
      ks->pre_rho = ks->rho;
      ks->rho = tot[1];
      ks->beta = (ks->alpha / ks->omega) * (ks->rho / ks->pre_rho);
      ks->restart = (ks->timestep < 10 || fabs(ks->pre_rho) > ks->restart_tol) ? 0 : 1;
      ks->restarts += ks->restart;
      ks->iters += 1;
    }
  }
}

// x += xl; xl = 0 (only when a replacement is due)
__global__ void __launch_bounds__(256) mr_fold_kernel(int64_t N, const KrylovScalars *__restrict__ ks,
                                                      double *__restrict__ x, float *__restrict__ xl) {
  if (ks->done || !ks->replace) return;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += stride) {
    x[r] += (double)xl[r];
    xl[r] = 0.0f;
  }
}

// rv = (T)(b - A64 x); partials (r.r) in FP64, (rv.r0)
template <typename T>
__global__ void __launch_bounds__(256) mr_replace_kernel(OpArgs a64, const KrylovScalars *__restrict__ ks,
                                                         const double *__restrict__ b, const double *__restrict__ x,
                                                         T *__restrict__ r32, const T *__restrict__ r0,
                                                         double *part) {
  if (ks->done || !ks->replace) return;
  double acc[2] = {0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < a64.N; base += stride) {
    const double ax = op_row_block(a64, base, x);
    const int64_t r = base + threadIdx.x;
    if (r >= a64.N) continue;
    const double rr = b[r] - ax;
    const T rf = (T)rr;
    r32[r] = rf;
    acc[0] += rr * rr;
    acc[1] += (double)rf * (double)r0[r];
  }
  block_partials<2>(acc, part);
}

__global__ void __launch_bounds__(FIN_THREADS) mr_replace_finalize(const double *part, int nblk, KrylovScalars *ks) {
  if (ks->done || !ks->replace) return;
  double tot[2];
  combine_partials<2>(part, nblk, tot);
  if (threadIdx.x == 0) {
    const double rt = sqrt(tot[0]);
    ks->replacements += 1;
    ks->relres = rt / ks->norm0;
    ks->replace = 0;
    if (ks->relres < ks->tol || ks->hit_maxit || ks->breakdown > 8) {
      ks->done = 1;
      return;
    }
    const bool broke = !(ks->alpha != 0.0 && ks->omega != 0.0);
    ks->rmax = rt;
    ks->pre_rho = ks->rho;
    ks->rho = tot[1];
    ks->beta = broke ? 0.0 : (ks->alpha / ks->omega) * (ks->rho / ks->pre_rho);
    ks->restart = broke ? 1 : ((ks->timestep < 10 || fabs(ks->pre_rho) > ks->restart_tol) ? 0 : 1);
    ks->restarts += ks->restart;
    ks->iters += 1;
  }
}

// p update, shared by both branches: runs unless the solve is done
template <typename T>
__global__ void __launch_bounds__(256) mr_p_update_kernel(int64_t N, const KrylovScalars *__restrict__ ks,
                                                          const T *__restrict__ r1, T *__restrict__ p1,
                                                          const T *__restrict__ ap, T *__restrict__ r0) {
  if (ks->done) return;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  if (ks->restart) {
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += stride) {
      r0[r] = r1[r];
      p1[r] = r1[r];
    }
    return;
  }
  const double beta = ks->beta, omega = ks->omega;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += stride)
    p1[r] = (T)((double)r1[r] + beta * ((double)p1[r] - omega * (double)ap[r]));
}

// the kernels of one iteration skip their work while a replacement is pending
template <typename T>
__global__ void __launch_bounds__(256) mr_s_update_kernel(int64_t N, const KrylovScalars *__restrict__ ks,
                                                          const T *__restrict__ r1, const T *__restrict__ ap,
                                                          T *__restrict__ s1) {
  if (ks->done || ks->replace) return;
  const double alpha = ks->alpha;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += stride)
    s1[r] = (T)((double)r1[r] - alpha * (double)ap[r]);
}

template <typename T>
__global__ void __launch_bounds__(256) mr_spmv_dot2_kernel(OpArgs a, const KrylovScalars *__restrict__ ks,
                                                           const T *__restrict__ s1, T *__restrict__ as,
                                                           double *part) {
  if (ks->done || ks->replace) return;
  double acc[2] = {0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < a.N; r += stride) {
    const T y = op_apply<T>(a, r, s1);
    ntstore(y, as + r);
    acc[0] += (double)y * (double)s1[r];
    acc[1] += (double)y * (double)y;
  }
  block_partials<2>(acc, part);
}

template <typename T, typename TX>
__global__ void __launch_bounds__(256) mr_xr_update_kernel(int64_t N, const KrylovScalars *__restrict__ ks,
                                                           TX *__restrict__ xl, const T *__restrict__ p1,
                                                           const T *__restrict__ s1, const T *__restrict__ as,
                                                           T *__restrict__ r1, const T *__restrict__ r0,
                                                           double *part) {
  if (ks->done || ks->replace) return;
  const double alpha = ks->alpha, omega = ks->omega;
  double acc[2] = {0.0, 0.0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < N; r += stride) {
    const double s = (double)s1[r];
    xl[r] = (TX)((double)xl[r] + (alpha * (double)p1[r] + omega * s));
    const T rn = (T)(s - omega * (double)as[r]);
    r1[r] = rn;
    acc[0] += (double)rn * (double)rn;
    acc[1] += (double)rn * (double)r0[r];
  }
  block_partials<2>(acc, part);
}

// T = float: FP32 vectors, FP32 iterate xl folded into the FP64 x.
// T = double: FP64 vectors on the FP32-valued operator; x updated directly.
template <typename T>
int reliable_solve(Ctx &c, const double *b, double *x, double tol, double delta, int maxit, int *replacements,
                   int *iters, double *relres) {
  if (!c.ell_ready || !c.val32) return fail(CFD_ERR_STATE, "FP32 ELL operator not assembled");
  const int64_t N = c.g.N;
  const int nb = blocks_for(N, 256, RED_MAX_BLOCKS);
  const OpArgs a64 = op_args(c, fp64_op(c));
  const OpArgs ain = op_args(c, std::is_same<T, float>::value ? CFD_OP_ELL : OP_ELL_VAL32);
  T *r0, *r1, *p1, *s1, *ap, *as;
  if constexpr (std::is_same<T, float>::value) {
    r0 = c.q32[0]; r1 = c.q32[1]; p1 = c.q32[2]; s1 = c.q32[3]; ap = c.q32[4]; as = c.q32[5];
  } else {
    r0 = c.r0; r1 = c.r1; p1 = c.p1; s1 = c.s1; ap = c.ap; as = c.as;
  }
  float *xl = std::is_same<T, float>::value ? c.q32[6] : nullptr;
  KrylovScalars *ks = c.ks32;
  double *P1 = red_part_host(c, RS_SPMV_DOT), *P2 = red_part_host(c, RS_SPMV_DOT2), *P3 = red_part_host(c, RS_XR),
         *P4 = red_part_host(c, RS_NORM);
  c.solves32++;
  ks_setup_kernel<<<1, 1, 0, c.stream>>>(ks, tol, 1e-7 * tol, maxit, c.solves32);
  set_delta_kernel<<<1, 1, 0, c.stream>>>(ks, delta);
  mr_init_kernel<T><<<nb, 256, op_lds_bytes(a64), c.stream>>>(a64, b, x, r1, r0, p1, (T *)xl,
                                                               red_part_host(c, RS_INIT));
  mr_init_finalize<<<1, FIN_THREADS, 0, c.stream>>>(red_part_host(c, RS_INIT), nb, ks);
  CFD_HIP(hipGetLastError());
  int batch = 4;
  double prev_rel = -1.0;
  int prev_it = 0;
  for (;;) {
    for (int it = 0; it < batch; ++it) {
      spmv_dot_kernel<T><<<nb, 256, op_lds_bytes(ain), c.stream>>>(ain, ks, p1, ap, r0, P1);
      mr_alpha_finalize<<<1, FIN_THREADS, 0, c.stream>>>(P1, nb, ks);
      mr_s_update_kernel<T><<<nb, 256, 0, c.stream>>>(N, ks, r1, ap, s1);
      mr_spmv_dot2_kernel<T><<<nb, 256, 0, c.stream>>>(ain, ks, s1, as, P2);
      mr_omega_finalize<<<1, FIN_THREADS, 0, c.stream>>>(P2, nb, ks);
      if constexpr (std::is_same<T, float>::value)
        mr_xr_update_kernel<T, float><<<nb, 256, 0, c.stream>>>(N, ks, xl, p1, s1, as, r1, r0, P3);
      else
        mr_xr_update_kernel<T, double><<<nb, 256, 0, c.stream>>>(N, ks, x, p1, s1, as, r1, r0, P3);
      mr_conv_finalize<<<1, FIN_THREADS, 0, c.stream>>>(P3, nb, ks);
      if constexpr (std::is_same<T, float>::value) mr_fold_kernel<<<nb, 256, 0, c.stream>>>(N, ks, x, xl);
      mr_replace_kernel<T><<<nb, 256, op_lds_bytes(a64), c.stream>>>(a64, ks, b, x, r1, r0, P4);
      mr_replace_finalize<<<1, FIN_THREADS, 0, c.stream>>>(P4, nb, ks);
      mr_p_update_kernel<T><<<nb, 256, 0, c.stream>>>(N, ks, r1, p1, ap, r0);
    }
    CFD_HIP(hipGetLastError());
    CFD_HIP(hipMemcpyAsync(c.hks, ks, sizeof(KrylovScalars), hipMemcpyDeviceToHost, c.stream));
    CFD_HIP(hipStreamSynchronize(c.stream));
    const KrylovScalars h = *c.hks;
    if (c.debug)
      fprintf(stderr, "[mixed] it %d rep %d brk %d restarts %d rn/nb %.3e true %.3e alpha %.3e omega %.3e rho %.3e\n",
              h.iters, h.replacements, h.breakdown, h.restarts, h.rnorm / h.norm0, h.relres, h.alpha, h.omega, h.rho);
    if (h.done) break;
    const double cur = h.rnorm / h.norm0;
    int next = batch * 2;
    if (prev_rel > 0.0 && cur > 0.0 && cur < prev_rel && h.iters > prev_it) {
      const double rate = std::log(cur / prev_rel) / (double)(h.iters - prev_it);
      const double need = std::log(tol / cur) / rate;
      if (need > 0.0 && std::isfinite(need)) next = (int)std::ceil(need * 1.05) + 1;
    }
    prev_rel = cur;
    prev_it = h.iters;
    batch = std::max(1, std::min(next, 64));
  }
  const KrylovScalars h = *c.hks;
  *replacements = h.replacements;
  *iters = h.iters + 1;
  *relres = h.relres;
  return CFD_OK;
}

}  // namespace

int mixed_reliable_solve(Ctx &c, const double *b, double *x, double tol, double delta, int maxit, int *replacements,
                         int *iters, double *relres) {
  if (c.prm.mixed_mode == CFD_MIXED_VALUES32)
    return reliable_solve<double>(c, b, x, tol, delta, maxit, replacements, iters, relres);
  return reliable_solve<float>(c, b, x, tol, delta, maxit, replacements, iters, relres);
}

}  // namespace cfd

// ---------------------------------------------------------------------------
// cfd_bicgstab_ell_noalloc: the BiCGSTAB solve of cfd_bicgstab on a
// caller-owned ELL operator and caller-owned vectors, with every buffer the
// solve needs beyond them taken from one static device array.  It calls no
// hipMalloc / hipFree and no allocating library routine, so it can run where
// allocation is not allowed (code under stream capture, tight serving loops).
//
// The array holds, per device, the solver's seven work vectors (r0, r1, p1,
// s1, ap, as and px1, the start value kept for the NaN reset) of at most
// CFD_NOALLOC_MAX_ROWS rows, the reduction partials and results, and the
// device scalars.  The host refers to it only through the device address
// hipGetSymbolAddress returns (taken once per device, with that device
// current); the array's own name is a host-side stand-in, not an address.
// Every call on a device shares that device's array and leaves its contents
// behind: calls that overlap on one device race.  Nothing in it needs to
// start at zero: each solve writes every vector and partial before it reads
// it and sets the scalars itself.
// ---------------------------------------------------------------------------
namespace cfd {
namespace {

constexpr int64_t NOALLOC_ROWS = CFD_NOALLOC_MAX_ROWS;
constexpr int NOALLOC_VECS = 7;  // r0 r1 p1 s1 ap as px1
constexpr int64_t NOALLOC_PARTIALS = (int64_t)RED_SITES * 3 * RED_MAX_BLOCKS;
constexpr int64_t NOALLOC_OUT = (int64_t)RED_SITES * 4;
constexpr int64_t NOALLOC_KS = (2 * sizeof(KrylovScalars) + 255) / 256 * 32;  // doubles, 256-byte multiple
constexpr int64_t NOALLOC_DOUBLES = NOALLOC_VECS * NOALLOC_ROWS + NOALLOC_PARTIALS + NOALLOC_OUT + NOALLOC_KS;
static_assert(NOALLOC_PARTIALS % 32 == 0 && NOALLOC_OUT % 32 == 0, "256-byte sections");

static __device__ __align__(256) double scratch[NOALLOC_DOUBLES];

constexpr int NOALLOC_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
double *g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};

// the device address of this device's `scratch`, looked up on the first call
int scratch_address(int dev, double **out) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return fail(CFD_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch_ptr[dev] = static_cast<double *>(ptr);
  }
  *out = g_scratch_ptr[dev];
  return CFD_OK;
}

}  // namespace
}  // namespace cfd

extern "C" int cfd_bicgstab_ell_noalloc(const int32_t *col, const double *val, const double *b, double *x,
                                        size_t n_rows, double tol, int maxit, void *stream, int *iters,
                                        double *relres) {
  using namespace cfd;
  if (!col || !val || !b || !x || !iters || !relres) return fail(CFD_ERR_ARG, "cfd_bicgstab_ell_noalloc: NULL argument");
  if (n_rows < 1) return fail(CFD_ERR_ARG, "cfd_bicgstab_ell_noalloc: n_rows must be >= 1");
  if ((int64_t)n_rows > NOALLOC_ROWS)
    return fail(CFD_ERR_ARG, "cfd_bicgstab_ell_noalloc: n_rows " + std::to_string(n_rows) + " exceeds the maximum " +
                                 std::to_string(NOALLOC_ROWS) + " (CFD_NOALLOC_MAX_ROWS)");
  if (maxit < 0 || !(tol >= 0.0)) return fail(CFD_ERR_ARG, "cfd_bicgstab_ell_noalloc: bad tol / maxit");
  int dev = 0;
  CFD_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) return fail(CFD_ERR_ARG, "cfd_bicgstab_ell_noalloc: device index too large");
  double *base = nullptr;
  if (int rc = scratch_address(dev, &base)) return rc;
  const int64_t N = (int64_t)n_rows;
  // a context on the stack that borrows the caller's operator and the
  // scratch sections; its host mirrors are stack variables (pageable)
  Ctx c;
  c.device = dev;
  c.stream = static_cast<hipStream_t>(stream);
  c.g.N = N;
  c.g.nxc = (int)N;
  c.g.nyc = c.g.nzc = 1;
  c.ell_sliced = 0;  // the caller's arrays are in the reference's slot-major layout
  c.col = const_cast<int32_t *>(col);
  c.val = const_cast<double *>(val);
  c.ell_ready = true;
  double *vec[NOALLOC_VECS];
  for (int q = 0; q < NOALLOC_VECS; ++q) vec[q] = base + (int64_t)q * NOALLOC_ROWS;
  double *tail = base + (int64_t)NOALLOC_VECS * NOALLOC_ROWS;
  c.red.partials = tail;
  c.red.out = tail + NOALLOC_PARTIALS;
  c.red.counters = nullptr;
  c.ks = reinterpret_cast<KrylovScalars *>(tail + NOALLOC_PARTIALS + NOALLOC_OUT);
  KrylovScalars hks{};
  double hred[64] = {};
  c.hks = &hks;
  c.hred = hred;
  // a fresh bicgstabRe2's first solve: timestep_ 1 (no restart rule), px2 zero
  Vecs<double> v{x, vec[0], vec[1], vec[2], vec[3], vec[4], vec[5], b, vec[6], nullptr};
  const int rc = solve_bicg<double>(c, op_args(c, CFD_OP_ELL), v, c.ks, 1, tol, maxit, iters, relres);
  c.stream = nullptr;  // borrowed: the stack context must not release anything
  return rc;
}
