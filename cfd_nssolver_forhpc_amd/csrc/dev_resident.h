// dev_resident.h -- BiCGSTAB iterations of a small ELL system in one launch.
//
// Below half a million rows an iteration of the launch path (launch_iters)
// is eight dependent kernels whose work takes a microsecond or two each: at
// 4096 and at 32768 rows it costs 35 us whatever the size, launch to drain.
// Here the whole solve is one kernel.  Every thread owns RES_ROWS rows and
// keeps their matrix entries and their entries of x, r, r0, p, A p, s and
// A s in registers; a workgroup keeps the entries of the gathered vector it
// needs (its own rows' and its halo's) in LDS.  What crosses workgroups per
// iteration is two halos (p and s) and three sums.
//
// Values cross workgroups as self-validating words (dev_exchange.h).
//
// The sums are those of the launch path bit for bit.  Its x / r update gives
// a thread the rows v, v + S, v + 2S, v + 3S (S: the threads of its grid, a
// multiple of 256); the rows are owned the same way here, so the partial
// sums run over the same rows in the same order.  Its SpMV-dots sum 512
// consecutive rows, the eight waves of a block in turn; a wave of this kernel
// holds the same 64 consecutive rows per slab, and resident_total adds the
// waves, the blocks and the finalize kernel's tree in that order.
//
// What bounds it is the latency of the five exchanges, about 2 us each, and,
// past 10^5 rows, the halo words.  Measured on one MI355X, us an iteration,
// launch path -> here: 512 rows 26.4 -> 4.7 (one workgroup: sums through
// LDS), 4096 33.0 -> 10.9, 32768 33.3 -> 11.8, 65536 34.4 -> 14.4, 303750
// 47.7 -> 22.4, 524288 53.1 -> 19.5.
#pragma once

#include "dev_common.h"
#include "dev_exchange.h"
#include "dev_spmv.h"

namespace cfd {

constexpr int RES_THREADS = 512;
constexpr int RES_ROWS = 4;             // rows a thread (the launch path's x / r update)
constexpr int RES_OWN = RES_THREADS * RES_ROWS;
constexpr int RES_MAX_BLOCKS = 256;     // one workgroup a CU, all resident
constexpr int64_t RES_MAX_N = (int64_t)RES_OWN * RES_MAX_BLOCKS;
// halo entries a workgroup holds: a slab of 512 consecutive rows of a 7-point
// stencil has 2 (1 + nz + 512) outside it at most for nz <= 512
constexpr int RES_HALO = 8256;
constexpr int RES_FETCH = 6;            // halo entries a thread has in flight
constexpr int RES_SLOTS = 1024;         // partial sums of the launch path at most (one per finalize thread)
static_assert(RES_MAX_N / 512 <= RES_SLOTS, "one slot a finalize thread");
static_assert(RES_OWN + RES_HALO < 65536, "16-bit LDS positions");
// words of one exchanged sum: 5 entries a slot (resident_put), two words each
constexpr int RES_RED_WORDS = RES_SLOTS * 5 * 2;

struct ResArgs {
  int64_t N, S;               // rows; rows between a thread's rows (256 nbx)
  int nbx, nblk;              // blocks of the launch path's x / r update, workgroups here
  int sliced;
  const int32_t *col;
  const double *val;
  double *x, *r0, *r1, *p1;
  uint64_t *ll0, *ll1;        // exchanged p and s: the two words of each row
  uint64_t *red[3];           // exchanged sums: 2 x RES_RED_WORDS words each
  KrylovScalars *ks;          // pad0: arrivals, pad1: RES_* state
  int chunk;                  // iterations this launch runs at most
};

struct ResLds {
  double vec[RES_OWN + RES_HALO];          // the gathered vector: own rows (m 512 + t), halo
  int32_t hcol[RES_HALO];                  // global column of a halo entry
  double wsum[2][RES_ROWS][RES_THREADS / 64];
  double fin[2][FIN_THREADS / 64];
  double one[2][4][2];                     // block sums of a lone workgroup (at most 4 slots)
  int nhalo, state, stuck;
};

// The workgroup's halo of the vector exchanged in ll, into its LDS entries.
__device__ inline void resident_halo(ResLds &L, const ResArgs &a, unsigned epoch) {
  const int nh = L.nhalo;
  for (int e0 = (int)threadIdx.x; e0 < nh; e0 += RES_THREADS * RES_FETCH) {
    const bool ok = ll_fetch<RES_FETCH>(
        a.ll0, a.ll1, epoch,
        [&](int u) { return e0 + u * RES_THREADS < nh ? (unsigned)L.hcol[e0 + u * RES_THREADS] : RES_NONE; },
        [&](int u, bool have, double v) {
          if (have) L.vec[RES_OWN + e0 + u * RES_THREADS] = v;
        });
    if (!ok) L.stuck = 1;
  }
}

// Where a workgroup leaves a slot's sum (e = 0) or the sum of its first half
// (e = 1): the exchange buffer, or, when it is the only one (N <= 2048), an
// LDS array.
__device__ inline void resident_put(const ResArgs &a, ResLds &L, uint64_t *red, int q, int slot, int e, double v,
                                    unsigned epoch) {
  if (a.nblk == 1) {
    L.one[q][slot][e] = v;
  } else {
    uint64_t *dst = red + (size_t)q * RES_RED_WORDS + (size_t)slot * 4 + 2 * e;
    ll_store(dst, dst + 1, v, epoch);
  }
}

// Block sums of the launch path's SpMV-dots, from this workgroup's wave sums
// L.wsum[q][m][wave]: slot b adds the 64-row waves 8b .. 8b + 7 in turn.  A
// slab's half of 256 rows is quad Q = 2 blk + h + m nbx, half Q & 1 of slot
// Q / 2.  Where a slab is a whole slot (nbx even, or m even short of the
// grid's end) one thread adds its eight waves.  Else the first half's sum
// goes to the workgroup that holds the second, which adds its four waves to
// it: one more hop, in every second slab of an odd nbx.  (Leaving the five
// parts for every reader to add instead took 58 us an iteration at 303750
// rows against 30: each workgroup reads every slot.)
template <int NV>
__device__ inline void resident_put_rows(const ResArgs &a, ResLds &L, uint64_t *red, unsigned epoch) {
  const int t = threadIdx.x;
  if (t >= NV * RES_ROWS * 2) return;
  const int q = t / (RES_ROWS * 2), m = (t >> 1) % RES_ROWS, h = t & 1;
  const int blk = blockIdx.x, Q = 2 * blk + h + m * a.nbx, slot = Q >> 1;
  if (2 * blk + h >= a.nbx) return;  // the empty half of the last workgroup of an odd nbx
  const double *ws = L.wsum[q][m] + 4 * h;
  const bool whole = (Q & 1) ? h == 1 : h == 0 && 2 * blk + 1 < a.nbx;  // the slot's other half is this slab's
  if (whole && h == 0) {
    double s = ws[0];
#pragma unroll
    for (int w = 1; w < 8; ++w) s += ws[w];
    resident_put(a, L, red, q, slot, 0, s, epoch);
  }
  if (!whole && (Q & 1) == 0)
    resident_put(a, L, red, q, slot, 1, ((ws[0] + ws[1]) + ws[2]) + ws[3], epoch);
  // The lanes that wait for another workgroup's first half come after the
  // lanes that leave one, in program order: they share a wave, and every
  // workgroup of the ring must have left its half before it waits.
  asm volatile("" ::: "memory");
  if (!whole && (Q & 1)) {
    double s = 0.0;
    if (a.nblk == 1) {
      // a lone workgroup holds both halves: the first is quad Q - 1, whose
      // four waves it adds itself
      const int Qf = Q - 1, mf = Qf / a.nbx, hf = Qf % a.nbx;
      const double *wf = L.wsum[q][mf] + 4 * hf;
      s = ((wf[0] + wf[1]) + wf[2]) + wf[3];
    } else if (!ll_fetch<1>(
                   red, red + 1, epoch, [&](int) { return (unsigned)(q * RES_RED_WORDS + slot * 4 + 2); },
                   [&](int, bool, double x) { s = x; })) {
      L.stuck = 1;
    }
    resident_put(a, L, red, q, slot, 0, (((s + ws[0]) + ws[1]) + ws[2]) + ws[3], epoch);
  }
}

// Block sums of the launch path's x / r update: slot b is one half of a
// workgroup's threads (256), its four waves in turn.  L.wsum[q][0][wave].
__device__ inline void resident_put_xr(const ResArgs &a, ResLds &L, uint64_t *red, unsigned epoch) {
  const int t = threadIdx.x;
  if (t < 4) {
    const int q = t >> 1, h = t & 1, slot = 2 * (int)blockIdx.x + h;
    if (slot < a.nbx) {
      const double *ws = L.wsum[q][0] + 4 * h;
      resident_put(a, L, red, q, slot, 0, ((ws[0] + ws[1]) + ws[2]) + ws[3], epoch);
    }
  }
}

// The totals of nslot slots in combine_partials' order: slot t belongs to
// finalize thread t, whose 64 lanes are summed by wave_sum and whose 16 waves
// in turn.
template <int NV>
__device__ inline void resident_total(const ResArgs &a, ResLds &L, const uint64_t *red, int nslot, unsigned epoch,
                                      double (&tot)[NV]) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __syncthreads();  // this workgroup's sums are left (L.one, or issued: RES_SPIN)
  if (a.nblk == 1) {
    if (wid < NV) {  // at most 4 slots: the first finalize wave's lanes
      double v = 0.0;
      if (lane < nslot) v = L.one[wid][lane][0];
      v = wave_sum(0.0 + v);
      if (lane == 0) L.fin[wid][0] = v;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NV; ++q) tot[q] = L.fin[q][0] + 0.0;  // the other 15 waves' sums are zero
    return;
  }
#pragma unroll 1
  for (int half = 0; half < FIN_THREADS / RES_THREADS; ++half) {
    double v[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) v[q] = 0.0;
    if (half * RES_THREADS < nslot) {  // uniform
      const int slot = (int)threadIdx.x + half * RES_THREADS;
      const bool mine = slot < nslot;
      const bool ok = ll_fetch<NV>(
          red, red + 1, epoch, [&](int q) { return mine ? (unsigned)(q * RES_RED_WORDS + slot * 4) : RES_NONE; },
          [&](int q, bool have, double x) { v[q] = have ? x : 0.0; });
      if (!ok) L.stuck = 1;
#pragma unroll
      for (int q = 0; q < NV; ++q) v[q] = wave_sum(0.0 + v[q]);  // combine_partials adds the slot to a zero
    }
    if (lane == 0) {
#pragma unroll
      for (int q = 0; q < NV; ++q) L.fin[q][wid + half * (RES_THREADS / 64)] = v[q];
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    double s = L.fin[q][0];
#pragma unroll
    for (int w = 1; w < FIN_THREADS / 64; ++w) s += L.fin[q][w];
    tot[q] = s;
  }
}

// y = A (the vector in L.vec) on the thread's rows: ell_row's FMA chain.
// pos holds two 16-bit positions a register; the empty asm keeps their
// unpacked forms from being hoisted out of the iteration (28 registers).
constexpr int RES_POS = (KSLOTS + 1) / 2;
__device__ inline void resident_rows(const ResLds &L, const double (&val)[RES_ROWS][KSLOTS],
                                     unsigned (&pos)[RES_ROWS][RES_POS], double (&y)[RES_ROWS]) {
#pragma unroll
  for (int m = 0; m < RES_ROWS; ++m) {
    double xv[KSLOTS];
#pragma unroll
    for (int s = 0; s < KSLOTS; ++s) {
      if ((s & 1) == 0) asm volatile("" : "+v"(pos[m][s >> 1]));
      xv[s] = L.vec[(s & 1) ? pos[m][s >> 1] >> 16 : pos[m][s >> 1] & 0xffffu];
    }
    double acc = 0.0;
#pragma unroll
    for (int s = 0; s < KSLOTS; ++s) acc = fma(val[m][s], xv[s], acc);
    y[m] = acc;
  }
}

// Iterations from the state init_kernel left (x, r0, r1, p1, ks) until the
// stop test, the iteration cap or a.chunk iterations.  Same arithmetic as
// launch_iters<double>'s kernels, expression for expression.  x and r0, which
// nothing gathers, stay in memory (each thread its own rows; the register
// file holds the rest).
__global__ void __launch_bounds__(RES_THREADS) bicg_resident_kernel(ResArgs a) {
  __shared__ ResLds L;
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  const unsigned N = (unsigned)a.N, S = (unsigned)a.S;
  const unsigned v = blockIdx.x * RES_THREADS + t;
  const unsigned vend = v < S ? N : 0;  // the last workgroup of an odd nbx is half empty
  auto own = [&](int m) { return v + m * S < vend; };
  if (a.ks->done) return;  // uniform over the grid: written by an earlier kernel
  double rho = a.ks->rho;
  const double norm0 = a.ks->norm0;
  const double tol = a.ks->tol, restart_tol = a.ks->restart_tol;
  const int maxit = a.ks->maxit, timestep = a.ks->timestep;
  int iters = a.ks->iters, restarts = a.ks->restarts;
  if (t == 0) {
    L.nhalo = a.nblk > 1 ? 1 : 0;  // entry 0: column N - 1, where every padding slot points
    L.hcol[0] = (int32_t)(N - 1);
    L.stuck = 0;
  }
  __syncthreads();
  double val[RES_ROWS][KSLOTS];
  unsigned pos[RES_ROWS][RES_POS];
  double r[RES_ROWS], p[RES_ROWS], ap[RES_ROWS], s[RES_ROWS], as[RES_ROWS];
  int fits = 1;
  const int64_t st = ell_stride(a.N, a.sliced);
#pragma unroll
  for (int m = 0; m < RES_ROWS; ++m) {
    const unsigned row = own(m) ? v + m * S : 0;
    const int64_t b = ell_base(row, a.sliced);
#pragma unroll
    for (int sl = 0; sl < KSLOTS; ++sl) {
      val[m][sl] = own(m) ? a.val[b + sl * st] : 0.0;
      unsigned at = 0;
      if (own(m)) {
        const unsigned c = (unsigned)a.col[b + sl * st];
        // the column's owner: thread c mod S of the grid, its (c / S)-th row
        const unsigned cm = c / S, cv = c - cm * S;
        if (cv / RES_THREADS == blockIdx.x) {
          at = cm * RES_THREADS + cv % RES_THREADS;
        } else if (c == N - 1) {
          at = RES_OWN;
        } else {
          const int e = atomicAdd(&L.nhalo, 1);
          if (e < RES_HALO) {
            L.hcol[e] = (int32_t)c;
            at = RES_OWN + e;
          } else {
            fits = 0;
          }
        }
      }
      if (sl & 1) pos[m][sl >> 1] |= at << 16;
      else pos[m][sl >> 1] = at;
    }
    r[m] = own(m) ? *at32(a.r1, row) : 0.0;
    p[m] = own(m) ? *at32(a.p1, row) : 0.0;
  }
  fits = __syncthreads_and(fits);
  if (resident_arrive(a.ks, a.nblk, &L.state, fits) != RES_GO) return;
  const int nslot = (int)((a.N + 511) / 512);
  double alpha = 0.0, omega = 0.0, beta = 0.0, pre_rho = 0.0, rnorm = 0.0, relres = 0.0;
  int done = 0, hit = 0, restart = 0;
#pragma unroll 1
  for (int it = 0; it < a.chunk && !done; ++it) {
    const unsigned epoch = (unsigned)it + 1u;  // of the sums; the halos of p and s are numbered 2 it + 1 and 2 it + 2
    // ap = A p, ap . r0
    double r0[RES_ROWS];
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m) {
      L.vec[m * RES_THREADS + t] = p[m];
      if (own(m) && a.nblk > 1) ll_store(at32(a.ll0, v + m * S), at32(a.ll1, v + m * S), p[m], 2 * epoch - 1);
      r0[m] = own(m) ? *at32(a.r0, v + m * S) : 0.0;
    }
    __syncthreads();  // every wave has issued its words (RES_SPIN)
    resident_halo(L, a, 2 * epoch - 1);
    __syncthreads();
    resident_rows(L, val, pos, ap);
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m) {
      double acc = 0.0;
      if (own(m)) acc += ap[m] * r0[m];
      acc = wave_sum(acc);
      if (lane == 0) L.wsum[0][m][wid] = acc;
    }
    __syncthreads();
    resident_put_rows<1>(a, L, a.red[0], epoch);
    double ta[1];
    resident_total<1>(a, L, a.red[0], nslot, epoch, ta);
    alpha = rho / ta[0];
    // s = r - alpha ap; as = A s, as . s, as . as
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m) {
      s[m] = r[m] - alpha * ap[m];
      L.vec[m * RES_THREADS + t] = s[m];
      if (own(m) && a.nblk > 1) ll_store(at32(a.ll0, v + m * S), at32(a.ll1, v + m * S), s[m], 2 * epoch);
    }
    __syncthreads();
    resident_halo(L, a, 2 * epoch);
    __syncthreads();
    resident_rows(L, val, pos, as);
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m) {
      double acc0 = 0.0, acc1 = 0.0;
      if (own(m)) {
        acc0 += as[m] * s[m];
        acc1 += as[m] * as[m];
      }
      acc0 = wave_sum(acc0);
      acc1 = wave_sum(acc1);
      if (lane == 0) {
        L.wsum[0][m][wid] = acc0;
        L.wsum[1][m][wid] = acc1;
      }
    }
    __syncthreads();
    resident_put_rows<2>(a, L, a.red[1], epoch);
    double to[2], xo[RES_ROWS];
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m) {
      xo[m] = own(m) ? *at32(a.x, v + m * S) : 0.0;
      r0[m] = own(m) ? *at32(a.r0, v + m * S) : 0.0;
    }
    resident_total<2>(a, L, a.red[1], nslot, epoch, to);
    omega = to[0] / to[1];
    // x += alpha p + omega s; r = s - omega as; r . r, r . r0
    double acc[2] = {0.0, 0.0};
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m) {
      if (own(m)) {
        *at32(a.x, v + m * S) = xo[m] + fma(omega, s[m], alpha * p[m]);  // xr_update_kernel's contraction
        const double rn = s[m] - omega * as[m];
        r[m] = rn;
        acc[0] += rn * rn;
        acc[1] += rn * r0[m];
      }
    }
    acc[0] = wave_sum(acc[0]);
    acc[1] = wave_sum(acc[1]);
    if (lane == 0) {
      L.wsum[0][0][wid] = acc[0];
      L.wsum[1][0][wid] = acc[1];
    }
    __syncthreads();
    resident_put_xr(a, L, a.red[2], epoch);
    double tc[2];
    resident_total<2>(a, L, a.red[2], a.nbx, epoch, tc);
    if (L.stuck) {  // a wait reached its bound
      if (t == 0) __hip_atomic_store(&a.ks->pad1, (int)RES_STUCK, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    // the stop test, beta and the restart rule (conv_finalize)
    rnorm = sqrt(tc[0]);
    relres = rnorm / norm0;
    if (relres < tol) {
      done = 1;
    } else if (iters >= maxit) {
      done = 1;
      hit = 1;
    } else {
      pre_rho = rho;
      rho = tc[1];
      beta = (alpha / omega) * (rho / pre_rho);
      restart = (timestep < 10 || fabs(pre_rho) > restart_tol) ? 0 : 1;
      restarts += restart;
      iters += 1;
      if (restart) {
#pragma unroll
        for (int m = 0; m < RES_ROWS; ++m) {
          p[m] = r[m];
          if (own(m)) *at32(a.r0, v + m * S) = r[m];
        }
      } else {
#pragma unroll
        for (int m = 0; m < RES_ROWS; ++m) p[m] = r[m] + beta * (p[m] - omega * ap[m]);
      }
    }
  }
  if (!done) {  // the next launch goes on from here
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m)
      if (own(m)) {
        *at32(a.r1, v + m * S) = r[m];
        *at32(a.p1, v + m * S) = p[m];
      }
  }
  if (blockIdx.x == 0 && t == 0) {  // everything but pad0 / pad1
    a.ks->alpha = alpha;
    a.ks->omega = omega;
    a.ks->rnorm = rnorm;
    a.ks->relres = relres;
    a.ks->rho = rho;
    a.ks->pre_rho = pre_rho;
    a.ks->beta = beta;
    a.ks->iters = iters;
    a.ks->done = done;
    a.ks->hit_maxit = hit;
    a.ks->restart = restart;
    a.ks->restarts = restarts;
  }
}

// no exchange has taken place: every word's number is 0 before a launch
__global__ void __launch_bounds__(256) resident_clear_kernel(ResArgs a) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < a.N) a.ll0[q] = a.ll1[q] = 0;
  if (q < 2 * RES_RED_WORDS) a.red[0][q] = a.red[1][q] = a.red[2][q] = 0;
  if (q == 0) a.ks->pad0 = a.ks->pad1 = 0;
}

}  // namespace cfd
