// dev_resident.h -- BiCGSTAB iterations of a small ELL system in one launch.
//
// Below half a million rows an iteration of the launch path (launch_iters)
// is five dependent kernels (fold_of) whose work takes a microsecond or two
// each: at 4096 and at 32768 rows it costs 24 us, launch to drain.  Here the
// whole solve is one kernel.  Every thread owns RES_ROWS rows and keeps their
// matrix entries and their entries of r, p, A p, s and A s in registers; a
// workgroup keeps the entries of the gathered vector it needs (its own rows' and
// its halo's) in LDS.  What crosses workgroups per iteration is two halos (p and
// s) and three sums.
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
// past 10^5 rows, the halo words.  Measured on one MI355X over whole solves of
// 2000 iterations, us an iteration, launches -> here: 512 rows 20.0 -> 4.6 (one
// workgroup: sums through LDS), 4096 23.8 -> 9.7, 32768 24.1 -> 10.6, 65536
// 25.1 -> 13.6, 303750 31.8 -> 22.8, 524288 29.9 -> 21.0.  Of the 12 us that 32768 rows took before
// the wave sums were packed, every wave formed the total of up to 128 slots
// itself and the next p left ahead of the stop test: halos 2.8, the sums'
// way 5.5, products with their wave sums 1.9, the rest 1.6.
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
// words of one exchanged sum: two entries a slot (resident_put), two words each
constexpr int RES_SLOT_WORDS = 4;
constexpr int RES_RED_WORDS = RES_SLOTS * RES_SLOT_WORDS;

struct ResArgs {
  int64_t N, S;               // rows; rows between a thread's rows (256 nbx)
  int nbx, nblk;              // blocks of the launch path's x / r update, workgroups here
  int sliced;
  const int32_t *col;
  const double *val;
  double *x, *r0, *r1, *p1;
  uint64_t *ll0, *ll1;        // exchanged p and s: the two words of each row
  uint64_t *red[3];           // exchanged sums: 2 x RES_RED_WORDS words each
  double *keep;               // x as it was before the solve
  KrylovScalars *ks;          // pad0: arrivals, pad1: RES_* state; ks[1].restarts as it was before the solve
  int chunk;                  // iterations this launch runs at most
  ResBounds bounds;
};

struct ResLds {
  double vec[RES_OWN + RES_HALO];          // the gathered vector: own rows (m 512 + t), halo
  int32_t hcol[RES_HALO];                  // global column of a halo entry
  double wsum[2][RES_ROWS][RES_THREADS / 64];
  double fin[2][FIN_THREADS / 64];
  double one[2][4][2];                     // block sums of a lone workgroup (at most 4 slots)
  int nhalo, state;
  alignas(8) int stuck;                    // a wait reached its bound
  int done;                                // the stop test's result, from the first wave
  double norm0, tol, restart_tol;
  int maxit, timestep;
};

// The workgroup's halo of the vector exchanged in ll, into its LDS entries.  An
// iteration has up to six of these waits, each with a share of the bound: to
// look at L.stuck in them as in the others takes 0.3 us of 22.6 at 303750 rows.
constexpr int RES_HALO_SHARE = 32;
template <bool SET>
__device__ inline void resident_halo(ResLds &L, const ResArgs &a, unsigned epoch) {
  const int nh = L.nhalo;
  for (int e0 = (int)threadIdx.x; e0 < nh; e0 += RES_THREADS * RES_FETCH) {
    const bool ok = ll_fetch<RES_FETCH, false>(
        a.ll0, a.ll1, epoch, (res_spin<SET>(a.bounds) + RES_HALO_SHARE - 1) / RES_HALO_SHARE, L.stuck,
        [&](int u) { return e0 + u * RES_THREADS < nh ? (unsigned)L.hcol[e0 + u * RES_THREADS] : RES_NONE; },
        [&](int u, bool have, double v) {
          if (have) L.vec[RES_OWN + e0 + u * RES_THREADS] = v;
        });
    if (!ok) L.stuck = 1;
  }
}

// wave_sum of two and of four values at once.  wave_sum adds neighbouring
// lanes, then neighbouring pairs, quads, .. and every lane of a group holds the
// group's sum; here the copies are given up for other values (lane & 1, lane &
// 3 says whose sum a lane holds), so that the steps are shared.  The sums are
// wave_sum's bit for bit in lanes 62, 63 and 60 .. 63: lanes of the last quad
// of 16, whose order of the quads is the one that wave_sum returns.
__device__ inline double wave_rows(double v) {  // the steps across quads and rows
  v += dpp_move<0x124>(v);                      // row_ror:4
  v += dpp_move<0x128>(v);                      // row_ror:8
  const long long b = __double_as_longlong(v);
  const auto l16 = __builtin_amdgcn_permlane16_swap((unsigned)b, (unsigned)b, false, false);
  const auto h16 = __builtin_amdgcn_permlane16_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
  v = __longlong_as_double((long long)h16[0] << 32 | l16[0]) + __longlong_as_double((long long)h16[1] << 32 | l16[1]);
  const long long d = __double_as_longlong(v);
  const auto l32 = __builtin_amdgcn_permlane32_swap((unsigned)d, (unsigned)d, false, false);
  const auto h32 = __builtin_amdgcn_permlane32_swap((unsigned)(d >> 32), (unsigned)(d >> 32), false, false);
  return __longlong_as_double((long long)h32[0] << 32 | l32[0]) + __longlong_as_double((long long)h32[1] << 32 | l32[1]);
}
__device__ inline double pair_pack(double a, double b) {  // even lanes: a of the pair, odd lanes: b
  const bool odd = threadIdx.x & 1;
  return (odd ? b : a) + dpp_move<0xb1>(odd ? a : b);
}
__device__ inline double wave_sum2(double a, double b) {
  double v = pair_pack(a, b);
  v += dpp_move<0x4e>(v);
  return wave_rows(v);
}
__device__ inline double wave_sum4(double a, double b, double c, double d) {
  const double ab = pair_pack(a, b), cd = pair_pack(c, d);
  const bool hi = threadIdx.x & 2;
  return wave_rows((hi ? cd : ab) + dpp_move<0x4e>(hi ? ab : cd));
}
__device__ inline double lane_value(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Where a workgroup leaves a slot's sum (e = 0) or the sum of its first half
// (e = 1): the exchange buffer, or, when it is the only one (N <= 2048), an
// LDS array.
__device__ inline void resident_put(const ResArgs &a, ResLds &L, uint64_t *red, int q, int slot, int e, double v,
                                    unsigned epoch) {
  if (a.nblk == 1) {
    L.one[q][slot][e] = v;
  } else {
    uint64_t *dst = red + (size_t)q * RES_RED_WORDS + (size_t)slot * RES_SLOT_WORDS + 2 * e;
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
template <int NV, bool SET>
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
                   red, red + 1, epoch, res_spin<SET>(a.bounds), L.stuck,
                   [&](int) { return (unsigned)(q * RES_RED_WORDS + slot * RES_SLOT_WORDS + 2); },
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
template <int NV, bool SET>
__device__ inline void resident_total(const ResArgs &a, ResLds &L, const uint64_t *red, int nslot, unsigned epoch,
                                      double (&tot)[NV]) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __syncthreads();  // this workgroup's sums are left (L.one, or issued: RES_SPIN)
  // Up to two of the finalize kernel's waves (N <= 65536): every wave of the
  // workgroup forms the total itself; the other waves' sums are zero.
  if (nslot <= 128) {
    double v[2][NV] = {};  // a wait that reaches its bound leaves zeros
    if (a.nblk == 1) {
#pragma unroll
      for (int q = 0; q < NV; ++q) {
        v[0][q] = lane < nslot ? L.one[q][lane & 3][0] : 0.0;
        v[1][q] = 0.0;
      }
    } else {
      const bool ok = ll_fetch<2 * NV>(
          red, red + 1, epoch, res_spin<SET>(a.bounds), L.stuck,
          [&](int u) {
            const int q = u % NV, slot = lane + u / NV * 64;
            return slot < nslot ? (unsigned)(q * RES_RED_WORDS + slot * RES_SLOT_WORDS) : RES_NONE;
          },
          [&](int u, bool have, double x) { v[u / NV][u % NV] = have ? x : 0.0; });
      if (!ok) L.stuck = 1;
    }
    // combine_partials adds the slot to a zero
    if constexpr (NV == 1) {
      const double w = wave_sum2(0.0 + v[0][0], 0.0 + v[1][0]);
      tot[0] = (lane_value(w, 62) + lane_value(w, 63)) + 0.0;
    } else {
      const double w = wave_sum4(0.0 + v[0][0], 0.0 + v[0][1], 0.0 + v[1][0], 0.0 + v[1][1]);
      tot[0] = (lane_value(w, 60) + lane_value(w, 62)) + 0.0;
      tot[1] = (lane_value(w, 61) + lane_value(w, 63)) + 0.0;
    }
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
          red, red + 1, epoch, res_spin<SET>(a.bounds), L.stuck,
          [&](int q) { return mine ? (unsigned)(q * RES_RED_WORDS + slot * RES_SLOT_WORDS) : RES_NONE; },
          [&](int q, bool have, double x) { v[q] = have ? x : 0.0; });
      if (!ok) L.stuck = 1;
      // combine_partials adds the slot to a zero
      if constexpr (NV == 1)
        v[0] = wave_sum(0.0 + v[0]);
      else
        v[0] = wave_sum2(0.0 + v[0], 0.0 + v[1]);
    }
    if (NV == 1 && lane == 0) L.fin[0][wid + half * (RES_THREADS / 64)] = v[0];
    if (NV == 2 && lane >= 62) L.fin[lane - 62][wid + half * (RES_THREADS / 64)] = v[0];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    double s = L.fin[q][0];
#pragma unroll 1
    for (int w = 0; w < FIN_THREADS / 64; w += 8) {  // eight in flight: the register file is full
      double f[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) f[u] = L.fin[q][w + u];
#pragma unroll
      for (int u = 0; u < 8; ++u) s = w + u ? s + f[u] : s;
    }
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
template <bool SET>
__global__ void __launch_bounds__(RES_THREADS) bicg_resident_kernel(ResArgs a) {
  __shared__ ResLds L;
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  const unsigned N = (unsigned)a.N, S = (unsigned)a.S;
  const unsigned v = blockIdx.x * RES_THREADS + t;
  const unsigned vend = v < S ? N : 0;  // the last workgroup of an odd nbx is half empty
  auto own = [&](int m) { return v + m * S < vend; };
  if (a.ks->done) return;  // uniform over the grid: written by an earlier kernel
  double rho = a.ks->rho;
  int iters = a.ks->iters, restarts = a.ks->restarts;
  if (t == 0) {
    L.nhalo = a.nblk > 1 ? 1 : 0;  // entry 0: column N - 1, where every padding slot points
    L.hcol[0] = (int32_t)(N - 1);
    L.stuck = L.done = 0;
    L.norm0 = a.ks->norm0;
    L.tol = a.ks->tol;
    L.restart_tol = a.ks->restart_tol;
    L.maxit = a.ks->maxit;
    L.timestep = a.ks->timestep;
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
  if (resident_arrive(a.ks, a.nblk, &L.state, fits, a.bounds.arrive) != RES_GO) return;
  const int nslot = (int)((a.N + 511) / 512);
  double alpha = 0.0, omega = 0.0, beta = 0.0, pre_rho = 0.0, rnorm = 0.0, relres = 0.0;
  int done = 0, hit = 0, restart = 0;
  auto publish_p = [&](unsigned epoch) {
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m) {
      L.vec[m * RES_THREADS + t] = p[m];
      if (own(m) && a.nblk > 1) ll_store(at32(a.ll0, v + m * S), at32(a.ll1, v + m * S), p[m], epoch);
    }
  };
  publish_p(1);
#pragma unroll 1
  for (int it = 0; it < a.chunk; ++it) {
    const unsigned epoch = (unsigned)it + 1u;  // of the sums; the halos of p and s are numbered 2 it + 1 and 2 it + 2
    // ap = A p, ap . r0
    double r0[RES_ROWS];
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m) r0[m] = own(m) ? *at32(a.r0, v + m * S) : 0.0;
    __syncthreads();  // every wave has issued its words (RES_SPIN)
    resident_halo<SET>(L, a, 2 * epoch - 1);
    __syncthreads();
    // Every wave leaves here or none: both flags are set before this barrier or
    // after the next, and waves whose waits failed have totals of their own, so
    // a wave's own `done` must not end its loop.  (The halo just fetched is of
    // the p that is published before the stop test.)
    if (L.stuck | L.done) break;
    resident_rows(L, val, pos, ap);
    double acc1[RES_ROWS], acc2[RES_ROWS];
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m) acc1[m] = own(m) ? fma(ap[m], r0[m], 0.0) : 0.0;
    const double w1 = wave_sum4(acc1[0], acc1[1], acc1[2], acc1[3]);
    if (lane >= 60) L.wsum[0][lane - 60][wid] = w1;
    __syncthreads();
    resident_put_rows<1, SET>(a, L, a.red[0], epoch);
    double ta[1];
    resident_total<1, SET>(a, L, a.red[0], nslot, epoch, ta);
    alpha = rho / ta[0];
    // s = r - alpha ap; as = A s, as . s, as . as
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m) {
      s[m] = r[m] - alpha * ap[m];
      L.vec[m * RES_THREADS + t] = s[m];
      if (own(m) && a.nblk > 1) ll_store(at32(a.ll0, v + m * S), at32(a.ll1, v + m * S), s[m], 2 * epoch);
    }
    __syncthreads();
    resident_halo<SET>(L, a, 2 * epoch);
    __syncthreads();
    resident_rows(L, val, pos, as);
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m) {
      acc1[m] = own(m) ? fma(as[m], s[m], 0.0) : 0.0;
      acc2[m] = own(m) ? fma(as[m], as[m], 0.0) : 0.0;
    }
    const double w2 = wave_sum4(acc1[0], acc1[1], acc1[2], acc1[3]);
    const double w3 = wave_sum4(acc2[0], acc2[1], acc2[2], acc2[3]);
    if (lane >= 60) {
      L.wsum[0][lane - 60][wid] = w2;
      L.wsum[1][lane - 60][wid] = w3;
    }
    __syncthreads();
    resident_put_rows<2, SET>(a, L, a.red[1], epoch);
    double to[2], xo[RES_ROWS];
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m) {
      xo[m] = own(m) ? *at32(a.x, v + m * S) : 0.0;
      r0[m] = own(m) ? *at32(a.r0, v + m * S) : 0.0;
    }
    resident_total<2, SET>(a, L, a.red[1], nslot, epoch, to);
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
    const double wx = wave_sum2(acc[0], acc[1]);
    if (lane >= 62) L.wsum[lane - 62][0][wid] = wx;
    __syncthreads();
    resident_put_xr(a, L, a.red[2], epoch);
    const double ao = alpha / omega;
    double tc[2];
    resident_total<2, SET>(a, L, a.red[2], a.nbx, epoch, tc);
    // beta, the restart rule and the next p (conv_finalize, p_update_kernel),
    // on its way before the stop test: nothing reads it after the last iteration
    const double next_beta = ao * (tc[1] / rho);
    const int next_restart = (L.timestep < 10 || fabs(rho) > L.restart_tol) ? 0 : 1;
#pragma unroll
    for (int m = 0; m < RES_ROWS; ++m) p[m] = next_restart ? r[m] : r[m] + next_beta * (p[m] - omega * ap[m]);
    publish_p(2 * epoch + 1);
    rnorm = sqrt(tc[0]);
    relres = rnorm / L.norm0;
    if (relres < L.tol) {
      done = 1;
    } else if (iters >= L.maxit) {
      done = 1;
      hit = 1;
    } else {
      pre_rho = rho;
      rho = tc[1];
      beta = next_beta;
      restart = next_restart;
      restarts += restart;
      iters += 1;
      if (restart) {
#pragma unroll
        for (int m = 0; m < RES_ROWS; ++m)
          if (own(m)) *at32(a.r0, v + m * S) = r[m];
      }
    }
    if (t == 0) L.done = done;
  }
  __syncthreads();
  if (L.stuck) {
    if (t == 0) __hip_atomic_store(&a.ks->pad1, (int)RES_STUCK, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
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

// no exchange has taken place: every word's number is 0 before a launch; the
// first one of a solve keeps what the solve changes and init_kernel does not set
__global__ void __launch_bounds__(256) resident_clear_kernel(ResArgs a, bool first) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (first && q < a.N) a.keep[q] = a.x[q];
  if (first && q == 0) a.ks[1].restarts = a.ks->restarts;
  if (q < a.N) a.ll0[q] = a.ll1[q] = 0;
  if (q < 2 * RES_RED_WORDS) a.red[0][q] = a.red[1][q] = a.red[2][q] = 0;
  if (q == 0) a.ks->pad0 = a.ks->pad1 = 0;
}

__global__ void __launch_bounds__(256) resident_restore_kernel(ResArgs a) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < a.N) a.x[q] = a.keep[q];
  if (q == 0) a.ks->restarts = a.ks[1].restarts;
}

}  // namespace cfd
