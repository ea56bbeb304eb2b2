// dev_exchange.h -- values exchanged between the workgroups of one launch.
//
// Values cross workgroups as self-validating words: a double travels as two
// 64-bit words, each half the value and the 32-bit number of the exchange
// (ll_store / ll_load).  Each word is one relaxed agent-scope atomic, so a
// reader that finds the number it waits for has the value, with no fence and
// no flag to read first; an exchange costs one store and one load to the
// level the XCDs share.  A buffer is rewritten only when its readers are known
// to be through: in the BiCGSTAB after a sum that every workgroup contributed to
// after its reads; in SorPipeLine, whose sweeps end in no sum that is waited for,
// a colour's values after the neighbours' next ones of the other colour, which
// they leave after their reads, and a maximum after every workgroup's next one.
#pragma once

#include <atomic>

#include "dev_common.h"

namespace cfd {

enum { RES_PENDING = 0, RES_GO = 1, RES_ABORT = 2, RES_STUCK = 3 };

// Element q of an array of 8-byte elements by its 32-bit byte offset (the
// arrays are at most 4 MB), so that an access is a scalar base and one
// 32-bit register instead of a 64-bit address held per array and row.
template <typename T>
__device__ inline T *at32(T *p, unsigned q) {
  static_assert(sizeof(T) == 8, "8-byte elements");
  return reinterpret_cast<T *>(reinterpret_cast<char *>(p) + (q << 3));
}
template <typename T>
__device__ inline const T *at32(const T *p, unsigned q) {
  return reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + (q << 3));
}

__device__ inline uint64_t ll_get(const uint64_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline void ll_store(uint64_t *p0, uint64_t *p1, double v, unsigned epoch) {
  const uint64_t b = (uint64_t)__double_as_longlong(v), e = (uint64_t)epoch << 32;
  __hip_atomic_store(p0, e | (b & 0xffffffffu), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(p1, e | (b >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline double ll_value(uint64_t w0, uint64_t w1) {
  return __longlong_as_double((long long)((w0 & 0xffffffffu) | (w1 << 32)));
}

// Once every workgroup is known to be resident, each wait ends when the
// others reach the same point, microseconds later.  No wave polls before
// every wave of its workgroup has issued the words others wait for (a barrier
// stands between): the memory pipeline takes older waves first, and waves
// that poll scattered words keep it full, so a younger wave's stores could
// wait for ever behind polls that wait for them.  The bound (a second of
// polling, counted in polls so that a preempted kernel does not run into it)
// holds for a workgroup, not for each of its waits: once one has run out, the
// others end RES_LOOK polls later (the resident BiCGSTAB's halos: a small part of
// the bound).  It is there so that the kernel ends whatever
// happens, with RES_STUCK: the host then takes the solve back to its start
// (every such solve keeps a copy of what it writes to) and runs it by launches.
constexpr unsigned RES_SPIN = 1u << 22, RES_LOOK = 1u << 10;
// polls of the arrival handshake before a workgroup gives the launch up (the CUs
// are held by other kernels): a millisecond, which is what the launches take for
// such a solve; workgroups that find their CUs arrive within some 20 us
constexpr unsigned RES_ARRIVE_SPIN = 1u << 12;

// the bounds of a launch: the arrival's, the first workgroup's and the others'
struct ResBounds {
  unsigned arrive, first, others;
  bool set;  // first or others is not RES_SPIN
};
inline ResBounds res_bounds(const OneLaunch &o) {
  ResBounds b;
  b.arrive = o.arrive > 0 ? (unsigned)o.arrive : RES_ARRIVE_SPIN;
  b.others = o.wait > 0 ? (unsigned)o.wait : RES_SPIN;
  b.first = o.wait_first > 0 ? (unsigned)o.wait_first : b.others;
  b.set = o.wait > 0 || o.wait_first > 0;
  return b;
}
// SET: as given (kept in registers for the whole solve, the given ones cost
// 0.2 us of 9.8 an iteration at 4096 rows), else RES_SPIN
template <bool SET>
__device__ inline unsigned res_spin(const ResBounds &b) {
  return !SET ? RES_SPIN : blockIdx.x ? b.others : b.first;
}

// Loads U pairs of words at a time until each carries the epoch: get(u) is
// the position of the u-th pair in w0 / w1 (RES_NONE: none), put(u, v) takes
// its value.  False when the bound was reached, here or (LOOK; stuck, in LDS, set
// by the callers) in another of the workgroup's waits.
constexpr unsigned RES_NONE = ~0u;
template <int U, bool LOOK = true, typename G, typename P>
__device__ inline bool ll_fetch(const uint64_t *p0, const uint64_t *p1, unsigned epoch, unsigned bound,
                                const int &stuck, G get, P put) {
  unsigned at[U];
#pragma unroll
  for (int u = 0; u < U; ++u) at[u] = get(u);
#pragma unroll 1
  for (unsigned spin = 0; spin < bound; ++spin) {
    uint64_t w0[U], w1[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned q = at[u] != RES_NONE ? at[u] : 0;  // position 0 exists; its words are not looked at
      w0[u] = ll_get(at32(p0, q));
      w1[u] = ll_get(at32(p1, q));
    }
    unsigned bad = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned d = ((unsigned)(w0[u] >> 32) ^ epoch) | ((unsigned)(w1[u] >> 32) ^ epoch);
      bad |= at[u] != RES_NONE ? d : 0u;
    }
    if (bad == 0) {
#pragma unroll
      for (int u = 0; u < U; ++u) put(u, at[u] != RES_NONE, ll_value(w0[u], w1[u]));
      return true;
    }
    if (LOOK && spin % RES_LOOK == RES_LOOK - 1 &&
        __hip_atomic_load(&stuck, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))
      break;
  }
  return false;
}

// Every workgroup resident, or none goes on: arrivals are counted, the last
// one sets RES_GO, and a workgroup that waits too long (other kernels hold the
// CUs) sets RES_ABORT instead; the first of the two to be set stands for all.
// What does not fit a workgroup (fits) aborts the same way.
__device__ inline int resident_arrive(KrylovScalars *ks, int nblk, int *state, bool fits, unsigned bound) {
  if (threadIdx.x == 0) {
    unsigned *const st = reinterpret_cast<unsigned *>(&ks->pad1);
    if (!fits) atomicCAS(st, (unsigned)RES_PENDING, (unsigned)RES_ABORT);
    if (atomicAdd(reinterpret_cast<unsigned *>(&ks->pad0), 1u) + 1u == (unsigned)nblk)
      atomicCAS(st, (unsigned)RES_PENDING, (unsigned)RES_GO);
    unsigned s = RES_PENDING;
    for (unsigned spin = 0; spin < bound; ++spin) {
      s = __hip_atomic_load(st, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (s != RES_PENDING) break;
    }
    if (s == RES_PENDING) {
      s = atomicCAS(st, (unsigned)RES_PENDING, (unsigned)RES_ABORT);
      if (s == RES_PENDING) s = RES_ABORT;
    }
    *state = (int)s;
  }
  __syncthreads();
  return *state;
}

// Workgroups of resident solves in flight on each device.  They hold a CU
// each, so a solve that would not find its CUs free takes the launch path.
constexpr int MAX_DEVICES = 64;
inline std::atomic<int> g_resident[MAX_DEVICES];

struct ResidentSlots {
  std::atomic<int> *n = nullptr;
  int blocks = 0;
  bool take(int device, int want) {
    if (device < 0 || device >= MAX_DEVICES) return false;
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return false;
    n = &g_resident[device];
    if (n->fetch_add(want) + want > cus) {
      n->fetch_sub(want);
      return false;
    }
    blocks = want;
    return true;
  }
  ~ResidentSlots() {
    if (blocks) n->fetch_sub(blocks);
  }
};

}  // namespace cfd
