// hmv_feed.h -- feeding the iterations of a device-resident solver.
//
// A solver's scalars and stopping tests live on the device.  The kernel that
// ends an iteration writes how many have ended, and whether the solve has
// stopped, to one word of pinned host memory; the host launches iterations
// so that at most kFeedWindow of them are on the stream beyond the last one it
// has seen end, and stops launching when it sees the stop.  A window of two
// keeps the stream busy (an iteration is launched while the one before it
// runs) and leaves at most one launched iteration that finds the solve
// stopped and does nothing.  Reading the state back after every 8 launches
// instead left up to 7 such iterations of 25 to 30 us each and an idle
// stream of 20 to 30 us at each read; one hipGraph launch per iteration left
// 5 to 8 us between iterations where direct launches of its 9 to 13 kernels
// leave none.  Together: BiCGSTAB at 5k unknowns 3.03 -> 2.76 ms, GCR
// refinement at 5k 4.4 -> 3.2, at 82k 17.5 -> 15.7, of 8 instances of 320 to
// 20,480 unknowns 11.4 -> 10.0.
#ifndef HMV_FEED_H
#define HMV_FEED_H

#include <hip/hip_runtime.h>

#include <algorithm>

#include "hmv_engine.h"

constexpr int kSolveMaxBlocks = 512;  // workgroups of a dot product over one vector

// Pinned host memory of an arena's solvers, written by their kernels.
struct HmvSolveHost {
  unsigned long long progress;  // iterations ended << 1 | stopped
  int step, status;             // valid once stopped
  double rnorm, bnorm;
  double part[2 * kSolveMaxBlocks];  // partial dot products read on the host
};

// ... followed by one of these for each instance of a multi-instance arena.
struct HmvInstHost {
  double rr, bb;           // summed dots of its segment
  int step, done, status;  // valid once stopped
  int stopped;             // written by the host, read by the kernels
};

namespace hmv {

constexpr int kFeedWindow = 2;

__host__ __device__ inline HmvInstHost *inst_host(HmvSolveHost *h) {
  return reinterpret_cast<HmvInstHost *>(h + 1);
}

// Has the values, loads still under way included, in registers here: the
// loads above are issued together and waited for once.  The solvers' vector
// kernels are a few dependent round trips of 0.7 us long, and without this
// each of flag, state, partials and first elements was one of them: BiCGSTAB
// at 1,280 unknowns 1.30 -> 1.25 ms, at 5k 2.61 -> 2.56.
__device__ inline void together(int a, double b, double c, double d) {
  asm volatile("" : : "v"(a), "v"(b), "v"(c), "v"(d));
}
__device__ inline void together(int a, double b, double c, double d, double e, double f, double g,
                                double h) {
  asm volatile("" : : "v"(a), "v"(b), "v"(c), "v"(d), "v"(e), "v"(f), "v"(g), "v"(h));
}

__device__ inline void publish(HmvSolveHost *h, int ticks, int done) {
  const unsigned long long v = ((unsigned long long)ticks << 1) | (done ? 1 : 0);
  if (done)
    __hip_atomic_store(&h->progress, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  else
    __hip_atomic_store(&h->progress, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The arena's pinned solver memory, made on its first solve and freed with
// it, with the progress word cleared; nothing on stream s may still write
// there, so s is drained first.
inline hipError_t solve_host(hmv_arena_s *a, hipStream_t s, HmvSolveHost *&h) {
  hipError_t e;
  if (!a->solve_host &&
      (e = hipHostMalloc((void **)&a->solve_host,
                         sizeof(HmvSolveHost) + a->seg.size() * sizeof(HmvInstHost),
                         hipHostMallocMapped | hipHostMallocCoherent)) != hipSuccess) {
    a->solve_host = nullptr;
    return e;
  }
  if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
  h = a->solve_host;
  __atomic_store_n(&h->progress, 0ull, __ATOMIC_RELEASE);
  return hipSuccess;
}

inline bool stopped(const HmvSolveHost *h) {
  return __atomic_load_n(&h->progress, __ATOMIC_ACQUIRE) & 1;
}

// Calls launch() (one iteration on stream s, ending in a publish) until
// `upto` iterations of the solve are launched or it has stopped.
template <class Launch>
hipError_t feed(const HmvSolveHost *h, hipStream_t s, int &launched, int upto, Launch &&launch) {
  hipError_t e;
  unsigned spins = 0;
  while (launched < upto) {
    const unsigned long long v = __atomic_load_n(&h->progress, __ATOMIC_ACQUIRE);
    if (v & 1) break;
    if (launched - (int)(v >> 1) < kFeedWindow) {
      if ((e = launch()) != hipSuccess) return e;
      ++launched;
      spins = 0;
    } else if ((++spins & 0xffff) == 0) {
      // a failed stream publishes nothing more
      e = hipStreamQuery(s);
      if (e == hipErrorNotReady)
        (void)hipGetLastError();
      else if (e != hipSuccess)
        return e;
      else if (__atomic_load_n(&h->progress, __ATOMIC_ACQUIRE) == v)
        return hipErrorUnknown;
    } else {
      __builtin_ia32_pause();
    }
  }
  return hipSuccess;
}

}  // namespace hmv

#endif
