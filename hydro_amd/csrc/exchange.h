// exchange.h -- partial results exchanged between the workgroups of one kernel.
//
// For solves of small grids that run in one launch: at most kWholeMaxWg
// workgroups, each waiting for all others once or more per iteration.  That is a
// quarter of the CUs, since kernels of four queues may run at once and the waits
// need a kernel's workgroups to run together; they are bounded (kWholeSpin polls,
// see wait_guard.h), and a solve that gave up is run again by kernels that do
// not wait.  A thread holds one cell while 16 workgroups hold the grid, then two,
// then four: 32 or 64 workgroups cost more per exchange than fewer cells per thread
// save, fewer than 16 less (figures at SplitWhole).
#pragma once

#include <algorithm>

#include "device_common.h"

namespace hg {

constexpr int kWholeThreads = 1024;
constexpr int kWholeMaxWg = 64;
constexpr long kWholeMaxCells = 4L * kWholeThreads * kWholeMaxWg;
constexpr int kWholeLds = 8000;  // doubles
constexpr int kWholeSpin = 1 << 17;
// exchange words [2 parities][4][64], the count of finished workgroups, the
// tags used so far
constexpr int kWholeDone = 2 * 4 * kWholeMaxWg, kWholeEpoch = kWholeDone + 1;
constexpr int kWholeWords = kWholeEpoch + 1;

// The split of n cells: K = 1, 2 or 4 per thread (max_k at most), `cells` per workgroup (a
// multiple of 64).  65025 cells of a Jacobi-PCG: 16 x 4096 4.6 us per
// iteration, 32 x 2048 5.0, 64 x 1024 5.8; 16384 cells: 16 x 1024 3.4,
// 8 x 2048 3.7, 4 x 4096 4.1.
struct WholeSplit {
  int k, wgs, cells;
};
inline WholeSplit SplitWhole(int n, int max_k = 4) {
  WholeSplit s;
  s.k = n <= 16 * kWholeThreads ? 1 : n <= 32 * kWholeThreads ? 2 : max_k;
  s.wgs = (n + s.k * kWholeThreads - 1) / (s.k * kWholeThreads);
  s.cells = ((n + s.wgs - 1) / s.wgs + 63) / 64 * 64;  // <= k kWholeThreads
  s.wgs = (n + s.cells - 1) / s.cells;
  return s;
}

// A value travels as one (float) or two words that each hold 32 bits of it
// under the exchange's number `tag`, so that it needs no flag behind it.
using Word = unsigned long long;
__device__ __forceinline__ Word TagLoad(const Word* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void TagStore(Word* p, unsigned tag, unsigned v) {
  __hip_atomic_store(p, Word(tag) << 32 | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double FromWords(Word lo, Word hi) {
  return __hiloint2double(int(unsigned(hi)), int(unsigned(lo)));
}

// Folds of non-negative maxima (0 for lanes and workgroups that are not there)
// and of sums, in a fixed order.
struct SumFold {
  template <int R>
  static __device__ __forceinline__ double Dpp(double v) {
    return DppSum<R>(v);
  }
};
struct MaxFold {
  template <int R>
  static __device__ __forceinline__ double Dpp(double v) {
    return DppMax<R>(v);
  }
};

// Folds v over all workgroups; `extra` = post(folded), formed in one wave.
// Words of a parity are written again two exchanges later, when every workgroup
// has read them.  `all` runs in every wave after the first barrier, `others` in
// all but the first, while that waits for the words.  False, in the whole
// workgroup: gave up.
template <class Fold, int NV, class Post, class All, class Others>
__device__ __forceinline__ bool Exchange(double (&v)[NV], double& extra, unsigned tag,
                                         Word* words, int spin, int* gave_up, Post&& post,
                                         All&& all_waves, Others&& others) {
  constexpr int kWaves = kWholeThreads / 64;  // at most 16: one row of lanes
  __shared__ double red[NV][kWaves];
  __shared__ double tot[NV + 1];
  const int lane = threadIdx.x & 63, W = gridDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const double s = Fold::template Dpp<6>(v[q]);
    if (lane == 63) red[q][wave] = s;
  }
  __syncthreads();
  all_waves();
  bool ok = true;
  if (wave == 0) {
#pragma unroll
    for (int q = 0; q < NV; ++q)
      v[q] = LaneOf(Fold::template Dpp<4>(lane < kWaves ? red[q][lane] : 0.), 15);
    if (W > 1) {
      Word* const mine = words + (tag & 1) * 4 * kWholeMaxWg;
      if (lane == 0) {
#pragma unroll
        for (int q = 0; q < NV; ++q) {
          TagStore(mine + 2 * q * kWholeMaxWg + blockIdx.x, tag, unsigned(__double2loint(v[q])));
          TagStore(mine + (2 * q + 1) * kWholeMaxWg + blockIdx.x, tag,
                   unsigned(__double2hiint(v[q])));
        }
      }
      Word g[2 * NV] = {};
      for (int n = 0;; ++n) {
        if (n == spin) {
          ok = false;
          break;
        }
        bool all = true;
#pragma unroll
        for (int i = 0; i < 2 * NV; ++i) g[i] = TagLoad(mine + i * kWholeMaxWg + min(lane, W - 1));
#pragma unroll
        for (int i = 0; i < 2 * NV; ++i) all = all && unsigned(g[i] >> 32) == tag;
        if (__all(all)) break;
      }
#pragma unroll
      for (int q = 0; q < NV; ++q)
        v[q] = LaneOf(
            Fold::template Dpp<6>(lane < W ? FromWords(g[2 * q], g[2 * q + 1]) : 0.), 63);
    }
    const double e = post(v);
    if (lane == 0) {
#pragma unroll
      for (int q = 0; q < NV; ++q) tot[q] = v[q];
      tot[NV] = e;
    }
  } else {
    ok = others();
  }
  if (!ok) *gave_up = 1;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] = tot[q];
  extra = tot[NV];
  return *gave_up == 0;
}

// The last workgroup of a solve to finish: the next solve's words.  True there.
__device__ __forceinline__ bool FinishWhole(Word* words, unsigned tag) {
  if (__hip_atomic_fetch_add(words + kWholeDone, Word(1), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT) != gridDim.x - 1)
    return false;
  words[kWholeDone] = 0;
  words[kWholeEpoch] = tag;
  return true;
}

// After a solve that gave up: no word of it is taken for one of the next solve.
// Its tags, from the epoch on, are used again, so every word goes back to the
// epoch, which the next solve has behind it.
static __global__ void __launch_bounds__(256) KWholeReset(Word* words, long n) {
  const Word epoch = words[kWholeEpoch];
  for (long i = blockIdx.x * 256l + threadIdx.x; i < n; i += gridDim.x * 256l)
    if (i != kWholeEpoch) words[i] = i == kWholeDone ? Word(0) : epoch << 32;
}
inline void WholeReset(Word* words, long n, hipStream_t st) {
  KWholeReset<<<unsigned(std::min((n + 255) / 256, 256l)), 256, 0, st>>>(words, n);
}

}  // namespace hg
