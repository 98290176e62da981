// sor.hip -- exact-order lexicographic SOR with many sweeps in flight.
//
// The reference's gauss_seidel (linear.hpp:685-715) updates cells in raw
// order; cell (i,j) of sweep s needs sweep s's values of its west and south
// neighbours and sweep s-1's of itself and its east and north neighbours.
// All cells with the same i + j + 2 s are therefore independent: a sweep can
// follow the one before it two wavefront steps behind.  One workgroup runs
// such a pipeline.  Let a be the shorter and b the longer side, t a cell's
// index along the short side and m along the long one.  Thread (q, t) takes
// the cells of line t for two consecutive sweeps ("stages" 2q and 2q + 1): at
// step T row m = T - t - 4q of the first and row m - 2 of the second.  A stage
// that reaches the end of its line goes on with the sweep P = 2Q later at
// once (b >= 2P + 4, so its predecessor is far enough ahead), and every
// thread is busy at every step: a sweep costs b / P steps instead of the
// a + b of one sweep at a time.
//
// Values pass between neighbouring threads and stages through LDS (written
// at one step, read at the next); the first stage reads the sweep before it
// from memory.  The rows' coefficients are repacked once per solve so that
// the cells of one step are contiguous: cell (t, m) sits in row (t + m) mod b
// at column t, which uses exactly a b entries.  (Read in place, the 64 lanes
// of a wave are on 64 rows, so each load of the sweep-at-a-time kernel
// touches 64 cache lines.)  A thread's second stage reuses the coefficients
// its first stage loaded two steps earlier from registers.
//
// The stop rule needs a whole sweep's max |corr|; later sweeps run on
// meanwhile, each writing its own buffer of a ring, and the sweep that ends
// the solve is then copied out.  Every cell value is computed with the same
// operations on the same operands as in the one-sweep kernel, and terms
// outside the grid enter as +0 (0 * 0), which changes no sum (the sum starts
// at +0), so the result is the reference's bit for bit.  Compiled with
// -ffp-contract=off.
//
// What bounds it: the instructions of a step (about 140 per thread for two
// cells, 52 of them FP64), with 2 Q a <= 2048 cells per step on one CU; and
// where the long side has room for several workgroups (KSorChain, below) the
// b / (G P) steps of a sweep, plus once per solve the a + b to fill the
// pipeline.  Per sweep, against the sweep-at-a-time kernel (101 sweeps unless
// noted): 64x64 3.7 against 34 us; 256x128 at 701 sweeps 3.7 (one workgroup 15.3)
// against 177 us; 333x217 9.8 (44) against 440 us.
// For one workgroup 1024 threads beat 512 and 256 (256x128: 15.3, 19.7, 30.9
// us); for each of several 512 (256x128: 3.7; 1024: 7.2, 256: 4.8 us).
#include "device_common.h"
#include "kernels.h"
#include "sor_plan.h"

namespace hg {

namespace {

// Barrier between steps.  It orders the LDS exchange and leaves the loads in
// flight; of the global stores it waits for those of two steps before and
// earlier (a step issues at least 3 loads and 2 stores per wave, vector
// memory operations complete in order on vmcnt, and at most 10 may be
// outstanding here), which the first stage reads four steps after they were
// issued at the earliest.  The workgroup's waves share one L1.
__device__ __forceinline__ void StepBarrier() {
  asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ void ChainBarrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  asm volatile("" ::: "memory");
}

// One cell's row: own (the neighbour before it on its line: new value),
// cross (the neighbour on the line before: new), xold (on the line after:
// old), nold (the next cell of its line: old), diagonal, constant.
struct SorRow {
  double2 oc, xn, ck;
};

// Rows into the skewed order, zero where the neighbour is outside the grid.
__global__ void __launch_bounds__(256)
KSorPack(int nx, int ny, Rows r, const double* __restrict__ k, int tr, double2* __restrict__ oc,
         double2* __restrict__ xn, double2* __restrict__ ck, double* __restrict__ xf,
         double* head, int head_doubles) {
  if (blockIdx.x == 0) {  // no sweep has ended, no steps done
    int* const h = reinterpret_cast<int*>(head);
    for (int z = threadIdx.x; z < 2 * head_doubles; z += 256) h[z] = z == 0 ? kNever : 0;
  }
  const int a = tr ? ny : nx, b = tr ? nx : ny;
  const int d = blockIdx.x * 256 + threadIdx.x;  // skewed index, so that stores coalesce
  if (d >= a * b) return;
  const int t = d % a, row = d / a;
  const int m = row >= t ? row - t : row - t + b;  // t < a <= b
  const int i = tr ? m : t, j = tr ? t : m;
  const int c = i + nx * j;
  const double s = j > 0 ? r.s[c] : 0., w = i > 0 ? r.w[c] : 0.;
  const double e = i < nx - 1 ? r.e[c] : 0., n = j < ny - 1 ? r.n[c] : 0.;
  oc[d] = tr ? double2{w, s} : double2{s, w};
  xn[d] = tr ? double2{n, e} : double2{e, n};
  // (+0 turns a constant of -0 into +0: the kernel's sum of products may be
  // -0 where the reference's, which starts at +0, is +0; k + sum is then the
  // same)
  ck[d] = double2{r.c[c], k[c] + 0.};
  if (xf) xf[d] = 0.;
}

__global__ void __launch_bounds__(256)
KSorUnpack(int nx, int ny, int tr, const double* __restrict__ ring,
           const double* __restrict__ head, double* __restrict__ x) {  // head[1]: the ring slot
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= nx * ny) return;
  const int a = tr ? ny : nx, b = tr ? nx : ny;
  const int i = c % nx, j = c / nx;
  const int t = tr ? j : i, m = tr ? i : j;
  const int row = t + m >= b ? t + m - b : t + m;
  const long slot = reinterpret_cast<const long long*>(head)[1];
  x[c] = ring[slot * nx * ny + long(row) * a + t];
}

// The same by `threads` threads of a workgroup that has formed the values, for grids
// so small (kCopyOutCells) that a launch of its own costs more: 101 sweeps of 24x24
// 197 us with the launch, 193 this way, 64x64 376 and 373.
template <bool TR>
__device__ __forceinline__ void CopyOut(int a, int b, const double* from, double* __restrict__ x,
                                        int t, int threads) {
  for (int d = t; d < a * b; d += threads) {
    const int row = d / a, l = d - row * a;
    const int m = row >= l ? row - l : row - l + b;
    x[TR ? m + b * l : l + a * m] = from[d];
  }
}

__device__ __forceinline__ double AgentLoad(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int AgentLoad(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <bool TR>
__device__ __forceinline__ double SorCell(const SorRow& r, double own, double cross, double xold,
                                          double nold, double old, double omega, double& dmax) {
  const double po = r.oc.x * own, pc = r.oc.y * cross;  // new: south and west
  const double px = r.xn.x * xold, pn = r.xn.y * nold;  // old: east and north
  double sum = po + pc;
  sum += TR ? pn : px;  // east
  sum += TR ? px : pn;  // north
  const double value = -(r.ck.y + sum) / r.ck.x;
  const double corr = value - old;
  dmax = fmax(dmax, fabs(corr));
  return old + corr * omega;
}

// ---- the first sweeps, one after another --------------------------------------
// A pipeline takes longer over its first sweep than a workgroup with nothing else
// to do, and a solve often ends there (a start that is nearly the solution).  So
// one more workgroup of the same launch runs the first kFirstSweeps sweeps one
// after another in xf; if the stop rule is met within them it ends the solve:
// info, the result's slot, `word` lowered to kEndedFirst.  The pipeline leaves
// when it sees that.  Where both end the solve they do at the same sweep, with
// the same values.  Neither waits for the other.
//
// Device time in us of a solve that ends in its first and second sweep (launches
// and the read back of info, about 40, in all of them): a sweep at a time in place,
// the pipeline alone, with this: 16x16 48, 62 | 55, 57 | 52, 58; 64x64 102, 135 |
// 162, 165 | 79, 102; 128x128 249, 338 | 411, 418 | 103, 160; 512x512 3490, 5690 |
// 1776, 1808 | 478, 890.  A third sweep would end after the pipeline could (512x512:
// two take 840 us, the pipeline's first decision 900) and gain little elsewhere.
//
// Thread t takes line t, one row per step.  The value before it on its line stays
// in a register, that of line t - 1 comes by a lane shift, between waves through
// LDS: wave w is w groups of kG steps behind the first, one barrier per group (kG 4,
// or 3 where 4 would make the kernel spill registers).
// All operands are loaded kG steps ahead; an old value is loaded before the step
// that writes its cell, by the same wave or by one a group behind.
template <bool TR, int kG>
__device__ __forceinline__ void FirstSweeps(int a, int b, const double2* __restrict__ oc,
                                            const double2* __restrict__ xn,
                                            const double2* __restrict__ ck, double* xf, double tol,
                                            int limit, double omega, long long slot, int* word,
                                            double* head, unsigned long long* __restrict__ info,
                                            double* __restrict__ x) {
  constexpr int kRing = 16;
  __shared__ double edge[kSorThreads / 64][kRing];  // values of a wave's last lane, by step
  __shared__ double red[kSorThreads / 64];
  const int t = threadIdx.x, nw = (a + 63) >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  if (wave >= nw) return;
  const unsigned tc = unsigned(min(t, a - 1)), tx = t < a - 1 ? tc + 1 : tc;
  const int ng = (a + b - 2 + kG) / kG;  // groups of the a + b - 1 steps
  for (int s = 0;; ++s) {
    struct Step {
      SorRow r;
      double next, cross;  // old values: the next cell of the line, the line after's
    } o[kG];
    int lrow = 0, srow = 0;  // rows of the next load and of the next store
    auto Load = [&](Step& q) {
      const int nrow = lrow + 1 == b ? 0 : lrow + 1;
      const size_t d = size_t(unsigned(lrow)) * unsigned(a);
      const size_t e = size_t(unsigned(nrow)) * unsigned(a);
      q.r.oc = (oc + d)[tc];
      q.r.xn = (xn + d)[tc];
      q.r.ck = (ck + d)[tc];
      q.next = (xf + e)[tc];
      q.cross = (xf + e)[tx];
      lrow = nrow;
    };
    double val = 0., old = xf[tc], dmax = 0., out[kG], e[kG];
#pragma unroll
    for (int i = 0; i < kG; ++i) Load(o[i]);
    for (int k = 0; k < wave; ++k) ChainBarrier();
    for (int g = 0; g < ng; ++g) {
#pragma unroll
      for (int i = 0; i < kG; ++i)
        e[i] = wave == 0 ? 0. : edge[wave - 1][(g * kG + i - 1) & (kRing - 1)];
#pragma unroll
      for (int i = 0; i < kG; ++i) {
        const int m = g * kG + i - t;
        const Step& q = o[i];
        const double cross = LaneNext<true>(val, e[i]);
        double d = 0.;
        val = SorCell<TR>(q.r, m == 0 ? 0. : val, cross, t < a - 1 ? q.cross : 0.,
                          m < b - 1 ? q.next : 0., old, omega, d);
        if (m >= 0 && m < b && t < a) {
          (xf + size_t(unsigned(srow)) * unsigned(a))[tc] = val;
          dmax = fmax(dmax, d);
        }
        old = q.next;
        out[i] = val;
        srow = srow + 1 == b ? 0 : srow + 1;
        __builtin_amdgcn_sched_barrier(0);
        Load(o[i]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (nw > 1) {
        if ((t & 63) == 63)
#pragma unroll
          for (int i = 0; i < kG; ++i) edge[wave][(g * kG + i) & (kRing - 1)] = out[i];
        ChainBarrier();
      }
    }
    for (int k = wave + 1; k < nw; ++k) ChainBarrier();
    const double md = LaneOf(DppMax<6>(dmax), 63);
    if ((t & 63) == 0) red[wave] = md;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the next sweep reads this one's values
    __syncthreads();
    double diff = red[0];
    for (int w = 1; w < nw; ++w) diff = fmax(diff, red[w]);
    const bool met = !(diff > tol);
    if (met || s == limit) {
      if (t == 0) {
        info[0] = (unsigned long long)(met ? s : s + 1);
        info[1] = (unsigned long long)__double_as_longlong(diff);
        reinterpret_cast<long long*>(head)[1] = slot;
        __hip_atomic_fetch_min(word, kEndedFirst, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      if (x) CopyOut<TR>(a, b, xf, x, t, 64 * nw);
      return;
    }
    if (s + 1 == kFirstSweeps) return;
  }
}

template <bool TR>
__global__ void __launch_bounds__(kSorThreads)
KSorPipe(int a, int b, int Q, int rounds, const double2* __restrict__ oc,
         const double2* __restrict__ xn, const double2* __restrict__ ck, double* ring, double* xf,
         double tol, int limit, double omega, double* head, unsigned long long* __restrict__ info,
         double* __restrict__ x) {
  // [2 step parities][Q][a + 2] values (first, second stage) with a zero
  // pad either side, then the sweeps' maxima
  extern __shared__ double2 lds2[];
  __shared__ int flag;  // 1 + the group of four steps in which a sweep ended the solve
  __shared__ int result;  // its ring slot, if a sweep of this workgroup did
  const int W = a + 2;
  double2* const val = lds2;
  unsigned long long* const sd = reinterpret_cast<unsigned long long*>(lds2 + 2 * Q * W);
  const int P = 2 * Q, R = rounds * P;
  int* const word = reinterpret_cast<int*>(head);  // kNever until FirstSweeps ends the solve
  if (blockIdx.x == 1) {
    FirstSweeps<TR, 3>(a, b, oc, xn, ck, xf, tol, limit, omega, R, word, head, info, x);
    return;
  }
  const int tid = threadIdx.x;
  for (int z = tid; z < 2 * Q * W; z += blockDim.x) val[z] = double2{0., 0.};
  for (int z = tid; z < R; z += blockDim.x) sd[z] = 0ull;
  if (tid == 0) {
    flag = 0;
    result = -1;
  }
  __syncthreads();
  const bool live = tid < Q * a;
  const int q = live ? tid / a : 0, t = live ? tid - q * a : 0;
  // Byte offsets, 32 bits (PlanSor): of a cell within an array of doubles,
  // of a sweep's buffer (slot) within the ring.
  const unsigned n8 = unsigned(a) * unsigned(b) * 8u, a8 = unsigned(a) * 8u;
  const unsigned round8 = unsigned(P) * n8, ring8 = unsigned(rounds) * round8;
  const char* const ringc = reinterpret_cast<const char*>(ring);
  // The first stage's cell: row m of line t, in round rd (sweep 2 q + P rd;
  // negative before the thread's start, when it works on whatever is there:
  // nothing it stores then is read before it is stored again in round 0 or
  // later).  The second stage's cell is the first's of two steps before, so
  // m == 0, 2 begin a line for the first / second stage and m == b - 1, 1
  // end one.
  int m = -t - 4 * q, rd = 0;
  while (m < 0) {
    m += b;
    --rd;
  }
  int rm = ((rd % rounds) + rounds) % rounds;  // the round's place in the ring
  unsigned slot = unsigned(2 * q) * n8 + unsigned(rm) * round8;
  const int row0 = ((-4 * q) % b + b) % b;
  unsigned off = unsigned(row0) * a8 + unsigned(t) * 8u;
  unsigned pos1 = 0u, pos2 = 0u;  // slot + off one and two steps ago (the second stage's cell)
  SorRow c[4];
  auto Load = [&](SorRow& o, unsigned at) {
    o.oc = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(oc) + 2u * at);
    o.xn = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(xn) + 2u * at);
    o.ck = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(ck) + 2u * at);
  };
  {
    const unsigned o1 = off >= a8 ? off - a8 : off - a8 + n8;
    const unsigned o2 = o1 >= a8 ? o1 - a8 : o1 - a8 + n8;
    Load(c[0], off);
    Load(c[3], o1);
    Load(c[2], o2);
    pos1 = slot + o1;
    pos2 = slot + o2;
  }
  // the first stage of q = 0 reads the sweep before its own (the last stage,
  // a round earlier) from the ring: the next cell of its line (which is also
  // the old value of the cell it takes next) and the line after's.  For the
  // step whose cell is row mm, in slot `sl`, `at` the offset one row on:
  // (raw values; the step that uses them drops what does not exist)
  auto LoadPrev = [&](double2& g, int mm, unsigned sl, unsigned at) {
    if (q == 0) {
      const unsigned last = round8 - n8;  // the round's last stage
      const unsigned before = (sl >= round8 ? sl - round8 : sl - round8 + ring8) + last;
      // at the line's end the next cell is the next round's
      const unsigned from = mm == b - 1 ? sl + last : before;
      g.x = *reinterpret_cast<const double*>(ringc + (from + at));
      // (the last line has no line after it: its own address, not used)
      g.y = *reinterpret_cast<const double*>(ringc + (before + at + (t < a - 1 ? 8u : 0u)));
    }
  };
  auto RowOn = [&](unsigned o) {
    o += a8;
    return o >= n8 ? o - n8 : o;
  };
  double2 g[2] = {double2{0., 0.}, double2{0., 0.}};
  LoadPrev(g[0], m, slot, RowOn(off));
  double2* const mine = val + q * W + t;
  double ownA = 0., ownB = 0., oldA = 0., h1 = 0., h2 = 0., dA = 0., dB = 0.;
  const int look = (a + b) / 4 + kFirstSweeps;
  int group = 0, ended = kNever;
  // sweep s (in ring slot `idx`) has just finished: the stop rule,
  // do { sweep } while (diff > tol && iter++ < limit), sweeps in order
  auto Decide = [&](int s, int idx) {
    const unsigned long long bits = sd[idx];
    sd[idx] = 0ull;
    if (flag) return;
    const double diff = __longlong_as_double((long long)bits);
    const bool met = !(diff > tol);
    if (met || !(s < limit)) {
      info[0] = (unsigned long long)(met ? s : s + 1);
      info[1] = bits;
      reinterpret_cast<long long*>(head)[1] = idx;
      result = idx;
      flag = group + 1;
    }
  };
  for (;; ++group) {
    // (from step a + b + 2 kFirstSweeps on this workgroup has decided them itself)
    if (group < look && tid == 0) {  // as the group before found it
      if (ended != kNever && !flag) flag = group + 1;
      ended = AgentLoad(word);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // the loads of step T + 1, then step T
      const unsigned noff = RowOn(off);
      Load(c[(i + 1) & 3], noff);
      int m1 = m + 1, rd1 = rd, rm1 = rm;
      unsigned slot1 = slot;
      if (m1 == b) {
        m1 = 0;
        ++rd1;
        ++rm1;
        slot1 += round8;
        if (rm1 == rounds) {
          rm1 = 0;
          slot1 -= ring8;
        }
      }
      LoadPrev(g[(i + 1) & 1], m1, slot1, RowOn(noff));
      if (live) {
        const SorRow &ca = c[i & 3], &cb = c[(i + 2) & 3];
        const double2* const pv = mine + ((i & 1) ^ 1) * Q * W;
        const double2 west = pv[0];      // line t - 1: both stages, new
        const double eastA = pv[2].x;    // line t + 1, first stage: old for the second
        double nextA, crossA;
        if (q == 0) {
          nextA = rd1 > 0 ? g[i & 1].x : 0.;  // (the next cell is of round rd1)
          crossA = (rd > 0 && t < a - 1) ? g[i & 1].y : 0.;
        } else {
          nextA = pv[1 - W].y;
          crossA = pv[2 - W].y;
        }
        if (t == a - 1 && (m == 0 || m == 2) && rd > 0) {
          // the last line ended at the last step: m == 0 the first stage's
          const int st = 2 * q + (m >> 1);
          Decide(st + P * (rd - 1), st + P * (rm == 0 ? rounds - 1 : rm - 1));
        }
        const double xA = SorCell<TR>(ca, m != 0 ? ownA : 0., west.x, crossA, m1 != 0 ? nextA : 0.,
                                      oldA, omega, dA);
        const double xB = SorCell<TR>(cb, m != 2 ? ownB : 0., west.y, eastA, m != 1 ? h1 : 0., h2,
                                      omega, dB);
        mine[(i & 1) * Q * W + 1] = double2{xA, xB};
        const unsigned pos = slot + off;
        *reinterpret_cast<double*>(reinterpret_cast<char*>(ring) + pos) = xA;
        *reinterpret_cast<double*>(reinterpret_cast<char*>(ring) + (pos2 + n8)) = xB;
        pos2 = pos1;
        pos1 = pos;
        if (m1 == 0) {  // the first stage's line ends
          if (rd >= 0)
            atomicMax(&sd[2 * q + P * rm], (unsigned long long)__double_as_longlong(dA));
          dA = 0.;
        }
        if (m == 1) {  // the second's, of the round before
          if (rd > 0)
            atomicMax(&sd[2 * q + 1 + P * (rm == 0 ? rounds - 1 : rm - 1)],
                      (unsigned long long)__double_as_longlong(dB));
          dB = 0.;
        }
        oldA = nextA;
        h2 = h1;
        h1 = xA;
        ownA = xA;
        ownB = xB;
      }
      off = noff;
      m = m1;
      rd = rd1;
      rm = rm1;
      slot = slot1;
      StepBarrier();
    }
    // a flag of this group or an earlier one: seen by every thread alike (a
    // thread ahead may already have set the next group's)
    const int f = flag;
    if (f != 0 && f <= group + 1) break;
  }
  if (x) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every wave's values are in the ring
    __syncthreads();
    if (result >= 0) CopyOut<TR>(a, b, ring + size_t(result) * (n8 / 8u), x, tid, blockDim.x);
  }
}

// ---- several workgroups -----------------------------------------------------
// The same pipeline over G workgroups: workgroup g runs stages g P .. g P +
// P - 1 (its threads' lines padded to whole waves, so that q is uniform in a
// wave), the last stage of one feeding the first of the next through memory,
// and the last workgroup's the first's, a round (b steps) later.  All
// workgroups count the same virtual steps: workgroup g's first stage starts
// at step g span, where G span <= b, so a line is span - 2 P >= kLag steps
// further on in the workgroup before than its reader needs.
//
// What a first stage reads was written kLag + 1 or more steps before, into the
// writer's log (row = step mod le).  Steps go in groups of four.  At a
// group's start the first stage's waves issue the loads for the next group;
// at its end the workgroup publishes the steps before the group, whose stores
// are complete (vmcnt) in every wave.  A reader so needs progress that was
// published about 12 steps ago and normally does not wait; it polls when it
// must, a bounded number of times, after which the solve is marked failed
// (stop = -1) and every workgroup leaves; the caller then runs the
// one-workgroup kernel.
// Log and flags are written and read with agent-scope accesses: the
// workgroups are on different XCDs, each with its own L2.
//
// A sweep's workgroup applies the stop rule and lowers `stop`; every
// workgroup runs on to the virtual step by which all earlier sweeps were
// decided too.  Only the lines between workgroups are kept, so the result is
// found by a second launch (tail) of one workgroup, which repeats the sweeps
// from the last logged one before the stop to the stop -- unless the solve
// ran to its last sweep, which is written as it is computed.
template <bool TR, int MAXT>
__global__ void __launch_bounds__(MAXT)
KSorChain(SorChain ch, const double2* __restrict__ oc, const double2* __restrict__ xn,
          const double2* __restrict__ ck, double* head, double* logs, double* out, double* xf,
          double tol, double omega, unsigned long long* __restrict__ info) {
  extern __shared__ double2 lds2[];  // as KSorPipe's; maxima [stage][4 rounds]
  __shared__ int lstop;
  int* const stop = reinterpret_cast<int*>(head);
  int* const progress = reinterpret_cast<int*>(head + kChainProgress);
  unsigned long long* const rec = reinterpret_cast<unsigned long long*>(head + kChainRec);
  const int a = ch.a, b = ch.b, Q = ch.Q, P = 2 * Q, W = a + 2, le = ch.le, span = ch.span;
  const long log_n = long(le) * a;
  int G = ch.G, wg = blockIdx.x, limit = ch.limit;
  if (wg == G) {
    FirstSweeps<TR, MAXT <= 512 ? 4 : 3>(a, b, oc, xn, ck, xf, tol, limit, omega, 1, stop, head, info,
                                           nullptr);
    return;
  }
  // where the first stage's input comes from: the log of workgroup `src`, the
  // values for this workgroup's step T in row T + shift; the zero start where
  // T - t < from
  int src = wg == 0 ? G - 1 : wg - 1, start = wg * span;
  int shift = wg == 0 ? (G - 1) * span + 2 * P - b - 1 : 2 * P - span - 1;
  int from = wg == 0 ? b : -1;
  if (ch.tail) {
    const int s = *stop;
    if (s == kEndedFirst) return;
    // gave up, or ran out of step numbers before every sweep up to s was decided
    // (kNever, the last number of 32 bits, is past them too: G P < b)
    if (s < 0 || ChainDoneStep(s, P, G * P, span, a, b) + 4 > kChainMaxStep) {
      if (threadIdx.x == 0) info[0] = ~0ull;
      return;
    }
    const int st = s % (G * P);
    if (threadIdx.x == 0) {
      const unsigned long long bits = rec[st];
      info[0] = (unsigned long long)(!(__longlong_as_double((long long)bits) > tol) ? s : s + 1);
      info[1] = bits;
    }
    if (s == limit) return;  // already written
    // sweeps s - p .. s again, p the stage within its workgroup, from the
    // sweep before them: logged by the workgroup before (a round earlier for
    // the first), or the zero start.  Its cell (t, m) is in log row src span
    // + 2 (P - 1) + t + rs b + m, and is read as the next cell of m - 1 at
    // step t + m - 1.
    const int p = st % P, w = st / P, rd = s / (G * P);
    const int rs = w == 0 ? rd - 1 : rd;
    src = w == 0 ? G - 1 : w - 1;
    shift = src * span + 2 * (P - 1) + rs * b + 1;
    from = rs < 0 ? kNever : -1;
    G = 1;
    wg = 0;
    start = 0;
    limit = p;
  }
  const bool wait = !ch.tail;
  // (there is nothing to wait for before a workgroup's start)
  if (threadIdx.x == 0 && wait)
    __hip_atomic_store(progress + 16 * wg, start, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int tid = threadIdx.x;
  double2* const val = lds2;
  unsigned long long* const sd = reinterpret_cast<unsigned long long*>(lds2 + 2 * Q * W);
  for (int z = tid; z < 2 * Q * W; z += blockDim.x) val[z] = double2{0., 0.};
  for (int z = tid; z < 4 * P; z += blockDim.x) sd[z] = 0ull;
  if (tid == 0) lstop = kNever;
  __syncthreads();
  const int q = __builtin_amdgcn_readfirstlane(tid / ch.ap);
  const int t = tid - q * ch.ap;
  const bool live = t < a, first = q == 0, last = q == Q - 1;
  const int ptot = G * P;  // sweeps per round
  // the step within the pipeline's round, and the cell's place: m == 0 when
  // tm == ez (see KSorPipe for m == 1, 2, b - 1); rd the lane's round
  int ez = t + 4 * q, rd = 0;
  while (ez >= b) {
    ez -= b;
    --rd;
  }
  if (ez > 0) --rd;
  int tm = 0;
  // the round in which a stage of these runs the last sweep (-1: none does)
  auto LimRound = [&](int stage) {
    const int d = limit - (wg * P + stage);
    return d >= 0 && d % ptot == 0 ? d / ptot : -1;
  };
  const int limA = LimRound(2 * q), limB = LimRound(2 * q + 1);
  int row = ((-4 * q) % b + b) % b;  // skewed row of the first stage's cells
  int pr1 = row >= 1 ? row - 1 : row - 1 + b, pr2 = row >= 2 ? row - 2 : row - 2 + b;
  SorRow c[4];
  const unsigned t16 = unsigned(live ? t : 0) * 16u;
  auto Load = [&](SorRow& o, int r) {
    const size_t base = size_t(unsigned(r)) * unsigned(a) * 16u;
    o.oc = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(oc) + base + t16);
    o.xn = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(xn) + base + t16);
    o.ck = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(ck) + base + t16);
  };
  Load(c[0], row);
  Load(c[3], pr1);
  Load(c[2], pr2);
  const double* const in = logs + src * log_n;
  double* const mylog = logs + wg * log_n;
  // first stage: its input for the group's four steps, and for the next
  // group's (next cell of the line, line after's cell)
  double2 cur[4], nxt[4];
  auto Fetch = [&](double2 (&g)[4], int T) {
    // rows below 0 are never used
    int r = T + shift;
    r = r < 0 ? 0 : r % le;
    const int tc = live ? t : 0, tx = t < a - 1 ? tc + 1 : tc;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double* const lr = in + long(r) * a;
      g[i].x = AgentLoad(lr + tc);
      g[i].y = AgentLoad(lr + tx);
      if (++r == le) r = 0;
    }
  };
  int seen = 0, ahead = 0, ahead_stop = kNever;
  // the source's steps below `need` are complete, or the solve has ended
  // (false: gave up)
  auto Await = [&](int need) {
    if (!wait) return true;
    seen = max(seen, ahead);
    for (int k = 0; seen < need; ++k) {
      if (k == ch.spin) {
        __hip_atomic_fetch_min(stop, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return false;
      }
      seen = AgentLoad(progress + 16 * src);
      if (seen >= need) break;
      if (AgentLoad(stop) != kNever) return true;
    }
    return true;
  };
  double ownA = 0., ownB = 0., oldA = 0., h1 = 0., h2 = 0., dA = 0., dB = 0.;
#pragma unroll
  for (int i = 0; i < 4; ++i) cur[i] = nxt[i] = double2{0., 0.};
  bool ok = true;
  if (first) {
    // step T uses row T + shift: for the steps start - 1 (the first cell's
    // old value) .. start + 3
    ok = Await(start + 4 + shift);
    if (ok) {
      Fetch(cur, start);
      if (t == 0 && from < 0 && start - 1 + shift >= 0)
        oldA = AgentLoad(in + long((start - 1 + shift) % le) * a);
    }
  }
  double2* const mine = val + q * W + t;
  auto Decide = [&](int stage, int r) {
    const int slot = 4 * stage + (r & 3), s = wg * P + stage + ptot * r;
    const unsigned long long bits = sd[slot];
    sd[slot] = 0ull;
    const double diff = __longlong_as_double((long long)bits);
    if (!ch.tail && s <= limit && (!(diff > tol) || s == limit)) {
      if (s < __hip_atomic_fetch_min(stop, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        rec[s % ptot] = bits;
    }
  };
  // (steps are counted in 32 bits: a solve that gets to kChainMaxStep has not
  // met the stop rule, and `stop` stays kNever)
  const int end = int(min(ChainDoneStep(limit, P, ptot, span, a, b) + 4, long(kChainMaxStep)));
  int lrow = start % le, done_steps = start;
  for (int T = start;; T += 4) {
    // ---- the next group's input
    if (first && ok) {
      ok = Await(T + 8 + shift);
      if (ok) Fetch(nxt, T + 4);
      if (wait) {
        ahead = AgentLoad(progress + 16 * src);
        if (tid == 0) ahead_stop = AgentLoad(stop);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int nrow = row + 1 == b ? 0 : row + 1;
      Load(c[(i + 1) & 3], nrow);
      const int tm1 = tm + 1 == b ? 0 : tm + 1;
      if (live) {
        const SorRow &ca = c[i & 3], &cb = c[(i + 2) & 3];
        const double2* const pv = mine + ((i & 1) ^ 1) * Q * W;
        const double2 west = pv[0];
        const double eastA = pv[2].x;
        double nextA, crossA;
        if (first) {
          const int u = T + i - t;  // (from >= 0 only where start is 0)
          nextA = u + 1 >= from ? cur[i].x : 0.;
          crossA = (u >= from && t < a - 1) ? cur[i].y : 0.;
        } else {
          nextA = pv[1 - W].y;
          crossA = pv[2 - W].y;
        }
        // the last line's ends: decide the sweeps that finished a step ago
        if (t == a - 1 && rd > 0) {
          if (tm == ez) Decide(2 * q, rd - 1);
          if (tm == (ez + 2 >= b ? ez + 2 - b : ez + 2)) Decide(2 * q + 1, rd - 1);
        }
        const bool m0 = tm == ez, mend = tm1 == ez;
        const int tb1 = tm >= 1 ? tm - 1 : tm - 1 + b, tb2 = tm >= 2 ? tm - 2 : tm - 2 + b;
        const bool mb1 = tb1 == ez, mb2 = tb2 == ez;
        const double xA = SorCell<TR>(ca, m0 ? 0. : ownA, west.x, crossA, mend ? 0. : nextA, oldA,
                                      omega, dA);
        const double xB = SorCell<TR>(cb, mb2 ? 0. : ownB, west.y, eastA, mb1 ? 0. : h1, h2, omega,
                                      dB);
        mine[(i & 1) * Q * W + 1] = double2{xA, xB};
        if (last && wait) {  // (the tail reads the logs)
          int r = lrow + i;
          if (r >= le) r -= le;
          __hip_atomic_store(mylog + long(r) * a + t, xB, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
        }
        if (limA >= 0 && rd == limA) out[long(row) * a + t] = xA;
        if (limB >= 0) {
          const int rdB = (m0 || mb1) ? rd - 1 : rd;  // (m == 0, 1: still the round before)
          if (rdB == limB) out[long(pr2) * a + t] = xB;
        }
        if (mend) {
          if (rd >= 0)
            atomicMax(&sd[8 * q + (rd & 3)], (unsigned long long)__double_as_longlong(dA));
          dA = 0.;
          ++rd;
        }
        if (mb1) {
          if (rd > 0)
            atomicMax(&sd[8 * q + 4 + ((rd - 1) & 3)],
                      (unsigned long long)__double_as_longlong(dB));
          dB = 0.;
        }
        oldA = nextA;
        h2 = h1;
        h1 = xA;
        ownA = xA;
        ownB = xB;
      }
      pr2 = pr1;
      pr1 = row;
      row = nrow;
      tm = tm1;
      if (i == 3) {
        // a wave with the last stage issues 16 vector memory operations per
        // group, of which at most 12 may be outstanding here: its log stores
        // before this group are complete
        asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
        if (tid == 0) lstop = ok ? ahead_stop : -1;
      }
      ChainBarrier();
    }
    lrow += 4;
    if (lrow >= le) lrow -= le;
    done_steps = T + 4;
    if (tid == 0 && wait)
      __hip_atomic_store(progress + 16 * wg, T, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (first) {
#pragma unroll
      for (int i = 0; i < 4; ++i) cur[i] = nxt[i];
    }
    const int s = lstop;
    const int stop_at =
        s == kNever ? end : s < 0 ? 0 : min(end, int(ChainDoneStep(s, P, ptot, span, a, b)) + 4);
    ChainBarrier();  // lstop is not written again before every thread read it
    if (T >= stop_at) break;
  }
  // what the last two groups wrote: the others need no more than this for the
  // sweeps up to the stop (and see the stop if they want more)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0 && wait)
    __hip_atomic_store(progress + 16 * wg, done_steps, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

long SorWorkspace(int nx, int ny, int limit) { return SorWorkspaceDoubles(nx, ny, limit); }

bool LaunchSor(hipStream_t st, int nx, int ny, Rows a, const double* k, double* x, double tol,
               int limit, double omega, unsigned long long* info, double* ws, long ws_doubles,
               bool wait, int polls) {
  const SorPlan p = PlanSor(nx, ny, limit, ws ? ws_doubles : 0);
  const SorPlan c = PlanChain(nx, ny, limit, ws ? ws_doubles : 0);
  const bool many = wait && UseChain(p, c);
  if (!p.ok && !many) {
    LaunchGsWavefront(st, nx, ny, a, k, x, tol, limit, omega, info);
    return false;
  }
  const long n = long(nx) * ny;
  const int tr = p.tr ? 1 : 0;
  double2* oc = reinterpret_cast<double2*>(ws + (many ? kChainHeader : kSorHeader));
  double2 *xn = oc + n, *ck = xn + n;
  double* ring = reinterpret_cast<double*>(ck + n);
  const unsigned grid = unsigned((n + 255) / 256);
  // the first sweeps' values, if there is room: behind the ring, or the chain's
  // result
  const bool first = many ? c.first : p.first;
  double* const xf = first ? ring + (many ? 1 : 2 * p.Q * p.rounds) * n : nullptr;
  KSorPack<<<grid, 256, 0, st>>>(nx, ny, a, k, tr, oc, xn, ck, xf, ws,
                                 many ? kChainRec : kSorHeader);
  if (many) {
    SorChain ch{c.a, c.b, (c.a + 63) / 64 * 64, c.Q, c.G, c.span, c.le, limit, 0,
                polls < 0 ? kSpin : polls};
    const int threads = c.Q * ch.ap;
    const size_t lds = size_t(2) * c.Q * (c.a + 2) * sizeof(double2) + size_t(8) * c.Q * 8;
    double *out = ring, *logs = out + (first ? 2 : 1) * n;
    for (int tail = 0; tail < 2; ++tail) {
      ch.tail = tail;
      const unsigned g = tail ? 1u : unsigned(c.G + first);
      auto launch = [&](auto kernel) {
        kernel<<<g, threads, lds, st>>>(ch, oc, xn, ck, ws, logs, out, xf, tol, omega, info);
      };
      if (threads > 512)
        launch(tr ? KSorChain<true, 1024> : KSorChain<false, 1024>);
      else
        launch(tr ? KSorChain<true, 512> : KSorChain<false, 512>);
    }
    KSorUnpack<<<grid, 256, 0, st>>>(nx, ny, tr, out, ws, x);
    return true;
  }
  double* const out = n <= kCopyOutCells ? x : nullptr;
  const int threads = (p.Q * p.a + 63) / 64 * 64;
  const size_t lds = size_t(2) * p.Q * (p.a + 2) * sizeof(double2) +
                     size_t(p.rounds) * 2 * p.Q * 8 + 16;
  if (p.tr)
    KSorPipe<true><<<1 + first, threads, lds, st>>>(p.a, p.b, p.Q, p.rounds, oc, xn, ck, ring, xf,
                                                    tol, limit, omega, ws, info, out);
  else
    KSorPipe<false><<<1 + first, threads, lds, st>>>(p.a, p.b, p.Q, p.rounds, oc, xn, ck, ring, xf,
                                                     tol, limit, omega, ws, info, out);
  if (!out) KSorUnpack<<<grid, 256, 0, st>>>(nx, ny, tr, ring, ws, x);
  return false;
}

}  // namespace hg
