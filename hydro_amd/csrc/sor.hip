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
// cells, 52 of them FP64), with 2 Q a <= 2048 cells per step on one CU.
// Per sweep, against the sweep-at-a-time kernel (101 and 701 sweeps): 64 x 64
// 3.6 against 34.6 us, 256 x 128 15.3 against 177 us, 333 x 217 43 against
// 534 us, 37 x 900 27 against 274 us.  1024 threads beat 512 and 256 (256 x
// 128: 15.3, 19.7, 30.9 us).
#include <algorithm>

#include "kernels.h"

namespace hg {

namespace {

constexpr int kSorThreads = 1024;
constexpr int kSorMaxQ = 32;
constexpr int kSorHeader = 32;  // doubles before the arrays: [0] the result's ring slot

struct SorPlan {
  bool ok = false;
  bool tr = false;   // threads along y (the short side), marching along x
  int a = 0, b = 0;  // short and long side
  int Q = 0, rounds = 0;
  long doubles = 0;
};

// The ring holds `rounds` rounds of P = 2 Q sweeps: sweep s's buffer is
// written again by sweep s + rounds P, which starts (rounds - 1) b steps after
// the round that follows s begins, and s is decided a + b + 5 steps after its
// own start at the latest.
SorPlan PlanSor(int nx, int ny, int limit, long max_doubles) {
  SorPlan p;
  p.tr = ny < nx;
  p.a = std::min(nx, ny);
  p.b = std::max(nx, ny);
  const long n = long(nx) * ny;
  p.rounds = p.a + 7 <= p.b ? 2 : 3;
  int q = std::min(std::min(kSorThreads / std::max(p.a, 1), (p.b - 4) / 4), kSorMaxQ);
  q = std::min(q, limit / 2 + 1);  // sweeps 0 .. limit
  for (; q >= 1; --q) {
    p.doubles = kSorHeader + (6 + 2L * q * p.rounds) * n;
    // (32-bit byte offsets in the kernel)
    if (p.doubles <= max_doubles && p.doubles < (1L << 29)) {
      p.Q = q;
      p.ok = true;
      break;
    }
  }
  return p;
}

// Barrier between steps.  It orders the LDS exchange and leaves the loads in
// flight; of the global stores it waits for those of two steps before and
// earlier (a step issues at most 3 + 2 loads and 2 stores per wave, vector
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

// One cell's row: own (the neighbour before it on its line: new value),
// cross (the neighbour on the line before: new), xold (on the line after:
// old), nold (the next cell of its line: old), diagonal, constant.
struct SorRow {
  double2 oc, xn, ck;
};

// Rows into the skewed order, zero where the neighbour is outside the grid.
__global__ void __launch_bounds__(256)
KSorPack(int nx, int ny, Rows r, const double* __restrict__ k, int tr, double2* __restrict__ oc,
         double2* __restrict__ xn, double2* __restrict__ ck) {
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
}

__global__ void __launch_bounds__(256)
KSorUnpack(int nx, int ny, int tr, const double* __restrict__ ring,
           const double* __restrict__ head, double* __restrict__ x) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= nx * ny) return;
  const int a = tr ? ny : nx, b = tr ? nx : ny;
  const int i = c % nx, j = c / nx;
  const int t = tr ? j : i, m = tr ? i : j;
  const int row = t + m >= b ? t + m - b : t + m;
  const long slot = reinterpret_cast<const long long*>(head)[0];
  x[c] = ring[slot * nx * ny + long(row) * a + t];
}

template <bool TR>
__global__ void __launch_bounds__(kSorThreads)
KSorPipe(int a, int b, int Q, int rounds, const double2* __restrict__ oc,
         const double2* __restrict__ xn, const double2* __restrict__ ck, double* ring, double tol,
         int limit, double omega, double* head, unsigned long long* __restrict__ info) {
  // [2 step parities][Q][a + 2] values (first, second stage) with a zero
  // pad either side, then the sweeps' maxima
  extern __shared__ double2 lds2[];
  __shared__ int flag;  // 1 + the group of four steps in which a sweep ended the solve
  const int W = a + 2;
  double2* const val = lds2;
  unsigned long long* const sd = reinterpret_cast<unsigned long long*>(lds2 + 2 * Q * W);
  const int P = 2 * Q, R = rounds * P;
  const int tid = threadIdx.x;
  for (int z = tid; z < 2 * Q * W; z += blockDim.x) val[z] = double2{0., 0.};
  for (int z = tid; z < R; z += blockDim.x) sd[z] = 0ull;
  if (tid == 0) flag = 0;
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
  int group = 0;
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
      reinterpret_cast<long long*>(head)[0] = idx;
      flag = group + 1;
    }
  };
  auto Cell = [&](const SorRow& r, double own, double cross, double xold, double nold, double old,
                  double& dmax) {
    const double po = r.oc.x * own, pc = r.oc.y * cross;  // new: south and west
    const double px = r.xn.x * xold, pn = r.xn.y * nold;  // old: east and north
    double sum = po + pc;
    sum += TR ? pn : px;  // east
    sum += TR ? px : pn;  // north
    const double value = -(r.ck.y + sum) / r.ck.x;
    const double corr = value - old;
    dmax = fmax(dmax, fabs(corr));
    return old + corr * omega;
  };
  for (;; ++group) {
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
        const double xA = Cell(ca, m != 0 ? ownA : 0., west.x, crossA, m1 != 0 ? nextA : 0., oldA,
                               dA);
        const double xB = Cell(cb, m != 2 ? ownB : 0., west.y, eastA, m != 1 ? h1 : 0., h2, dB);
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
}

}  // namespace

long SorWorkspace(int nx, int ny) {
  const SorPlan p = PlanSor(nx, ny, 1 << 30, 1L << 60);
  return p.ok ? p.doubles : 0;
}

void LaunchSor(hipStream_t st, int nx, int ny, Rows a, const double* k, double* x, double tol,
               int limit, double omega, unsigned long long* info, double* ws, long ws_doubles) {
  const SorPlan p = PlanSor(nx, ny, limit, ws ? ws_doubles : 0);
  if (!p.ok) {
    LaunchGsWavefront(st, nx, ny, a, k, x, tol, limit, omega, info);
    return;
  }
  const long n = long(nx) * ny;
  double2* oc = reinterpret_cast<double2*>(ws + kSorHeader);
  double2 *xn = oc + n, *ck = xn + n;
  double* ring = reinterpret_cast<double*>(ck + n);
  const unsigned grid = unsigned((n + 255) / 256);
  KSorPack<<<grid, 256, 0, st>>>(nx, ny, a, k, p.tr ? 1 : 0, oc, xn, ck);
  const int threads = (p.Q * p.a + 63) / 64 * 64;
  const size_t lds = size_t(2) * p.Q * (p.a + 2) * sizeof(double2) +
                     size_t(p.rounds) * 2 * p.Q * 8 + 16;
  if (p.tr)
    KSorPipe<true><<<1, threads, lds, st>>>(p.a, p.b, p.Q, p.rounds, oc, xn, ck, ring, tol, limit,
                                            omega, ws, info);
  else
    KSorPipe<false><<<1, threads, lds, st>>>(p.a, p.b, p.Q, p.rounds, oc, xn, ck, ring, tol,
                                             limit, omega, ws, info);
  KSorUnpack<<<grid, 256, 0, st>>>(nx, ny, p.tr ? 1 : 0, ring, ws, x);
}

}  // namespace hg
