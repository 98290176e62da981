// sor_plan.h -- how an exact-order SOR solve (sor.hip) is split over threads and
// workgroups, and the chain's step numbers.  Plain C++, also for host programs.
#pragma once

#include <algorithm>

#ifdef __HIPCC__
#define HG_HOST_DEVICE __host__ __device__
#else
#define HG_HOST_DEVICE
#endif

namespace hg {

constexpr int kSorThreads = 1024;
constexpr int kSorMaxQ = 32;
constexpr int kSorHeader = 32;  // doubles before the arrays: [0] kNever, [1] the result's slot
constexpr int kFirstSweeps = 2;  // of FirstSweeps
constexpr int kEndedFirst = -2;
constexpr long kCopyOutCells = 4096;

// (several workgroups, below)
constexpr int kLag = 20;
constexpr int kSpin = 1 << 20;
constexpr int kNever = 0x7fffffff;

constexpr int kSorMaxG = 64, kSorMaxStages = 1024;
// Bounds of the workspace, in doubles: 512 MB, or for a ring of two sweeps at any
// size (about what a solve's own arrays take); 32 MB for the ring that only a
// chain that gave up would use.
constexpr long kSorMaxDoubles = 1L << 26, kRetryMaxDoubles = 1L << 22;
// Workspace header, in doubles: the smallest sweep that ended the solve
// (int `stop`; -1: gave up, kEndedFirst), the result's slot (0 the chain's, 1 the
// first sweeps'), then a 64-byte line of progress per workgroup, then the max
// |corr| of the sweep each stage last found to end it.
constexpr int kChainProgress = 8, kChainRec = kChainProgress + 8 * kSorMaxG;
constexpr int kChainHeader = kChainRec + kSorMaxStages;

struct SorChain {
  int a, b, ap;           // short and long side, line padded to waves
  int Q, G, span, le;     // thread groups per workgroup, workgroups, log rows
  int limit, tail;
  int spin;               // bound on a wait's polls
};

struct SorPlan {
  bool ok = false;
  bool tr = false;   // threads along y (the short side), marching along x
  int a = 0, b = 0;  // short and long side
  int Q = 0, rounds = 0;
  int G = 1, span = 0, le = 0;  // several workgroups (G > 1): see KSorChain
  bool first = false;  // room for FirstSweeps, too (not at the cost of sweeps in flight)
  long doubles = 0;
};

// The ring holds `rounds` rounds of P = 2 Q sweeps: sweep s's buffer is
// written again by sweep s + rounds P, which starts (rounds - 1) b steps after
// the round that follows s begins, and s is decided a + b + 5 steps after its
// own start at the latest.
inline SorPlan PlanSor(int nx, int ny, int limit, long max_doubles) {
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
      p.first = p.doubles + n <= max_doubles;
      p.doubles += p.first ? n : 0;
      p.Q = q;
      p.ok = true;
      break;
    }
  }
  return p;
}

// The several-workgroup plan: 512 threads (1024 where a line needs them),
// as many workgroups as keep kLag steps between them.  A log keeps what the
// tail may read: a + b rows of a line, up to b + span steps after its end (a
// workgroup is at most the sum of the lags, under b, ahead of another).
inline SorPlan PlanChain(int nx, int ny, int limit, long max_doubles) {
  SorPlan p;
  p.tr = ny < nx;
  p.a = std::min(nx, ny);
  p.b = std::max(nx, ny);
  const long n = long(nx) * ny;
  const int ap = (p.a + 63) / 64 * 64;
  if (ap > kSorThreads) return p;
  p.Q = std::max(512 / ap, 1);
  const int P = 2 * p.Q;
  int g = std::min(std::min(p.b / (2 * P + kLag), kSorMaxG), kSorMaxStages / P);
  g = std::min(g, limit / P + 1);
  for (; g >= 2; --g) {
    p.span = p.b / g;
    p.le = p.a + 2 * p.b + p.span + 64;
    p.doubles = kChainHeader + 7 * n + long(g) * p.le * p.a;
    if (p.doubles <= std::min(max_doubles, kSorMaxDoubles)) {
      p.first = p.doubles + n <= max_doubles;
      p.doubles += p.first ? n : 0;
      p.G = g;
      p.ok = true;
      break;
    }
  }
  return p;
}

// Virtual step of the chain by which sweep s is decided and every earlier one
// too (P sweeps per workgroup, ptot per round).  In 64 bits: a limit of 2^31 - 1
// sweeps, which asks for a stop by the tolerance alone, is past 2^31 steps.
HG_HOST_DEVICE inline long ChainDoneStep(int s, int P, int ptot, int span, int a, int b) {
  const int st = s % ptot;
  return long(st / P) * span + 2 * (st % P) + long(s / ptot) * b + a + b;
}
// The kernel counts steps in 32 bits; a solve that gets to this one without a
// stop (after minutes) is run again by KSorPipe, which counts sweeps only.
constexpr int kChainMaxStep = 1 << 30;

// Several workgroups where they hold more sweeps than one does.  Measured per
// sweep at 701 sweeps, one | several (stages held): 64x256 7.6 | 3.2 us (32 | 64),
// 256x128 15.3 | 3.7 (16 | 56), 333x217 40 | 6.1 (8 | 44), 512x512 130 | 11.4
// (4 | 42), 30x700 10.1 | 3.1 (64 | 208); where they do not: 16x256 2.6 | 3.4 us
// (64 | 64), 32x128 2.2 | 3.0 (62 | 32), 64x128 4.0 | 3.1 (32 | 32), as the lines
// are padded to waves.
// Nor on lines of under 16 cells, of which one workgroup holds 64 sweeps: solves
// of few sweeps, which take a chain twice as long (it repeats them), then lose
// against a sweep at a time.  3x700 at 9 | 101 sweeps 468 | 800 us by one, 1353 |
// 1257 by several, 9x1030 721 | 1419 and 1442 | 1359, 16x600 430 | 830 and 875 |
// 833; a sweep at a time 9x1030 takes 4 sweeps in 1230 us, 16x600 in 1050.
inline bool UseChain(const SorPlan& one, const SorPlan& many) {
  return many.ok && (!one.ok || (many.G * many.Q > one.Q && many.a >= 16));
}

// The workspace of a solve of at most limit + 1 sweeps.
inline long SorWorkspaceDoubles(int nx, int ny, int limit) {
  auto first = [&](SorPlan p) {
    if (p.ok && !p.first) p.doubles += long(nx) * ny;
    return p;
  };
  auto ring = [&](long cap) {
    const SorPlan p = PlanSor(nx, ny, limit, cap);
    return first(p.ok ? p : PlanSor(nx, ny, std::min(limit, 0), 1L << 60));
  };
  const SorPlan p = ring(kSorMaxDoubles), c = first(PlanChain(nx, ny, limit, kSorMaxDoubles));
  if (!UseChain(p, c)) return p.ok ? p.doubles : 0;
  const SorPlan retry = ring(std::max(c.doubles, kRetryMaxDoubles));
  return std::max(c.doubles, retry.ok ? retry.doubles : 0);
}

}  // namespace hg
