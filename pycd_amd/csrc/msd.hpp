// Windowed-origin squared displacements (PyCD/core.py:2996-3007) on gfx950,
// shared by pycd_msd and the batched form.  For one carrier's path r of P
// rows, the sums over origins
//   s[tau] = sum_{t0 < P - tau} |r(t0 + tau) - r(t0)|^2,  tau < M.
//
// One workgroup of kMsdWaves wavefronts takes a unit (one carrier's path) or
// a part of its origins.  Positions pass through LDS (x, y and z of a row
// side by side) in windows read from global memory once each.  A pass takes
// kMsdBlocks blocks of 4 kQ lags; in block b lane q of a group of kQ lanes
// owns the kMsdL consecutive lags pass0 + 4 kQ b + kMsdL q + i.  A wavefront
// holds 64 / kQ groups, which walk different origins: kQ = 64 leaves most
// lanes without a lag when M is small (100 lags: 39 lanes of 64), so kQ is
// the one that takes the fewest steps (msd_lanes).  For a block, a group walks consecutive origins t0 and keeps r(t0 + lag) of its
// lane's lags in a ring of kMsdRing registers, so a step reads the origin
// (one address for the group) and one new position, and forms kMsdL squared
// distances.  Origin t0 has work in block b only while
// t0 < P - pass0 - 4 kQ b, so the blocks of high lags have fewer origins;
// the segment's (block, origin) steps are cut into equal runs, one per group
// (a run may end one block and start the next), and the steps near the end
// of the rows, where some of a lane's lags fall past them, mask those lags.
// Rows are held with one pad row after every 4, so the rows of lanes l and
// l + 1 (4 apart) sit 15 doubles apart and the lanes of a group's LDS access
// fall on distinct banks.  Runs start at multiples of 4 rows, so within a
// run every LDS address is a base plus an immediate offset.  For the first
// pass the window holds rows [T0, T0 + S + span - 1), which contain the
// segment's S origins; later passes keep the origins in their own S rows
// ahead of the window.
//
// Bound by FP64 issue: 3 subtractions and 3 FMAs per distance, 92% of the
// SIMDs' cycles at 500 lags of 2001 rows (batched, 17.3 ms).  4096 trajectories
// of 1-64 carriers, 100 lags of up to 801 rows: 4.9 ms at kQ = 64, 3.1 ms at
// kQ = 32.
#pragma once

#include "common.hpp"

#include <cstdint>

namespace pycd {

constexpr int kMsdL = 4;               // lags per lane and block
constexpr int kMsdBlocks = 2;          // blocks per pass
constexpr int kMsdRing = 8;            // ring registers (> kMsdL)
constexpr int kMsdWin = 1024;          // path rows held in LDS
constexpr int kMsdPlane = kMsdWin + kMsdWin / 4;  // with the pad rows
constexpr int kMsdXcds = 8;
constexpr int kMsdWaves = 4;           // wavefronts per unit
constexpr int kMsdThreads = 64 * kMsdWaves;
static_assert(kMsdRing % 4 == 0, "a ring turn keeps the runs' row phase");

// Origins per segment of the pass at pass0 of M lags (a multiple of 4): a
// run reads rows below wofs + S + 4 kQ nblk + 4, inside the window.
__host__ __device__ inline int msd_segment(int kq, int64_t pass0, int64_t M) {
  const int block = kMsdL * kq;
  const int64_t span =
      M - pass0 < kMsdBlocks * block ? M - pass0 : kMsdBlocks * block;
  const int nblk = int((span + block - 1) / block);
  const int room = kMsdWin - block * nblk - 4;
  return (pass0 == 0 ? room : room / 2) & ~3;
}

// Wavefront steps of a path of P rows and M lags with groups of kq lanes: its
// (block, origin) steps over the groups, and what a block of a segment costs
// besides (its runs' first reads, the masked steps), 10, 28 and 16 steps at kq
// = 64, 32 and 16 (in proportion below 150 origins).
inline double msd_cost(int kq, int64_t P, int64_t M) {
  const int64_t block = kMsdL * kq, pass = kMsdBlocks * block;
  const double extra = kq == 64 ? 10 : kq == 32 ? 28 : 16;
  double steps = 0.0;
  for (int64_t p0 = 0; p0 < M && p0 < P; p0 += pass) {
    const int64_t S = msd_segment(kq, p0, M), n = P - p0;
    const double segments = n < 150 ? n / 150.0 : double((n + S - 1) / S);
    for (int64_t lag = p0; lag < p0 + pass && lag < M; lag += block)
      steps += extra * segments +
               (P > lag ? double(P - lag) * kq / (64 * kMsdWaves) : 0.0);
  }
  return steps;
}

// Lanes per group, 64, 32 or 16, for `n` kinds of paths: case_of(k) gives
// their rows, lags and number.  Fewest steps; the wider group on a tie (it
// needs fewer passes over the rows).  Over 211 pairs of 20 to 5001 rows and 5
// to 1500 lags, each timed with all three, the choice takes 0.4% longer than
// the best on average and 12% at most; by the lags in whole blocks alone it
// was up to 33% (401 rows, 130 lags: 64 lanes 0.21 ms, 32 0.25, 16 0.23; 64
// lags 0.19, 0.13, 0.08).
struct MsdCase {
  int64_t P, M;
  double paths;
};
template <typename F>
inline int msd_lanes(int64_t n, F&& case_of) {
  int best = 64;
  double least = 0.0;
  for (int kq = 64; kq >= 16; kq /= 2) {
    double cost = 0.0;
    for (int64_t k = 0; k < n; ++k) {
      const MsdCase c = case_of(k);
      cost += msd_cost(kq, c.P, c.M) * c.paths;
    }
    if (kq == 64 || cost < least) {
      best = kq;
      least = cost;
    }
  }
  return best;
}

// Lags of a pass.
__host__ __device__ constexpr int msd_pass(int kq) {
  return kMsdBlocks * kMsdL * kq;
}

// LDS position of window row r
__device__ inline int msd_row(int r) { return r + (r >> 2); }

// One group's run over the relative origins [ra, rb) of a block (ra a
// multiple of 4).  L: the window, window row r at L[3 msd_row(r) + k] for
// coordinate k; lo: the lane's first lag relative to the pass; hi: the
// block's last lag below the pass's span; lim: P - pass0 - T0, the relative
// origin bound; base: window row of relative origin 0's lag-0 row.  It reads
// the rows below base + rb + lo + kMsdRing and the origins below rb + 2.
// kExec: the masked steps under exec masks, which skip what no lane needs
// (one group per wavefront: 1024 x 32 paths of 2001 rows, 500 lags 6.94 -> 6.63
// ms), else by selects (four groups, some of whose lanes nearly always have
// work: 2048 x 32 of 401 rows, 60 lags 0.69 ms, 0.73 under exec masks).  Two
// groups lie between: 120 lags of the same paths 1.17 and 1.12 ms, 100 lags of
// 4096 x 16 of 801 rows 1.99 and 1.97.
template <bool kExec>
__device__ inline void msd_run(const double* L, int ra, int rb, int lo,
                               int hi, int lim, int base, double* acc) {
  constexpr int kR = kMsdRing;
  // rows are read at vb + immediate and origins at ob + immediate, both at
  // multiples of 4 rows: msd_row(4a + p) = 5a + p + (p >> 2)
  int vb = 3 * (((base + ra + lo) >> 2) * 5);
  int ob = 3 * ((ra >> 2) * 5);
  auto off = [](int p) { return 3 * (p + (p >> 2)); };
  double wx[kR], wy[kR], wz[kR], ox[2], oy[2], oz[2];
#pragma unroll
  for (int p = 0; p < kR; ++p) {
    wx[p] = L[vb + off(p)];
    wy[p] = L[vb + off(p) + 1];
    wz[p] = L[vb + off(p) + 2];
  }
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    ox[p] = L[ob + off(p)];
    oy[p] = L[ob + off(p) + 1];
    oz[p] = L[ob + off(p) + 2];
  }
  // Sums in three levels, so that no chain of roundings is long: a turn's in
  // s, those of the run in r, the runs in acc.  (One level: 2-norm error of
  // the batch's means 1e-15; 4 turns to a chain 1.4e-16; this 0.9e-16, as
  // NumPy's pairwise sums, for 2.5% of the time of one level at 500 lags.)
  double r[kMsdL], s[kMsdL];
#pragma unroll
  for (int i = 0; i < kMsdL; ++i) r[i] = 0.0;
  // below fast_end every lane's lags up to hi have rows inside the written
  // rows
  const int fast_end = min(rb, lim - hi);
  int o = ra;
  // at step j of a turn slot (p % kR) holds r(o + lo + p) for
  // p = j .. j + kR - 1 and origin slot (j % 2) holds r(o + j); after its
  // pairs the step loads position j + kR and origin j + 2 into the slots
  // that position j and origin j left (the scheduling barrier keeps those
  // loads after the pairs, so a slot keeps its registers)
  auto load = [&](int j) {
    __builtin_amdgcn_sched_barrier(0);
    wx[j] = L[vb + off(j + kR)];
    wy[j] = L[vb + off(j + kR) + 1];
    wz[j] = L[vb + off(j + kR) + 2];
    ox[j & 1] = L[ob + off(j + 2)];
    oy[j & 1] = L[ob + off(j + 2) + 1];
    oz[j & 1] = L[ob + off(j + 2) + 2];
  };
  auto turned = [&] {
    o += kR;
    vb += 3 * (kR / 4 * 5);
    ob += 3 * (kR / 4 * 5);
  };
  auto add_turn = [&] {
#pragma unroll
    for (int i = 0; i < kMsdL; ++i) r[i] += s[i];
  };
  while (o + kR <= fast_end) {
#pragma unroll
    for (int j = 0; j < kR; ++j) {
#pragma unroll
      for (int i = 0; i < kMsdL; ++i) {
        const int q = (j + i) % kR;
        const double dx = wx[q] - ox[j & 1], dy = wy[q] - oy[j & 1],
                     dz = wz[q] - oz[j & 1];
        // (a turn's first square needs no zero to be added to)
        const double x2 = j == 0 ? dx * dx : fma(dx, dx, s[i]);
        s[i] = fma(dz, dz, fma(dy, dy, x2));
      }
      load(j);
    }
    turned();
    add_turn();
  }
  // masked steps: pair i of step j counts while lo + i < lim - o - j, for
  // each pair a first part of a group's lanes
  auto masked_step = [&](int j) {
    const int c = lim - (o + j);
#pragma unroll
    for (int i = 0; i < kMsdL; ++i) {
      const int q = (j + i) % kR;
      const double dx = wx[q] - ox[j & 1], dy = wy[q] - oy[j & 1],
                   dz = wz[q] - oz[j & 1];
      if (lo + i < c) {
        if constexpr (kExec) asm volatile("");  // else selects
        s[i] = fma(dz, dz, fma(dy, dy, fma(dx, dx, s[i])));
      }
    }
    load(j);
  };
  // whole turns, then the last part of a turn
  auto zero = [&] {
#pragma unroll
    for (int i = 0; i < kMsdL; ++i) s[i] = 0.0;
  };
  while (o + kR <= rb) {
    zero();
#pragma unroll
    for (int j = 0; j < kR; ++j) masked_step(j);
    turned();
    add_turn();
  }
  zero();
#pragma unroll
  for (int j = 0; j < kR; ++j) {
    if (o + j >= rb) break;
    masked_step(j);
  }
  add_turn();
#pragma unroll
  for (int i = 0; i < kMsdL; ++i) acc[i] += r[i];
}

// Running sum with the roundings kept apart (Knuth's TwoSum).
struct ExactSum {
  double hi = 0.0, lo = 0.0;
  __device__ void add(double v) {
#pragma clang fp contract(off)
    const double t = hi + v, b = t - hi;
    lo += (hi - (t - b)) + (v - b);
    hi = t;
  }
  __device__ double value() const {
    // (an infinite or NaN sum leaves NaN in lo)
    const double v = hi + lo;
    return v == v ? v : hi;
  }
};

// The sums of a path of P rows (w3 doubles apart, from src) for the lags
// [lag0, M), lag0 a multiple of a pass's, over the origins of segments part,
// part + parts, ...; those of one pass where `one`: put(tau, sum) for every
// such lag, each wavefront group's sums added in order.  A segment is as long
// as the window allows, at most `seg` origins (a multiple of 4).
template <int kQ, typename Put>
__device__ __forceinline__ void msd_unit(
    const __attribute__((address_space(1))) double* src, int64_t w3,
    int64_t P, int64_t lag0, int64_t M, bool one, int part, int parts, int seg,
    Put&& put) {
  constexpr int kBlock = kMsdL * kQ;            // lags per block
  constexpr int kPass = msd_pass(kQ);           // lags per pass
  constexpr int kRuns = kMsdWaves * (64 / kQ);  // groups
  // the window; after a pass its space takes the groups' lag sums
  __shared__ double L[3 * kMsdPlane];
  static_assert(kRuns * kPass <= 3 * kMsdPlane, "lag sums fit");
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & (kQ - 1);
  const int run = wave * (64 / kQ) + (tid & 63) / kQ;
  const int64_t lag1 = one ? min<int64_t>(lag0 + kPass, M) : M;
  for (int64_t pass0 = lag0; pass0 < lag1; pass0 += kPass) {
    const int span = int(min<int64_t>(kPass, M - pass0));
    double acc[kMsdBlocks][kMsdL];
#pragma unroll
    for (int b = 0; b < kMsdBlocks; ++b)
#pragma unroll
      for (int i = 0; i < kMsdL; ++i) acc[b][i] = 0.0;
    const bool first = pass0 == 0;
    const int nblk = (span + kBlock - 1) / kBlock;
    // origins t0 < P - pass0 have a lag of this pass inside the rows
    const int64_t t_end = P - pass0;
    const int S = min(msd_segment(kQ, pass0, M), seg);
    const int wofs = first ? 0 : S;  // window row of path row T0 + pass0
    for (int64_t T0 = int64_t(part) * S; T0 < t_end; T0 += int64_t(parts) * S) {
      const int64_t T1 = min<int64_t>(T0 + S, t_end);
      // ---- stage the window (and, after the first pass, the origins)
      const int64_t wlo = T0 + pass0;
      const int nw = int(min<int64_t>(P, T1 - 1 + pass0 + span) - wlo);
      __syncthreads();
      for (int r = tid; r < nw; r += kMsdThreads) {
        const int64_t o = (wlo + r) * w3;
        const int pr = 3 * msd_row(wofs + r);
        L[pr] = src[o];
        L[pr + 1] = src[o + 1];
        L[pr + 2] = src[o + 2];
      }
      if (!first)
        for (int r = tid; r < T1 - T0; r += kMsdThreads) {
          const int64_t o = (T0 + r) * w3;
          const int pr = 3 * msd_row(r);
          L[pr] = src[o];
          L[pr + 1] = src[o + 1];
          L[pr + 2] = src[o + 2];
        }
      __syncthreads();
      // block b has the relative origins [0, n_b); the blocks' steps, each
      // count rounded up to a multiple of 4, are cut into kRuns runs
      const int lim = int(min<int64_t>(t_end - T0, int64_t(1) << 30));
      const int seg = int(T1 - T0);
      int n[kMsdBlocks], tot = 0;
#pragma unroll
      for (int b = 0; b < kMsdBlocks; ++b) {
        n[b] = b < nblk ? max(0, min(seg, lim - kBlock * b)) : 0;
        tot += (n[b] + 3) & ~3;
      }
      const int Q = ((tot + kRuns - 1) / kRuns + 3) & ~3;
      const int a = run * Q, e = min(a + Q, tot);
      int boff = 0;
#pragma unroll
      for (int b = 0; b < kMsdBlocks; ++b) {
        const int ra = max(a - boff, 0), rb = min(e - boff, n[b]);
        if (ra < rb)
          msd_run<kQ == 64>(L, ra, rb, kBlock * b + kMsdL * lane,
                  min(span, kBlock * (b + 1)) - 1, lim, wofs, acc[b]);
        boff += (n[b] + 3) & ~3;
      }
    }
    // the groups' sums of each lag added in order
    __syncthreads();
#pragma unroll
    for (int b = 0; b < kMsdBlocks; ++b)
#pragma unroll
      for (int i = 0; i < kMsdL; ++i)
        L[run * kPass + kBlock * b + kMsdL * lane + i] = acc[b][i];
    __syncthreads();
    for (int l = tid; l < span; l += kMsdThreads) {
      ExactSum v;
#pragma unroll
      for (int w = 0; w < kRuns; ++w) v.add(L[w * kPass + l]);
      put(pass0 + l, v.value());
    }
  }
}

}  // namespace pycd
