// Batched KMC: thousands of independent Run.do_kmc_steps trajectories
// (PyCD/core.py:2668-2861) of uneven supercell size and carrier count in
// one persistent launch on gfx950.
//
// Families are cell-periodic: a supercell of nx x ny x nz unit cells with
// n_unit sites each, numbered cell-major, site = ((cx ny + cy) nz + cz)
// n_unit + sub (the order of Material.generate_sites, PyCD/core.py:154-241).
// On such a lattice the pair table, the lattice potential, the site
// energies and every hop slot are invariant under cell translations, so a
// family keeps only the table rows of the n_unit sites of cell 0 and one
// hop record per (sublattice, slot):
//   A[a, b] = C[sub(a), b shifted by -cell(a)].
// The host checks that invariance on the full table and the slot tables
// before it accepts a family.  Only the order in which a site lists its
// slots may differ from cell 0's (neighbour lists are sorted by site index,
// which wraps at the supercell boundary); one word per site holds that
// permutation (3 bits per slot), so every site keeps the slot order, and
// with it the process order of the selection, that its own table gives.
// The compact rows and the hop differences (0.6 + 2.4 MB for an 8x8x8
// corundum supercell against 302 MB for the full table) stay in the L2 of
// the XCDs the family's trajectories are dealt to, so the per-hop gathers
// are cache hits rather than HBM round trips.  Sites are carried packed:
// cx | cz << 8 | cy << 16 | sub << 24.
//
// Scheduling: one wavefront (64 lanes, one workgroup) owns one trajectory at
// a time and takes the next from a global atomic queue when it finishes, in
// the order given by the host (longest expected work first).  The queue has
// an exit condition every wave reaches (index >= n_traj), so the grid drains.
//
// Per-hop algebra is the plain path's (q.A[x,:] = phi_L[x] + psi[x]), but
// psi is maintained incrementally: when carrier m hops s -> n, every slot
// value changes by q (A[n, x] - A[s, x]), one gather per slot from the
// family's hop differences (two table gathers without them), and carrier
// m's new slots are summed from scratch (n_c gathers each); every `refresh`
// hops all of psi is recomputed from the table to bound the rounding.
//
// A lane holds its processes' targets, psi and table indexes and one
// carrier's site row in registers, so that a hop goes through LDS only for
// the psi of the processes' carrier sites and their rate inputs; the
// selected process is read lane to lane.  The mover's new slots are summed
// by rows of 16 lanes, a lane taking every 16th carrier, which leaves each
// sum in the row that a lane permute hands to its process.  What bounds it:
// alone on a SIMD, the latencies of a hop (LDS, scan, one round of gathers,
// row sums); four to a SIMD, the issue of its ~350 vector instructions
// and the ~170 cache lines that its gathers touch, about one per cycle of a
// CU's vector cache.
// With sites, psi and process records in LDS instead (442 vector, 244
// scalar, 44 LDS instructions, now 351, 106, 21) a hop took 2.26 us alone
// and 3.09 among four at up to 16 carriers; now 1.10 and 2.0.  (The checks
// between hops behind one counter, and the entries of several carriers in
// flight where psi is formed anew, are 0.08 of that; FP64 rates, which form
// it every 64 hops, 1.86 -> 1.74 at two wavefronts a SIMD.)  The loop is
// instantiated per processes-per-lane count: with one instance for up to 4
// the large trajectories' register spills made 4096 mixed trajectories 8%
// slower.
//
// Random numbers: each trajectory carries its CPython MT19937 state (624
// words + position) in LDS and draws 4 words per hop exactly like
// random.random() (u1 selects, u2 advances the clock), so a batched
// trajectory consumes the same stream as the plain path would.
//
// Rates: FP64 (bit-faithful mode) or FP32 (throughput mode); the prefix
// sum of k / k_tot, the selection and the clock are FP64 in both.
#include "common.hpp"
#include "msd.hpp"
#include "mt19937.hpp"
#include "packed_sites.hpp"
#include "wave.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace pycd {

struct SubRec {       // hop slot j of sublattice s
  uint32_t tgt;       // packed cell offset (each in [0, n)) | target sub << 24
  int32_t pad0;
  double lam;         // lambda (Hartree)
  double vab;         // V_ab (Hartree)
  double tself;       // A[s, s] - A[s, n]
  double dphi;        // q_L . (A[n, :] - A[s, :])
  double dE;          // E[n] - E[s]
  double vec[3];      // hop vector (bohr)
};

struct FamDev {
  const double* C64;      // n_unit x N: table rows of the sites of cell 0
  const float* C32;
  const SubRec* subs;     // n_unit x z
  const uint32_t* perm;   // N: slot j of the site is slot
                          //    (perm >> 3 j) & 7 of its sublattice
  const double* phiL;     // n_unit
  // n_unit z x N or NULL: row s z + j holds A[n, x] - A[s, x] at the
  // column of x in s's row, n the target of slot j of sublattice s (the two
  // entries as the hop loop reads them, FP32 ones in the FP32 table mode)
  const double* D;
  int64_t N;
  int32_t nx, ny, nz, nu;
  int32_t z, pad;
  double qLAqL;
};

struct TrajDev {
  int32_t fam, nc;
  double q;           // carrier charge
  double field[3];    // au
  double kT;          // Hartree
  double dt;          // path-step width (au time)
  double ewald_neut;
  int64_t P;          // path rows
  int64_t max_hops;   // <= 0: run until the path is full
  int64_t row_off;    // offset (doubles) of this trajectory's path rows
  int64_t occ_off;    // offset of its initial occupancy
};

struct TrajOut {
  double t;
  double energy;
  int64_t hops;
  int64_t start;
  int32_t no_select;
  int32_t done;      // 1: the trajectory reached max_hops or filled its path
  int32_t started;   // 1: state arrays hold a run in progress
  int32_t simd;      // SIMD key (XCC, SE, CU, SIMD) of its last wavefront
  double busy;       // wall-clock ticks the trajectory's wavefront spent on it
};

struct BatchArgs {
  const FamDev* fams;
  const TrajDev* trajs;
  const int32_t* order;
  const int64_t* occ0;
  const uint32_t* mt0;      // n_traj x 625
  double* rows;             // all path rows
  double* drift;            // n_traj x 64 x 3 (nc <= kMaxCarriers)
  TrajOut* out;
  // work queue: `order` holds n_bins bins back to back, bin b at
  // [bin_start[b], bin_start[b + 1]); counter[b] counts bin b's pops and
  // counter[n_bins] all pops.  key_bin maps a SIMD's hardware key to the bin
  // its wavefronts start from (-1: none; NULL when n_bins is 1).
  uint32_t* counter;
  const uint32_t* bin_start;
  const int16_t* key_bin;
  int32_t n_bins;
  // wavefronts on its SIMD from which one hands its trajectory over
  int32_t hand_busy;
  // remaining hops of the wavefront in each SIMD wave slot (kSimdKeys x 16,
  // zeroed before the launch), for pacing, followed by the hand-over words
  // (see claim_mailbox); NULL: no pacing and no hand-over
  uint32_t* progress;
  // resumable state (slices): MT words, occupancy, displacement/base/drift
  uint32_t* mts;            // n_traj x 625
  uint32_t* st_occ;         // n_traj x kMaxCarriers (packed sites)
  double* st_vec;           // n_traj x 3 x (3 kMaxCarriers)
  double* st_psi;           // n_traj x kPsiStride
  int64_t slice_hops;       // <= 0: run each trajectory to its end
  int64_t refresh;          // recompute every psi from the table each
                            // `refresh` hops of a trajectory (<= 0: never)
  int32_t n_traj;
  int32_t nc_max;
  int32_t z_max;
  int32_t sub_max;          // largest n_unit z of a family the launch uses
  double nu;
};

constexpr int kMaxCarriers = 64;
constexpr int kMaxPer = 8;    // processes per lane: n_c z <= 512
constexpr int kPsiStride = kMaxCarriers * 8;  // n_c (1 + z), z <= 7
constexpr int kVecStride = 3 * 3 * kMaxCarriers;
constexpr int kMaxSubSlots = 256;  // n_unit z of a family
constexpr int kMaxCells = 255;     // cells per axis, sites per cell
constexpr double kLog2E = 1.4426950408889634;  // log2(e)

// Values every lane holds identically, moved to scalar registers.
__device__ inline int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline uint32_t uni(uint32_t v) {
  return uint32_t(__builtin_amdgcn_readfirstlane(int(v)));
}
__device__ inline double uni(double v) {
  const uint64_t b = __double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(b));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(uint32_t(b >> 32));
  return __longlong_as_double((int64_t(hi) << 32) | lo);
}



// The family's arrays are reached through pointers read from memory, which
// the compiler would treat as generic (flat) addresses; flat loads also
// count against the LDS wait counter, so every LDS wait would wait for the
// gathers as well.  These casts make them global loads.
template <typename T>
using gptr = const __attribute__((address_space(1))) T*;
template <typename T>
__device__ inline gptr<T> as_global(const T* p) {
  return (gptr<T>)p;
}
// (the host pass of this file sees plain pointers: its compiler has no
// constant address space to bind the records' copy constructors to)
#if defined(__HIP_DEVICE_COMPILE__)
template <typename T>
using cptr = const __attribute__((address_space(4))) T*;
#else
template <typename T>
using cptr = const T*;
#endif
template <typename T>
__device__ inline cptr<T> as_const(const T* p) {
  return (cptr<T>)p;
}
template <typename T>
using gmut = __attribute__((address_space(1))) T*;
template <typename T>
__device__ inline gmut<T> as_global_mut(T* p) {
  return (gmut<T>)p;
}

__device__ inline SubRec load_rec(const FamDev& f, uint32_t k) {
  const gptr<SubRec> p = as_global(f.subs) + k;
  SubRec r;
  r.tgt = p->tgt;
  r.pad0 = 0;
  r.lam = p->lam;
  r.vab = p->vab;
  r.tself = p->tself;
  r.dphi = p->dphi;
  r.dE = p->dE;
  r.vec[0] = p->vec[0];
  r.vec[1] = p->vec[1];
  r.vec[2] = p->vec[2];
  return r;
}

template <typename TT>
__device__ inline gptr<TT> crow(const FamDev& f, uint32_t sub);
template <>
__device__ inline gptr<double> crow<double>(const FamDev& f, uint32_t sub) {
  return as_global(f.C64) + int64_t(sub) * f.N;
}
template <>
__device__ inline gptr<float> crow<float>(const FamDev& f, uint32_t sub) {
  return as_global(f.C32) + int64_t(sub) * f.N;
}

// The family's compact table (n_unit rows of N entries) reached by 32-bit
// byte offsets from one base, so that every gather takes the scalar base
// and one vector offset (the family check keeps the table under 4 GiB).
template <typename TT>
struct Tab {
  gptr<char> base;
  uint32_t row_bytes;  // N sizeof(TT)
  __device__ uint32_t row(uint32_t sub) const { return sub * row_bytes; }
  __device__ TT at(uint32_t row_off, uint32_t col) const {
    return *(gptr<TT>)(base + (row_off + col * uint32_t(sizeof(TT))));
  }
};
template <typename TT>
__device__ inline Tab<TT> tab_of(const FamDev& f) {
  Tab<TT> t;
  t.base = (gptr<char>)crow<TT>(f, 0);
  t.row_bytes = uint32_t(f.N) * uint32_t(sizeof(TT));
  return t;
}

// A[a, b] for packed sites a, b.
template <typename TT>
__device__ inline double pair_entry(const Tab<TT>& t, const GeoPk& p,
                                    uint32_t a, uint32_t b) {
  return double(t.at(t.row(a >> 24), rel_col(a, b, p)));
}

// sum_c q A[x, occ[c]] of a lane's kN rows x, over the carriers in order;
// the entries of 4 carriers (2 from 4 rows on) are loaded before the first
// is used.
template <typename TT, int kN>
__device__ __forceinline__ void psi_from_table(const Tab<TT>& t,
                                               const GeoPk& gp, double q,
                                               int nc,
                                               const uint32_t (&x)[kN],
                                               const uint32_t* occ,
                                               double (&acc)[kN]) {
  constexpr int kU = kN < 4 ? 4 : 2;
#pragma unroll
  for (int i = 0; i < kN; ++i) acc[i] = 0.0;
  int c2 = 0;
#pragma unroll 1
  for (; c2 + kU <= nc; c2 += kU) {
    TT v[kN][kU];
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const RowKey key = row_key(x[i], gp);
      const uint32_t row = t.row(key.sub);
#pragma unroll
      for (int u = 0; u < kU; ++u)
        v[i][u] = t.at(row, rel_col(key, occ[c2 + u], gp));
    }
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int i = 0; i < kN; ++i) acc[i] = fma(q, double(v[i][u]), acc[i]);
  }
#pragma unroll 1
  for (; c2 < nc; ++c2)
#pragma unroll
    for (int i = 0; i < kN; ++i)
      acc[i] = fma(q, pair_entry<TT>(t, gp, x[i], occ[c2]), acc[i]);
}

// Per (sublattice, slot) of the trajectory's family: the static part of a
// hop's dG0 and its rate inputs for the trajectory's charge and field, and
// the hop vector and target.  FP32 rates: 2 q (dphi + q tself) + dE, lambda,
// 1 / (4 lambda), V_ab + field shift; FP64 rates: the six terms as the
// reference adds them.
struct alignas(16) PTabF32 {
  double g0s;
  float lam, i4l, vs;
  uint32_t tgt;       // the hop record's packed target offset
  double vec[3];
};
struct PTabF64 {
  double dphi, tq, dE, lam, vab, shift;
  double vec[3];
  uint32_t tgt, pad;
};
template <bool kF32Rate>
using PTab = typename std::conditional<kF32Rate, PTabF32, PTabF64>::type;

// The part of an entry that a rate takes.
struct RateF32 {
  double g0s;
  float lam, i4l, vs;
  __device__ RateF32() = default;
  __device__ explicit RateF32(const PTabF32& p)
      : g0s(p.g0s), lam(p.lam), i4l(p.i4l), vs(p.vs) {}
};
struct RateF64 {
  double dphi, tq, dE, lam, vab, shift;
  __device__ RateF64() = default;
  __device__ explicit RateF64(const PTabF64& p)
      : dphi(p.dphi), tq(p.tq), dE(p.dE), lam(p.lam), vab(p.vab),
        shift(p.shift) {}
};
template <bool kF32Rate>
using Rate = typename std::conditional<kF32Rate, RateF32, RateF64>::type;

// Shared-memory layout of one wavefront:
//   mt     624 words (2560 B)        MT19937 block
//   psis   64 doubles                potential at each carrier's site
//   dsp    64 x 3 doubles            displacements since the last path row
//   drf    64 x 3 doubles            drifts
//   occ    64 words                  packed carrier sites (at the start and
//                                    when psi is formed anew)
//   ptab   sub_max PTab entries      per (sublattice, slot), see PTab
__host__ __device__ inline size_t batch_smem_bytes(bool f32rate, int sub_max) {
  const size_t pt = f32rate ? sizeof(PTabF32) : sizeof(PTabF64);
  return 2560 + (7 * 8 + 4) * size_t(kMaxCarriers) + pt * size_t(sub_max);
}

template <bool kF32Rate>
__device__ inline void fill_ptab(PTab<kF32Rate>& e, const SubRec& rec,
                                 double q, const double* field,
                                 bool field_on) {
  const double tq = q * rec.tself;
  const double shift =
      field_on ? 0.5 * (field[0] * rec.vec[0] + field[1] * rec.vec[1] +
                        field[2] * rec.vec[2])
               : 0.0;
  if constexpr (kF32Rate) {
    e.g0s = 2 * q * (rec.dphi + tq) + rec.dE;
    e.lam = float(rec.lam);
    e.i4l = float(0.25 / rec.lam);
    e.vs = float(rec.vab) + float(shift);
  } else {
    e.pad = 0;
    e.dphi = rec.dphi;
    e.tq = tq;
    e.dE = rec.dE;
    e.lam = rec.lam;
    e.vab = rec.vab;
    e.shift = shift;
  }
  e.vec[0] = rec.vec[0];
  e.vec[1] = rec.vec[1];
  e.vec[2] = rec.vec[2];
  e.tgt = rec.tgt;
}

// kPer: processes per lane (n_c z <= 64 kPer); kZp: slots per carrier
// (z + 1 <= kZp).  Instantiated for the batch's maxima so that the per-lane
// arrays stay small and several wavefronts fit per SIMD.
// Where this wavefront runs: XCC << 10 | SE << 7 | SH << 6 | CU << 2 | SIMD
// (13 bits), from the XCC_ID and HW_ID hardware registers.
__device__ inline uint32_t simd_key() {
  // s_getreg operand: (bits - 1) << 11 | offset << 6 | register id
  const uint32_t hw = __builtin_amdgcn_s_getreg((31 << 11) | 4);   // HW_ID
  const uint32_t xcc = __builtin_amdgcn_s_getreg((15 << 11) | 20); // XCC_ID
  const uint32_t simd = (hw >> 4) & 3u, cu = (hw >> 8) & 15u,
                 sh = (hw >> 12) & 1u, se = (hw >> 13) & 7u;
  return ((xcc & 7u) << 10) | (se << 7) | (sh << 6) | (cu << 2) | simd;
}
constexpr int kSimdKeys = 1 << 13;

// simd_key() << 4 | the wavefront's slot in its SIMD (HW_ID bits 3:0).
__device__ inline uint32_t wave_slot() {
  return (simd_key() << 4) | (__builtin_amdgcn_s_getreg((3 << 11) | 4) & 15u);
}

// Wavefronts sharing a SIMD pace each other.  Each publishes the hops it
// has left and takes a priority by rank among its SIMD's wavefronts, most
// hops left highest, so that the SIMD's trajectories advance together and
// end together; left alone, the SIMD favours its older wavefronts, whose
// trajectories end first while the rest finish on a half-idle SIMD.
__device__ inline int pace(uint32_t* prog, uint32_t slot, uint32_t left,
                            int lane) {
  if (lane == 0)
    __hip_atomic_store(prog + slot, left, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  const uint32_t base = slot & ~15u, me = slot & 15u;
  uint32_t v = 0;
  if (lane < 16)
    v = __hip_atomic_load(prog + base + lane, __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_AGENT);
  const bool before = lane < 16 && uint32_t(lane) != me &&
                      (v > left || (v == left && uint32_t(lane) < me));
  const int rank = __popcll(__ballot(before));
  if (rank == 0)
    __builtin_amdgcn_s_setprio(3);
  else if (rank == 1)
    __builtin_amdgcn_s_setprio(2);
  else if (rank == 2)
    __builtin_amdgcn_s_setprio(1);
  else
    __builtin_amdgcn_s_setprio(0);
  return __popcll(__ballot(v != 0u));
}

// Index into `order` of this wavefront's next trajectory, or n_traj once
// the queue is empty (lane 0 only).  Pops from `bin` first, then moves on
// to the next bins; stops scanning as soon as every trajectory is taken.
__device__ inline uint32_t pop_ticket(const BatchArgs& a, int& bin) {
  uint32_t* taken = a.counter + a.n_bins;
  for (int k = 0; k < a.n_bins; ++k) {
    const uint32_t lo = a.bin_start[bin], n = a.bin_start[bin + 1] - lo;
    if (n > 0 &&
        __hip_atomic_load(a.counter + bin, __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_AGENT) < n) {
      const uint32_t t = atomicAdd(a.counter + bin, 1u);
      if (t < n) {
        atomicAdd(taken, 1u);
        return lo + t;
      }
    }
    if (__hip_atomic_load(taken, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >=
        uint32_t(a.n_traj))
      break;
    bin = bin + 1 == a.n_bins ? 0 : bin + 1;
  }
  return uint32_t(a.n_traj);
}

// Hand-over of running trajectories to idle wavefronts (batch launches with
// SIMD bins: the words after the pacing slots).  Which trajectories fill
// their path early is not known ahead, and SIMDs of the same chip run the
// same work at speeds up to ~8% apart, so with every trajectory resident
// from the start the launch would end with the fullest and slowest SIMDs.
// Instead, a wavefront that finds the queue empty opens a mailbox and waits;
// a wavefront whose trajectory has hops to spare saves the trajectory's
// resumable state (exact, as at the end of a slice), puts its index in a
// waiting mailbox and leaves.  A hop takes 1.2 us alone on a SIMD, 2.0 among
// four (16 carriers), so with three or more wavefronts per SIMD a wavefront
// waits beside up to one busy one and hands over only from three up; with
// fewer the launch hands over from any busy SIMD to idle ones (4096 mixed
// trajectories of 4000 hops, 1-64 carriers, whole run with its MSD: 22.3 ms
// with idle SIMDs only and 2048 hops to spare, 20.8 so).  Words of `hand`:
//   [kHandLeft] trajectories not yet finished
//   [kHandTaken] mailboxes taken by donors
//   [kHandOpened] mailboxes opened
//   [kHandCap] mailboxes (0: hand-over off)
//   [kHandHdr + k] mailbox k: 0 empty, kMailClosed, or trajectory index + 1.
// The counts sit on cache lines of their own: atomics on one line, of whatever
// XCD, are carried out one after another (side by side in one line, 4096
// trajectories that fill their paths after 2 hops took 0.50 ms, now 0.25; of
// 600 hops and 2 carriers 1.36, now 1.27).
// Every wait ends: a mailbox is filled only while its donor's trajectory is
// unfinished, an empty mailbox is closed (by CAS) once none is, and a wait
// also gives up after kHandWaitTicks.  A trajectory is handed over at most
// once (a wavefront never passes on what it received), so at most
// grid + n_traj mailboxes are opened.
constexpr int kHandLeft = 0, kHandTaken = 32, kHandOpened = 64,
              kHandCap = 96, kHandHdr = 128;
constexpr uint32_t kMailClosed = 0xffffffffu;
constexpr uint32_t kHandMinHops = 256;           // hops left to be worth it
constexpr uint64_t kHandWaitTicks = 2000000000;  // 20 s at 100 MHz

__device__ inline uint32_t* hand_words(uint32_t* progress) {
  return progress + kSimdKeys * 16;
}

// Mailbox index of a waiting wavefront taken for a hand-over, or -1
// (lane 0 only).
__device__ inline int claim_mailbox(uint32_t* hand) {
  const uint32_t cap = hand[kHandCap];
  for (int attempt = 0; attempt < 4; ++attempt) {
    const uint32_t head = __hip_atomic_load(
        hand + kHandTaken, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t open =
        min(__hip_atomic_load(hand + kHandOpened, __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_AGENT),
            cap);
    if (head >= open) return -1;
    uint32_t expect = head;
    if (__hip_atomic_compare_exchange_strong(
            hand + kHandTaken, &expect, head + 1, __ATOMIC_RELAXED,
            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      return int(head);
  }
  return -1;
}

// Opens a mailbox and waits for a trajectory: its index, or -1 when none
// is left to hand over or hand-over is off (lane 0 only).
__device__ inline int wait_for_trajectory(uint32_t* hand) {
  const uint32_t cap = hand[kHandCap];
  if (cap == 0u) return -1;
  const uint32_t k = atomicAdd(hand + kHandOpened, 1u);
  if (k >= cap) return -1;
  uint32_t* box = hand + kHandHdr + k;
  const uint64_t t0 = wall_clock64();
  // Relaxed polls: an acquire here would invalidate the caches of the
  // wavefronts still running on every look; the caller takes one acquire
  // fence once a trajectory has arrived.
  for (uint32_t it = 0;; ++it) {
    const uint32_t v =
        __hip_atomic_load(box, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (v != 0u) return int(v - 1u);
    // the shared count only every 8th look, to keep the waiters off it
    if ((it & 7u) == 7u &&
        (__hip_atomic_load(hand + kHandLeft, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT) == 0u ||
         wall_clock64() - t0 > kHandWaitTicks)) {
      uint32_t expect = 0u;
      if (__hip_atomic_compare_exchange_strong(
              box, &expect, kMailClosed, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
              __HIP_MEMORY_SCOPE_AGENT))
        return -1;
      return int(expect - 1u);  // filled meanwhile
    }
    __builtin_amdgcn_s_sleep(127);
    __builtin_amdgcn_s_sleep(127);
  }
}

// Marks the hardware key of every SIMD that runs one of its wavefronts in
// `seen` (kSimdKeys bits).  Each wavefront sleeps `spin` x ~8k cycles
// after, so that a grid of several wavefronts per SIMD occupies all of
// them at once.
__global__ void __launch_bounds__(64) simd_probe(uint32_t* seen, int spin) {
  if (threadIdx.x == 0) {
    const uint32_t k = simd_key();
    atomicOr(seen + (k >> 5), 1u << (k & 31u));
  }
  for (int i = 0; i < spin; ++i) __builtin_amdgcn_s_sleep(127);
}

// f(std::integral_constant<int, kP>) for the smallest instance that holds
// `per` processes per lane: 1 to 4 (kPer = 4), or 2, 4 or 8.
template <int kPer, typename F>
__device__ __forceinline__ void with_processes(int per, F&& f) {
  if (kPer <= 4 && per == 1) {
    if constexpr (kPer <= 4) f(std::integral_constant<int, 1>{});
  } else if (per <= 2) {
    f(std::integral_constant<int, 2>{});
  } else if (kPer <= 4 && per == 3) {
    if constexpr (kPer <= 4) f(std::integral_constant<int, 3>{});
  } else if (per <= 4) {
    f(std::integral_constant<int, 4>{});
  } else if constexpr (kPer > 4) {
    f(std::integral_constant<int, kPer>{});
  }
}

// *p += v in LDS.
__device__ inline void lds_add(double* p, double v) {
  (void)__hip_atomic_fetch_add(
      (__attribute__((address_space(3))) double*)p, v, __ATOMIC_RELAXED,
      __HIP_MEMORY_SCOPE_WORKGROUP);
}

// v of lane addr / 4 (mod 64).
__device__ inline uint32_t lane_at(int addr, uint32_t v) {
  return uint32_t(__builtin_amdgcn_ds_bpermute(addr, int(v)));
}

// Wavefronts per SIMD the register allocation targets: 4 (16 per CU, every
// trajectory of a 4096-trajectory batch resident at once, in 128 VGPRs with
// only the per-trajectory set-up spilling) for FP32 rates with at most 4
// processes per lane; 2 otherwise (the FP64-rate and large instances would
// spill heavily in 128).
#ifndef PYCD_BATCH_WAVES_PER_EU
#define PYCD_BATCH_WAVES_PER_EU(f32, per) ((f32) && (per) <= 4 ? 4 : 2)
#endif
template <typename TT, bool kF32Rate, int kPer, int kZp>
__device__ __forceinline__ void kmc_batched_body(const BatchArgs& a) {
  extern __shared__ unsigned char smem_raw[];
  const int lane = threadIdx.x;
  uint32_t* mt = reinterpret_cast<uint32_t*>(smem_raw);
  double* psis = reinterpret_cast<double*>(smem_raw + 2560);
  double* dsp = psis + kMaxCarriers;
  double* drf = dsp + 3 * kMaxCarriers;
  uint32_t* occ = reinterpret_cast<uint32_t*>(drf + 3 * kMaxCarriers);
  PTab<kF32Rate>* ptab =
      reinterpret_cast<PTab<kF32Rate>*>(occ + kMaxCarriers);

  const uint32_t pslot = a.progress ? wave_slot() : 0u;
  int bin = 0;
  if (a.n_bins > 1) {
    const int b = a.key_bin[simd_key()];
    bin = uni(b >= 0 ? b : int(blockIdx.x % uint32_t(a.n_bins)));
  }
  int again = -1;  // a trajectory whose hand-over fell through
  for (;;) {
    int tr;
    bool stolen = false;  // handed over by another wavefront
    uint32_t ti = uint32_t(a.n_traj);
    if (again < 0) {
      if (lane == 0) ti = pop_ticket(a, bin);
      ti = uni(uint32_t(__shfl(int(ti), 0, 64)));
      bin = uni(__shfl(bin, 0, 64));
    }
    if (again >= 0) {
      tr = again;  // resumed from the state saved for the hand-over
      again = -1;
    } else if (ti < uint32_t(a.n_traj)) {
      tr = uni(a.order[ti]);
    } else {
      if (!a.progress) break;
      // wait for a hand-over only on a SIMD that has nearly run out of work,
      // so that a trajectory moves from a busy SIMD to an idle one
      uint32_t busy_here = 0;
      if (lane < 16)
        busy_here = __hip_atomic_load(a.progress + (pslot & ~15u) + lane,
                                      __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
      if (__popcll(__ballot(busy_here != 0u)) > max(a.hand_busy - 2, 0)) break;
      int got = -1;
      if (lane == 0) got = wait_for_trajectory(hand_words(a.progress));
      got = uni(__shfl(got, 0, 64));
      if (got < 0) break;
      // the donor's saved state, released before its mailbox write
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      tr = got;
      stolen = true;
    }
    const TrajOut o0 = a.out[tr];
    if (uni(o0.done)) {
      if (a.progress && lane == 0)
        atomicSub(hand_words(a.progress) + kHandLeft, 1u);
      continue;
    }
    const bool resume = uni(o0.started) != 0;
    const uint64_t w_start = wall_clock64();
    // The launch never writes the trajectory and family records: read
    // through the constant address space they are scalar loads, and their
    // fields (table base, row stride, sizes) live in scalar registers rather
    // than in vector registers read back with readfirstlane at every use.
    const TrajDev td = as_const(a.trajs)[tr];
    const FamDev f = as_const(a.fams)[uni(td.fam)];
    const Geo g{uni(f.nx), uni(f.ny), uni(f.nz), uni(f.nu)};
    const GeoPk gp = geo_pk(g);
    const Tab<TT> tab = tab_of<TT>(f);
    // the family's hop differences (absent: two table entries per slot row)
    Tab<double> dtab;
    dtab.base = (gptr<char>)as_global(f.D);
    dtab.row_bytes = uint32_t(f.N) * uint32_t(sizeof(double));
    const bool use_d = f.D != nullptr;
    const int nc = uni(td.nc), z = uni(f.z), zp = z + 1;
    const int nproc = nc * z;
    const int per = (nproc + 63) / 64;
    const double q = td.q;
    double* rows = a.rows + td.row_off;
    const int w = 3 * nc;
    const bool field_on =
        td.field[0] != 0.0 || td.field[1] != 0.0 || td.field[2] != 0.0;

    // resumable per-trajectory state in global memory (what changes from
    // hop to hop is held in registers while the trajectory runs)
    uint32_t* mts = a.mts + int64_t(tr) * 625;
    uint32_t* socc = a.st_occ + int64_t(tr) * kMaxCarriers;
    double* svec = a.st_vec + int64_t(tr) * kVecStride;
    const gmut<double> svec_g = as_global_mut(svec);
    const gmut<double> sdisp = svec_g;
    double* sbase = svec + 3 * kMaxCarriers;
    const gmut<double> sdrift = svec_g + 6 * kMaxCarriers;
    double* spsi = a.st_psi + int64_t(tr) * kPsiStride;

    // ---- load or start the state
    const uint32_t* m0 = resume ? mts : a.mt0 + int64_t(tr) * 625;
    for (int k = lane; k < 624; k += 64) mt[k] = m0[k];
    int mti = uni(int(m0[624]));
    for (int k = lane; k < f.nu * z; k += 64) {
      fill_ptab<kF32Rate>(ptab[k], load_rec(f, k), q, td.field, field_on);
    }
    if (!resume)
      for (int k = lane; k < w; k += 64) {
        sbase[k] = 0.0;
        rows[k] = 0.0;  // path row 0: the initial positions
      }
    // displacements since the last path row and drifts, zero past n_c
#pragma unroll
    for (int c3 = 0; c3 < 3; ++c3) {
      const int k = lane + 64 * c3;
      dsp[k] = resume && k < w ? sdisp[k] : 0.0;
      drf[k] = resume && k < w ? sdrift[k] : 0.0;
    }
    // the site of carrier `lane`, in its lane while the trajectory runs (site
    // 0 past n_c)
    uint32_t sx = 0;
    if (lane < nc)
      sx = resume ? socc[lane]
                  : site_pack(uint32_t(a.occ0[td.occ_off + lane]), g);
    occ[lane] = sx;
    __syncthreads();
    double t_clk, energy;
    // path rows are int32 (the host keeps n_path below 2^31)
    const int32_t P = int32_t(td.P);
    int32_t start;
    int64_t hops;
    int no_select;
    if (resume) {
      t_clk = o0.t;
      energy = o0.energy;
      start = uni(int32_t(o0.start));
      hops = int64_t(uni(uint32_t(o0.hops))) |
             (int64_t(uni(uint32_t(o0.hops >> 32))) << 32);
      no_select = uni(o0.no_select);
    } else {
      // initial energy: ewald_neut + q_L A q_L + sum_c q (2 phi_L + psi_self)
      double e_loc = 0.0;
      if (lane < nc) {
        double inner = 0.0;
        for (int c2 = 0; c2 < nc; ++c2)
          inner = fma(q, pair_entry<TT>(tab, gp, sx, occ[c2]), inner);
        e_loc += q * (2.0 * as_global(f.phiL)[sx >> 24] + inner);
      }
      energy = td.ewald_neut + (f.qLAqL + wave_sum(e_loc));
      t_clk = 0.0;
      start = 1;
      hops = 0;
      no_select = 0;
    }
    int64_t slice_done = 0;
    bool finished = false;
    // next hop count that is a positive multiple of `refresh`
    int64_t next_refresh = INT64_MAX;
    if (a.refresh > 0)
      next_refresh =
          hops == 0 ? a.refresh : (hops + a.refresh - 1) / a.refresh * a.refresh;
    // FP32 rates: nu exp(-gs / kT) = 2^(gs (-log2(e) / kT) + log2(nu)),
    // one FMA ahead of v_exp_f32
    const float exp_scale = __uint_as_float(
        uni(__float_as_uint(float(-kLog2E / td.kT))));
    const float exp_bias =
        __uint_as_float(uni(__float_as_uint(float(log2(a.nu)))));
    const double inv_dt = uni(1.0 / td.dt);

    // Uniforms of the coming hops, one hop per lane: at a refill (mti = m)
    // lane l takes u1 and log(u2) (-inf for u2 = 0) of the hop that draws
    // words m + 4 l .. m + 4 l + 3 of the MT block in LDS, and lane c_next
    // holds the next hop's.  Only hops whose four words all lie in the
    // block are cached, so the block is never regenerated ahead of the hops
    // that consume it; a hop whose words straddle the block's end draws
    // them directly.  Each lane takes one FP64 log per up to 64 hops
    // instead of every lane taking one per hop.
    double c_u1 = 0.0, c_lu2 = 0.0;
    int c_next = 0, c_n = 0;
    int box = -1;  // mailbox of the wavefront taking the trajectory over
    // Hops this launch may still make: to max_hops (which finishes the
    // trajectory) and to the end of the slice (which pauses it).  The hop
    // loop counts them down in 32 bits and asks again when they run out, so
    // a budget above 2^31 - 1 is taken in parts.
    auto budget = [&]() __attribute__((always_inline)) {
      int64_t h = INT64_MAX;
      if (td.max_hops > 0) h = td.max_hops - hops;
      if (a.slice_hops > 0) h = min(h, a.slice_hops - slice_done);
      return h;
    };
    uint32_t left = 0, todo = 0;
    // The hops of this launch, kP processes per lane (per <= kP), and the
    // state written back: outputs and resumable state, at the trajectory's
    // end, at the slice's, or at a hop boundary when it is handed over.
    with_processes<kPer>(per, [&](auto n_per) __attribute__((always_inline)) {
      constexpr int kP = decltype(n_per)::value;
      // Process p = lane per + i (the rest: carrier -1, rate 0): its
      // carrier << 9 | its slot << 6, its target, the target's table index
      // << 24 | slot permutation, and psi of the target
      int pd[kP];
      uint32_t px[kP], pinfo[kP];
      double psi[kP];
#pragma unroll
      for (int i = 0; i < kP; ++i) {
        const int p = lane * per + i;
        const bool real = i < per && p < nproc;
        const int c = real ? p / z : 0, j = real ? p - c * z : 0;
        pd[i] = (real ? c << 9 : -512) | (j << 6);
        const uint32_t s = occ[c];
        const uint32_t k = (s >> 24) * z +
                           ((as_global(f.perm)[site_index(s, g)] >> (3 * j)) & 7u);
        px[i] = site_add(s, ptab[k].tgt, g);
        pinfo[i] = (k << 24) | as_global(f.perm)[site_index(px[i], g)];
        if (resume) psi[i] = spsi[c * zp + 1 + j];
      }
      // psi at the site of carrier `lane`
      double psi_s = resume && lane < nc ? spsi[lane * zp] : 0.0;
      auto psi_anew = [&]() __attribute__((always_inline)) {
        uint32_t x[kP + 1];
        double v[kP + 1];
#pragma unroll
        for (int i = 0; i < kP; ++i) x[i] = px[i];
        x[kP] = sx;
        psi_from_table<TT>(tab, gp, q, nc, x, occ, v);
#pragma unroll
        for (int i = 0; i < kP; ++i) psi[i] = v[i];
        psi_s = v[kP];
      };
      if (!resume) psi_anew();
      // lane fc + 16 r forms row r of the fresh sums with the carriers
      // fc + 16 u
      const int fc = lane & 15;
      uint32_t fo[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) fo[u] = occ[fc + 16 * u];
      for (;;) {
        // Conditions on the lane and on the trajectory's sizes are formed
        // again each hop from these copies, which the compiler cannot move
        // out of the loop.  Hoisted, each such condition is a 64-bit lane
        // mask held across the loop, and there are more of them than
        // registers.
        int lane_h = lane, z_h = z, nc_h = nc;
        asm volatile("" : "+v"(lane_h));
        asm volatile("" : "+s"(z_h), "+s"(nc_h));
        const int fc_h = lane_h & 15;
#pragma unroll
        for (int i = 0; i < kP; ++i) asm volatile("" : "+v"(pd[i]));
        // Whatever happens between hops only now and then, at a check: the
        // budget, pacing and hand-over every 64 hops, psi formed anew every
        // `refresh`; `todo` hops follow without one.
        if (todo == 0) {
          if (left == 0) {
            const int64_t b = budget();
            if (b <= 0) {
              finished = td.max_hops > 0 && hops >= td.max_hops;
              break;
            }
            left = uint32_t(min<int64_t>(b, INT32_MAX));
          }
          if (a.progress && (uint32_t(hops) & 63u) == 0) {
            const int busy = pace(a.progress, pslot, left, lane_h);
            if (!stolen && busy >= a.hand_busy && left > kHandMinHops) {
              if (lane_h == 0) box = claim_mailbox(hand_words(a.progress));
              box = uni(__shfl(box, 0, 64));
              if (box >= 0) break;  // hand over at this hop boundary
            }
          }
          if (hops == next_refresh) {
            next_refresh += a.refresh;
            // bound the rounding carried by the incremental updates
            occ[lane_h] = sx;
            __syncthreads();
            psi_anew();
          }
          todo = left;
          if (a.progress) todo = min(todo, 64u - (uint32_t(hops) & 63u));
          todo = uint32_t(min<int64_t>(todo, next_refresh - hops));
          left -= todo;
          slice_done += todo;
        }
        --todo;
        psis[lane_h] = psi_s;
        // ---- two uniforms, as random.random() draws them
        if (c_next >= c_n && mti <= kMtN - 4) {
          c_n = min(64, (kMtN - mti) / 4);
          c_next = 0;
          if (lane_h < c_n) {
            const int w = mti + 4 * lane_h;
            c_u1 = mt_uniform(mt_temper(mt[w]), mt_temper(mt[w + 1]));
            const double u2 =
                mt_uniform(mt_temper(mt[w + 2]), mt_temper(mt[w + 3]));
            c_lu2 = u2 > 0.0 ? log(u2) : -INFINITY;
          }
        }
        double u1, lu2;
        if (c_next < c_n) {
          u1 = read_lane(c_u1, c_next);
          lu2 = read_lane(c_lu2, c_next);
          ++c_next;
          mti += 4;
        } else {
          uint32_t wd[4];
          mt_next4(mt, mti, lane_h, wd);
          u1 = uni(mt_uniform(wd[0], wd[1]));
          const double u2 = mt_uniform(wd[2], wd[3]);
          lu2 = uni(u2 > 0.0 ? log(u2) : -INFINITY);
        }
        __syncthreads();
        // ---- rates: psi of the carriers' sites and the rate inputs of all
        // processes are read before the first is used
        double kv[kP], gv[kP], ps[kP];
        Rate<kF32Rate> e[kP];
        double ksum = 0.0;
#pragma unroll
        for (int i = 0; i < kP; ++i) ps[i] = psis[max(pd[i], 0) >> 9];
#pragma unroll
        for (int i = 0; i < kP; ++i) e[i] = Rate<kF32Rate>(ptab[pinfo[i] >> 24]);
#pragma unroll
        for (int i = 0; i < kP; ++i) {
          const bool real = pd[i] >= 0;
          const double dpsi = psi[i] - ps[i];
          double g0;
          if constexpr (kF32Rate) {
            g0 = e[i].g0s + 2 * q * dpsi;
            const float gf = float(g0);
            const float gs =
                (e[i].lam + gf) * (e[i].lam + gf) * e[i].i4l - e[i].vs;
            const float kf =
                __builtin_amdgcn_exp2f(fmaf(gs, exp_scale, exp_bias));
            kv[i] = double(real ? kf : 0.0f);
          } else {
            g0 = 2 * q * ((e[i].dphi + dpsi) + e[i].tq) + e[i].dE;
            const double lam = e[i].lam;
            const double gs =
                (((lam + g0) * (lam + g0) / (4 * lam)) - e[i].vab) - e[i].shift;
            const double k = a.nu * numpy_e_pow(-gs / td.kT);
            kv[i] = real ? k : 0.0;
          }
          gv[i] = g0;
          ksum = i == 0 ? kv[0] : ksum + kv[i];
        }
        // ---- FP64 prefix and selection.  FP64 rates: the prefix of the
        // quotients k / k_tot against u1, as the reference forms it; FP32
        // rates: one scan of the rates themselves against u1 k_tot.
        double k_tot, thr, cum;
        double xq[kP];
        if (kF32Rate) {
          const double incl = wave_incl_scan(ksum);
          k_tot = read_lane(incl, 63);
          cum = dpp_f64<kDppWaveShr1, 0xf, true>(incl);
          thr = u1 * k_tot;
#pragma unroll
          for (int i = 0; i < kP; ++i) xq[i] = kv[i];
        } else {
          k_tot = wave_sum(ksum);
          double xs = 0.0;
#pragma unroll
          for (int i = 0; i < kP; ++i) {
            xq[i] = kv[i] / k_tot;
            xs += xq[i];
          }
          cum = wave_excl_scan(xs);
          thr = u1;
        }
        // The selected process is the first (lane, i), lane-major, whose
        // running sum cum + xq[0] + ... + xq[i] exceeds thr.  The terms are
        // non-negative, so each lane's running sums do not decrease: the
        // count of them that stay <= thr is the index of the lane's first
        // crossing (a lane crosses iff the count is below per, and its first
        // process is real: processes past nproc add zero at the lane's end).
        int nb = 0;
#pragma unroll
        for (int i = 0; i < kP; ++i) {
          cum += xq[i];
          nb += cum > thr ? 0 : 1;
        }
        const unsigned long long mask =
            __ballot(int(pd[0] >= 0) & int(nb < per));
        int src, isel = 0;
        if (mask) {
          src = uni(__ffsll(static_cast<long long>(mask)) - 1);
          if constexpr (kP > 1) isel = __builtin_amdgcn_readlane(nb, src);
        } else {
          // rounding left every running sum <= thr: take the last process
          src = (nproc - 1) / per;
          isel = nproc - 1 - src * per;
          ++no_select;
        }
        int m = 0;
        uint32_t s_new = 0, info_sel = 0;
        double gsel = 0.0, ksel = 0.0;
#pragma unroll
        for (int i = 0; i < kP; ++i)
          if (kP == 1 || i == isel) {
            m = __builtin_amdgcn_readlane(pd[i], src) >> 9;
            s_new = uint32_t(__builtin_amdgcn_readlane(int(px[i]), src));
            info_sel = uint32_t(__builtin_amdgcn_readlane(int(pinfo[i]), src));
            gsel = read_lane(gv[i], src);
            ksel = read_lane(kv[i], src);
          }
        // ---- one round of independent loads for the whole update
        const uint32_t s_old = uint32_t(__builtin_amdgcn_readlane(int(sx), m));
        const uint32_t sub_new = s_new >> 24;
        const uint32_t perm_new = info_sel & 0xffffffu;
        const uint32_t rec_old = info_sel >> 24;
        // Slot k of the new site in the 16 lanes of row k mod 4: its target,
        // the target's table index and slot permutation, and the entries of
        // every carrier there (in FP32 or FP64, used after the update: the
        // loads overlap)
        constexpr int kT = kZp > 5 ? 2 : 1;  // rounds of 4 slots
        uint32_t nsite[kT], ninfo[kT];
        TT fent[kT][4];
#pragma unroll
        for (int u = 0; u < 4; ++u) fo[u] = fc_h + 16 * u == m ? s_new : fo[u];
#pragma unroll
        for (int t = 0; t < kT; ++t) {
          const int k4 = (lane_h >> 4) + 4 * t, k = k4 < z_h ? k4 : 0;
          const uint32_t rec = sub_new * z_h + ((perm_new >> (3 * k)) & 7u);
          nsite[t] = site_add(s_new, ptab[rec].tgt, g);
          ninfo[t] =
              (rec << 24) | as_global(f.perm)[site_index(nsite[t], g)];
          const uint32_t row = tab.row(nsite[t] >> 24);
          const RowKey key = row_key(nsite[t], gp);
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            fent[t][u] = TT(0);
            if (16 * u < nc_h) fent[t][u] = tab.at(row, rel_col(key, fo[u], gp));
          }
        }
        // Every row's change q (A[n, x] - A[s, x]) is loaded before any is
        // used: one entry of the family's hop differences (row rec_old, x's
        // column in s_old's row) where it has them, else both table entries
        const uint32_t rn = tab.row(sub_new), ro = tab.row(s_old >> 24);
        const RowKey key_new = row_key(s_new, gp), key_old = row_key(s_old, gp);
        const uint32_t rd = dtab.row(rec_old);
        double dx[kP], ds;
        if (use_d) {
#pragma unroll
          for (int i = 0; i < kP; ++i)
            dx[i] = dtab.at(rd, rel_col(key_old, px[i], gp));
          ds = dtab.at(rd, rel_col(key_old, sx, gp));
        } else {
          TT an[kP], ao[kP];
#pragma unroll
          for (int i = 0; i < kP; ++i) {
            an[i] = tab.at(rn, rel_col(key_new, px[i], gp));
            ao[i] = tab.at(ro, rel_col(key_old, px[i], gp));
          }
          const TT sn = tab.at(rn, rel_col(key_new, sx, gp));
          const TT so = tab.at(ro, rel_col(key_old, sx, gp));
#pragma unroll
          for (int i = 0; i < kP; ++i) dx[i] = double(an[i]) - double(ao[i]);
          ds = double(sn) - double(so);
        }
        // ---- clock, while the loads are in flight
        int32_t end;
        if (lu2 > -INFINITY) {  // u2 > 0
          t_clk -= lu2 / k_tot;
          // path step int(t / dt) of the correctly rounded quotient: below
          // 1e6, t (1/dt) is within 4e-10 of it, so more than 1e-9 away from
          // an integer its integer part is the quotient's; otherwise divide
          const double qf = t_clk * inv_dt;
          const double fr = qf - floor(qf);
          if (fr > 1e-9 && fr < 1.0 - 1e-9 && qf < 1.0e6) {
            end = int32_t(qf);
          } else {
            asm volatile("");  // the division only where it is needed
            const double qq = t_clk / td.dt;
            end = qq < double(P) ? int32_t(qq) : P;
          }
        } else {
          t_clk = INFINITY;
          end = P;
        }
        energy += gsel;
        // carrier m's displacement and drift, a lane per axis
        if (lane_h < 3) {
#pragma clang fp contract(off)
          const double v = ptab[rec_old].vec[lane_h];
          lds_add(dsp + 3 * m + lane_h, v);
          if (field_on) lds_add(drf + 3 * m + lane_h, v * ksel);
        }
        // ---- apply
#pragma unroll
        for (int i = 0; i < kP; ++i) psi[i] = fma(q, dx[i], psi[i]);
        psi_s = fma(q, ds, psi_s);
        double v_new = 0.0;
#pragma unroll
        for (int i = 0; i < kP; ++i)
          if (kP == 1 || i == isel) v_new = read_lane(psi[i], src);
        const double v_old = read_lane(psi_s, m);
        // the fresh rows' sums over the carriers: fc + 32 to fc, those of
        // fc + 16 and fc + 48 to them, then over the 16 lanes
        double fresh[kT];
#pragma unroll
        for (int t = 0; t < kT; ++t) {
          double part[4];
#pragma unroll
          for (int u = 0; u < 4; ++u)
            part[u] = fc_h + 16 * u < nc_h ? q * double(fent[t][u]) : 0.0;
          double x = part[0];
          if (nc_h > 16) {
            if (nc_h > 32) x += part[2];
            x += nc_h > 48 ? part[1] + part[3] : part[1];
          }
          x += dpp_f64<kDppRowRor + 8, 0xf, true>(x);
          x += dpp_f64<kDppRowRor + 4, 0xf, true>(x);
          x += dpp_f64<kDppRowRor + 2, 0xf, true>(x);
          x += dpp_f64<kDppRowRor + 1, 0xf, true>(x);
          // (the slot that returns to s_old has its row already)
          fresh[t] = nsite[t] != s_old ? x : v_old;
        }
        // carrier m's new processes and site row
#pragma unroll
        for (int i = 0; i < kP; ++i) {
          uint32_t nx = lane_at(pd[i], nsite[0]);
          uint32_t ni = lane_at(pd[i], ninfo[0]);
          uint32_t nl = lane_at(pd[i], lo32(fresh[0]));
          uint32_t nh = lane_at(pd[i], hi32(fresh[0]));
          if constexpr (kT > 1)
            if (z_h > 4) {
              const bool far = pd[i] & 256;  // slots 4 to 7
              const uint32_t fx = lane_at(pd[i], nsite[1]);
              const uint32_t fi = lane_at(pd[i], ninfo[1]);
              const uint32_t fl = lane_at(pd[i], lo32(fresh[1]));
              const uint32_t fh = lane_at(pd[i], hi32(fresh[1]));
              nx = far ? fx : nx;
              ni = far ? fi : ni;
              nl = far ? fl : nl;
              nh = far ? fh : nh;
            }
          const bool mine = (pd[i] >> 9) == m;
          px[i] = mine ? nx : px[i];
          pinfo[i] = mine ? ni : pinfo[i];
          psi[i] = mine ? from32(nl, nh) : psi[i];
        }
        sx = lane_h == m ? s_new : sx;
        psi_s = lane_h == m ? v_new : psi_s;
        // ---- path rows [start, end), written by the owner lane of each entry
        ++hops;
        bool full = false;
        if (end >= start + 1) {
          if (end >= P) end = P;
          for (int k = lane_h; k < 3 * nc_h; k += 64) {
            const double v = sbase[k] + dsp[k];
            dsp[k] = 0.0;
            for (int32_t r = start; r < end; ++r) rows[int64_t(r) * w + k] = v;
            sbase[k] = v;
          }
          start = end;
          full = end >= P;
        }
        __syncthreads();
        if (full) {
          finished = true;
          break;
        }
      }
      // (the psi rows of carrier c: its site's, then its targets')
#pragma unroll
      for (int i = 0; i < kP; ++i)
        if (pd[i] >= 0) spsi[(pd[i] >> 9) * zp + 1 + ((pd[i] >> 6) & 7)] = psi[i];
      if (lane < nc) spsi[lane * zp] = psi_s;
    });
    if (a.progress) {  // nothing left: out of its SIMD mates' way
      if (lane == 0)
        __hip_atomic_store(a.progress + pslot, 0u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      __builtin_amdgcn_s_setprio(0);
    }
    // every carrier slot of the output, zero past the trajectory's own
    static_assert(kMaxCarriers == 64, "one carrier per lane");
#pragma unroll
    for (int c3 = 0; c3 < 3; ++c3) {
      const int k = lane + 64 * c3;
      a.drift[int64_t(tr) * 3 * kMaxCarriers + k] = drf[k];
      if (k < w) {
        sdisp[k] = dsp[k];
        sdrift[k] = drf[k];
      }
    }
    for (int k = lane; k < 624; k += 64) mts[k] = mt[k];
    if (lane < nc) socc[lane] = sx;
    if (lane == 0) {
      mts[624] = uint32_t(mti);
      TrajOut o;
      o.t = t_clk;
      o.energy = energy;
      o.hops = hops;
      o.start = start;
      o.no_select = no_select;
      o.done = box < 0 && finished ? 1 : 0;
      o.started = 1;
      o.simd = int32_t(simd_key());
      o.busy = (resume ? o0.busy : 0.0) + double(wall_clock64() - w_start);
      a.out[tr] = o;
    }
    __syncthreads();
    if (box >= 0) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      int handed = 0;
      if (lane == 0) {
        uint32_t expect = 0u;
        handed = __hip_atomic_compare_exchange_strong(
            hand_words(a.progress) + kHandHdr + box, &expect,
            uint32_t(tr) + 1u, __ATOMIC_RELEASE, __ATOMIC_RELAXED,
            __HIP_MEMORY_SCOPE_AGENT);
      }
      // the trajectory lives on in the wavefront it was handed to
      if (uni(__shfl(handed, 0, 64))) return;
      again = tr;  // that wavefront stopped waiting: resume it here
      continue;
    }
    if (a.progress && lane == 0)
      atomicSub(hand_words(a.progress) + kHandLeft, 1u);
  }
}

template <typename TT, bool kF32Rate, int kPer, int kZp>
__global__ void __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(PYCD_BATCH_WAVES_PER_EU(kF32Rate, kPer))))
kmc_batched_kernel(BatchArgs a) {
  kmc_batched_body<TT, kF32Rate, kPer, kZp>(a);
}

// The serving pool's slices: the same body under its own name, so that a
// profile tells the batch launch from the pool's launches.
template <typename TT, bool kF32Rate, int kPer, int kZp>
__global__ void __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(PYCD_BATCH_WAVES_PER_EU(kF32Rate, kPer))))
kmc_pool_kernel(BatchArgs a) {
  kmc_batched_body<TT, kF32Rate, kPer, kZp>(a);
}

// Squared displacement per trajectory, averaged over its carriers:
//   msd[t, tau] = mean_c mean_{t0 < P_t - tau} |r_c(t0 + tau) - r_c(t0)|^2
// (P_t: the path rows the run wrote).  msd_unit_kernel: one workgroup per
// (trajectory, carrier) unit, sums over origins (msd.hpp), unscaled, per
// (unit, lag) to scratch.  msd_reduce_kernel: one thread per (trajectory,
// lag) sums the carriers in order and scales by scale^2 / (P_t - tau) / n_c:
// the same order in every launch, so results repeat bit for bit.
//
// Workgroup b runs on XCD b mod 8 (workgroups are dealt to the XCDs in
// turn); the host deals each trajectory's units to one XCD, so the cache
// lines of path rows that its carriers share come from HBM once.
struct MsdTraj {
  int64_t row_off;
  int64_t P;
  int32_t nc;
  int32_t traj;     // index into the trajectory results (rows written)
  int64_t out_off;
  int64_t M;
  int64_t sbase;    // scratch offset of carrier 0's M lag sums
};

template <int kQ>
__global__ void __launch_bounds__(kMsdThreads)
__attribute__((amdgpu_waves_per_eu(4, 4)))
msd_unit_kernel(const double* __restrict__ rows,
                const MsdTraj* __restrict__ tr,
                const TrajOut* __restrict__ outs,
                const int32_t* __restrict__ units,
                double* __restrict__ scratch) {
  const int32_t u = units[blockIdx.x];
  if (u < 0) return;  // padding of an XCD's list (the whole workgroup)
  const MsdTraj d = tr[u >> 6];
  const int c = u & 63;
  // only the rows written by the run: [0, start) (all P when the path filled)
  const int64_t written = outs[d.traj].start;
  const int64_t P = written < 1 ? 1 : (written < d.P ? written : d.P);
  double* out = scratch + d.sbase + int64_t(c) * d.M;
  msd_unit<kQ>((gptr<double>)(rows + d.row_off + 3 * c), 3 * int64_t(d.nc), P,
               0, d.M, false, 0, 1, kMsdWin,
               [&](int64_t tau, double v) { out[tau] = v; });
}

__global__ void __launch_bounds__(256)
msd_reduce_kernel(const MsdTraj* __restrict__ tr, int64_t n_traj,
                  const TrajOut* __restrict__ outs,
                  const double* __restrict__ scratch, double scale,
                  double* __restrict__ out) {
  const int64_t k = blockIdx.x;
  if (k >= n_traj) return;
  const MsdTraj d = tr[k];
  const int64_t written = outs[d.traj].start;
  const int64_t P = written < 1 ? 1 : (written < d.P ? written : d.P);
  const double s2 = scale * scale;
  for (int64_t tau = threadIdx.x; tau < d.M; tau += blockDim.x) {
    double v = 0.0;
    if (tau >= 1 && tau < P) {
      double acc = 0.0;
      for (int c = 0; c < d.nc; ++c) acc += scratch[d.sbase + c * d.M + tau];
      v = acc * s2 / double(P - tau) / double(d.nc);
    }
    out[d.out_off + tau] = v;
  }
}

__global__ void fill_u32(uint32_t* p, int64_t n, uint32_t v) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x)
    p[i] = v;
}

// Hand-over words before a launch: `active` unfinished trajectories, no
// mailbox taken or opened, `cap` mailboxes (0: off), every mailbox empty.
__global__ void hand_reset(uint32_t* h, int64_t n, uint32_t active,
                           uint32_t cap) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x)
    h[i] = i == kHandLeft ? active : (i == kHandCap ? cap : 0u);
}

__global__ void reset_outputs(TrajOut* o, int64_t n) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x) {
    o[i].done = 0;
    o[i].started = 0;
  }
}

__global__ void fill_f64(double* p, int64_t n, double v) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x)
    p[i] = v;
}

// Family preparation kernels.
__global__ void to_f32(const double* __restrict__ a, float* __restrict__ b,
                       int64_t n) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x)
    b[i] = float(a[i]);
}

// Largest |A[i, j] - C[sub(i), rel(i, j)]| over the full table A, whose
// first n_unit rows are C, as the bit pattern of a non-negative double
// (ordered like the values).  One workgroup of 256 per 4 rows.
__global__ void __launch_bounds__(256)
compact_check(const double* __restrict__ A, int64_t N, Geo g,
              unsigned long long* __restrict__ worst) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double m = 0.0;
  for (int64_t i = int64_t(blockIdx.x) * 4 + wave; i < N;
       i += int64_t(gridDim.x) * 4) {
    const uint32_t a = site_pack(uint32_t(i), g);
    const double* row = A + i * N;
    const double* crow0 = A + int64_t(a >> 24) * N;
    for (int64_t j = lane; j < N; j += 64) {
      const uint32_t b = site_pack(uint32_t(j), g);
      m = nan_max(m, fabs(row[j] - crow0[rel_col(a, b, geo_pk(g))]));
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    m = nan_max(m, __shfl_xor(m, off, 64));
  if (lane == 0)
    atomicMax(worst, static_cast<unsigned long long>(__double_as_longlong(m)));
}

}  // namespace pycd

// ------------------------------------------------------------------- host --
using namespace pycd;

struct BatchFamily {
  DevBuf<double> C64, phiL, D;
  DevBuf<float> C32;
  DevBuf<SubRec> subs;
  DevBuf<uint32_t> perm;
  int64_t N = 0;
  int z = 0, mz = 0;
  Geo g{1, 1, 1, 1};
  double qLAqL = 0.0;
  std::vector<char> hop_sub;  // per sublattice: its sites hop
  size_t device_bytes = 0;
};

struct pycd_batch {
  pycd_ctx* ctx = nullptr;
  std::vector<BatchFamily*> fams;
  DevBuf<FamDev> d_fams;
  int table_prec = 0;  // 0 FP64, 1 FP32
  bool use_diff = true;  // launches read the families' hop differences
  int64_t refresh = 1024;   // set from the rate precision at creation
  int rate_prec = 0;   // 0 FP64, 1 FP32
  double nu = 0.0;
  // per-run buffers
  DevBuf<TrajDev> d_trajs;
  DevBuf<int32_t> d_order;
  DevBuf<int64_t> d_occ;
  DevBuf<uint32_t> d_mt, d_counter, d_bins;
  DevBuf<int16_t> d_keybin;
  // pacing slots, one per SIMD wave slot, then the hand-over words (binned
  // runs)
  DevBuf<uint32_t> d_prog;
  int n_bins = 1;
  uint32_t hand_cap = 0;  // mailboxes (0 for the serving pool)
  int32_t hand_busy = 1;  // see BatchArgs
  bool handover = true;
  DevBuf<double> d_rows, d_drift, d_msd;
  DevBuf<TrajOut> d_out;
  DevBuf<uint32_t> d_mts;
  DevBuf<uint32_t> d_socc;
  DevBuf<double> d_svec, d_spsi;
  // slot pool (serving)
  bool pool = false;
  int64_t rows_capacity = 0;
  std::vector<char> slot_busy;
  std::vector<MsdTraj> msd_host;
  DevBuf<MsdTraj> d_msdtr;
  // MSD launch plan: (trajectory, carrier) units in workgroup order and
  // the per-unit lag sums
  DevBuf<int32_t> d_msd_units;
  DevBuf<double> d_msd_scratch;
  int64_t msd_units = 0;
  int msd_kq = 64;  // lanes per group of the MSD kernel (msd.hpp)
  std::vector<TrajDev> trajs;
  std::vector<int64_t> msd_off;
  int64_t n_traj = 0, rows_total = 0, msd_total = 0;
  int nc_max = 0, z_max = 0;
  int sub_max = kMaxSubSlots;
  double msd_scale = 1.0;
  size_t smem = 0;
  int grid = 0;
  hipGraphExec_t graph = nullptr;
  float last_ms = 0.f;
  float kernel_ms = 0.f;  // the KMC kernel alone, last eager run or step
  ~pycd_batch() {
    if (graph) (void)hipGraphExecDestroy(graph);
    for (auto* f : fams) delete f;
  }
};

#include "batch_api.inc"

