// Plain (one-trajectory) KMC loop of PyCD's Run.do_kmc_steps on gfx950.
//
// Per hop (PyCD/core.py:2787-2861, rates from :1989-2050):
//   dG0_p = 2 q_s [ q.(A[n,:] - A[s,:]) + q_s (A[s,s] - A[s,n]) ] + E[n] - E[s]
//   dGs_p = ((lambda + dG0)^2 / (4 lambda) - V_ab) - 0.5 F.d
//   k_p   = nu * e**(-dGs / kT)
//   select the first p with cumsum(k / k_tot)_p > u1; t -= ln(u2) / k_tot
//
// The N-long dot product is never formed.  With q = q_lattice + sum_c q_c
// e_{occ_c},  q.A[x,:] = phi_L[x] + psi[x],  where phi_L = A q_lattice is
// computed once per table and psi[x] = sum_c q_c A[x, occ_c] covers the
// sites x that matter: every carrier's site and its z hop targets.  The
// value of q.(A[n,:] - A[s,:]) is the same up to rounding.
//
// One persistent workgroup runs the trajectory (the hop chain is serial);
// psi of every row is kept from hop to hop, see kmc_hop_kernel.
#include "common.hpp"
#include "packed_sites.hpp"
#include "wave.hpp"

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <cmath>

namespace pycd {

struct KmcScalars {
  double t;
  double energy;
  int64_t start;
  int64_t hops;
  int32_t finished;
  int32_t no_select;  // hops where rounding left no cum > u1 (last taken)
};

// What the hop loop reads once and the state it begins with and leaves.
struct KmcDev {
  const uint32_t* pk;  // packed code of every site (cell-0 rows only)
  const double* cq;
  int32_t* occ;
  double* disp;
  double* base;
  double* drift;
  KmcScalars* sc;
};

// log(u2) of every uniform pair ahead of the hop loop (0 where u2 = 0, a
// value the loop does not use), so that no hop waits for an FP64 log.
__global__ void __launch_bounds__(256)
log_u2_kernel(const double* __restrict__ U, int64_t n,
              double* __restrict__ lu) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x) {
    const double u2 = U[2 * i + 1];
    lu[i] = u2 > 0.0 ? log(u2) : 0.0;
  }
}

// ---------------------------------------------------------------------------
// Inputs of the hop loop.  Per (site, slot) a 64-byte record:
// the self term A[s, s] - A[s, n], lambda, 1 / (4 lambda), V_ab plus the
// field shift 0.5 F.d, the hop vector d and the lattice part
// q_L . (A[n, :] - A[s, :]) of the hop's potential difference; per site
// (phi_L, E); per (site, slot) the target and its packed code (0 without
// cell-0 rows).
struct alignas(16) SlotRec {
  double tself, lam, i4l, vs;
  double v[3];
  double dphi;
};

// What the hop loop reads, by value; state read only before and after it
// comes from a KmcDev in device memory.
struct HopArgs {
  const char* tab;       // the table (full, or the rows of cell 0)
  uint32_t row_bytes;    // N sizeof(double)
  GeoPk gp;
  const SlotRec* rec;
  const double2* pe;
  const int2* nbr2;
  double* rows;
  double* epath;
  double* dpath;
  const double* U;
  const double* LU;
  double* hop_time;
  int32_t* hop_proc;
  int32_t nc, z, mz, field_on;
  double nu, nkt, dt;  // nkt = -1 / kT
  int64_t P, n_pairs, max_hops;
};

// Records of every (site, slot) from the slot tables (products and sums
// rounded one by one).
__global__ void pack_slot_records(int64_t NM, const double* __restrict__ tself,
                                  const double* __restrict__ dphi,
                                  const double* __restrict__ lam,
                                  const double* __restrict__ vab,
                                  const double* __restrict__ vec,
                                  const int32_t* __restrict__ nbr,
                                  const uint32_t* __restrict__ nbr_pk,
                                  double f0, double f1, double f2,
                                  int field_on, SlotRec* __restrict__ rec,
                                  int2* __restrict__ nbr2) {
#pragma clang fp contract(off)
  const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k >= NM) return;
  SlotRec r;
  r.tself = tself[k];
  r.lam = lam[k];
  r.i4l = 1.0 / (4 * r.lam);
  r.v[0] = vec[3 * k];
  r.v[1] = vec[3 * k + 1];
  r.v[2] = vec[3 * k + 2];
  const double shift =
      field_on ? 0.5 * (f0 * r.v[0] + f1 * r.v[1] + f2 * r.v[2]) : 0.0;
  r.vs = vab[k] + shift;
  r.dphi = dphi[k];
  rec[k] = r;
  nbr2[k] = make_int2(nbr[k], nbr_pk ? int(nbr_pk[k]) : 0);
}

__global__ void pack_site_pe(int64_t N, const double* __restrict__ phiL,
                             const double* __restrict__ E,
                             double2* __restrict__ pe) {
  const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k < N) pe[k] = make_double2(phiL[k], E[k]);
}

template <typename T>
using gmem = const __attribute__((address_space(1))) T*;

// ---------------------------------------------------------------------------
// Sums carried as an unevaluated pair h + l (about 106 bits), so that a sum
// that is kept up by adding and taking away terms for the whole trajectory
// stays the correctly rounded sum of its terms.
struct Dd {
  double h = 0.0, l = 0.0;
};

__device__ __forceinline__ void dd_add(Dd& a, double v) {
#pragma clang fp contract(off)
  const double s = a.h + v, b = s - a.h;
  a.l += (a.h - (s - b)) + (v - b);
  a.h = s;
}

// a += q v, the product's rounding error included.
__device__ __forceinline__ void dd_add_prod(Dd& a, double q, double v) {
#pragma clang fp contract(off)
  const double p = q * v;
  const double e = fma(q, v, -p);
  dd_add(a, p);
  a.l += e;
}

__device__ __forceinline__ void dd_add(Dd& a, const Dd& b) {
#pragma clang fp contract(off)
  dd_add(a, b.h);
  a.l += b.l;
}

// h becomes the nearest double of the sum.
__device__ __forceinline__ void dd_norm(Dd& a) {
#pragma clang fp contract(off)
  const double s = a.h + a.l;
  a.l -= s - a.h;
  a.h = s;
}

// A sum over each row of 16 lanes, in every lane of the row.
template <int kRor>
__device__ __forceinline__ void dd_rotate_add(Dd& a) {
  Dd o;
  o.h = dpp_f64<kDppRowRor + kRor, 0xf, true>(a.h);
  o.l = dpp_f64<kDppRowRor + kRor, 0xf, true>(a.l);
  dd_add(a, o);
}

__device__ __forceinline__ void dd_row_sum(Dd& a) {
  dd_rotate_add<8>(a);
  dd_rotate_add<4>(a);
  dd_rotate_add<2>(a);
  dd_rotate_add<1>(a);
  dd_norm(a);
}

// f(std::integral_constant<int, n>) for the run-time n in [kMin, kMax],
// small n first.
template <int kMin, int kMax, typename F>
__device__ __forceinline__ void with_count_up(int n, F&& f) {
  if constexpr (kMin <= kMax) {
    if (n == kMin)
      f(std::integral_constant<int, kMin>{});
    else
      with_count_up<kMin + 1, kMax>(n, f);
  }
}

// The hop loop.
//
// A block of wavefronts in three roles.  Process wavefronts: a lane owns a
// process, its target row of psi and its rate inputs in registers.  Site
// wavefronts: lane c owns carrier c's site row, displacement, path base and
// drift; they keep the clock and write the path.  Helpers: the mover's new
// rows.  psi[x] = sum_c q_c A[x, occ_c] of a row is a Dd that the hops keep
// up: when carrier m hops s -> n every row gains q_m A[x, n] and loses
// q_m A[x, s].  The mover's new site row continues the row of n; its z
// slots are summed afresh by the helpers, four rows of 16 lanes at a time,
// a lane over every 16th carrier.  A hop takes 2 n_c (1 + z) + z n_c
// gathers in one round instead of the n_c (1 + z) n_c of summing every row,
// and psi is the correctly rounded sum, where a chain over the carriers
// carries a rounding per term.
//
// What bounds it is the chain of latencies of a hop: rates, their scan and
// the selection, the LDS reads that the selected process names, one round
// of gathers, the updates.  Two barriers per hop: after the rates, which
// every wavefront sums and selects from by itself, and after the update;
// both wait for LDS operations only.  What a hop changes in LDS that others
// still read in its update (targets, sites) is written in the next hop's
// rates phase.  With the look-ahead (every process's targets' targets in
// LDS) no gather address waits for another load.
//
// Per hop, z = 4, before (n_c <= 64: one wavefront with every row's entries
// in LDS; more: a workgroup that gathered them all again) and now: 1.40 and
// 0.96 us with 1 carrier, 1.65 and 1.07 with 16 (6144 sites, 2600 cycles),
// 21.6 and 1.5 with 96 (2592 sites).  At n_c = 16 a hop is about 660
// cycles of rates, 660 of scan and selection, 700 to 1200 of LDS reads,
// gathers and the clock, 200 of updates, the rest at the barriers; with 96
// carriers the helper's z n_c gathers are the longest of the three.
struct HopLds {
  int nc, z, look;
  __host__ __device__ constexpr int np() const { return nc * z; }
  // rates of p at (p mod per) kStride + p / per, so that lane l's processes
  // l per .. l per + per - 1 are read on distinct banks
  static constexpr int kStride = 65;
  __host__ __device__ constexpr int per() const { return (np() + 63) / 64; }
  // psi of the site rows, charges, rates, dG0, hop vectors, the mover's
  // rows; sites, targets and look-ahead with their codes; the end flag
  __host__ __device__ constexpr size_t bytes() const {
    return 8 * (2 * size_t(nc) + size_t(per()) * kStride + 4 * size_t(np()) +
                2 * size_t(z) + 2) +
           8 * (size_t(nc) + size_t(np()) + (look ? size_t(np()) * z : 0)) + 8;
  }
};

// Wavefronts of each role: n_c z <= 640 processes, n_c <= 320 carriers; a
// helper for every 4 slots while there is room (three for any z > 8: 64 slots
// took 6 rounds of gathers a hop, 3.05 us with 1 carrier, where the workgroup
// kernel before had 2.79; now 2.39).
constexpr int kHopWaves = 16;  // at most
struct HopRoles {
  int process, site, helper;
  HopRoles() = default;
  constexpr HopRoles(int nc, int z)
      : process((nc * z + 63) / 64), site((nc + 63) / 64),
        helper(std::max(1, std::min((z + 3) / 4,
                                    kHopWaves - process - site))) {}
  constexpr int threads() const { return 64 * (process + site + helper); }
  // Every process and carrier is owned by a lane, a lane sums at most 10
  // processes, and the block holds the wavefronts.
  constexpr bool fit(int nc, int z) const {
    return process <= 10 && threads() <= 64 * kHopWaves &&
           64 * process >= nc * z && 64 * site >= nc;
  }
};

// The sessions that pycd_kmc_create takes: n_c (104 z + 88) <= kSessionMost
// (z = 4: 121 carriers), all of which the hop kernel can run.
constexpr int64_t kSessionMost = 61424;
constexpr bool session_fits(int64_t nc, int64_t z) {
  return nc * (104 * z + 88) <= kSessionMost;
}
constexpr bool every_session_runs() {
  for (int z = 1; z <= 64; ++z)
    for (int nc = 1; session_fits(nc, z); ++nc)
      if (!HopRoles(nc, z).fit(nc, z) || HopLds{nc, z, 0}.bytes() > 65536)
        return false;
  return true;
}
static_assert(every_session_runs(), "the hop kernel holds every session");

template <bool kCompact, bool kLook>
__global__ void __launch_bounds__(64 * kHopWaves)
kmc_hop_kernel(HopArgs a, const KmcDev* __restrict__ dv, HopRoles roles,
               int32_t* __restrict__ status) {
  extern __shared__ double smem[];
  __shared__ double ext[64];  // 2^(j/64)
  const int nc = a.nc, z = a.z, nproc = nc * z;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kT = blockDim.x;
  const HopLds lay{nc, z, kLook ? 1 : 0};
  const int per = lay.per();
  double* psis = smem;                             // nc
  double* cqs = psis + nc;                         // nc
  double* kks = cqs + nc;                          // per kStride
  double* dgs = kks + per * HopLds::kStride;       // nproc
  double* pv3 = dgs + nproc;                       // 3 nproc
  double* fresh = pv3 + 3 * nproc;                 // z pairs (h, l)
  double* box = fresh + 2 * z;                     // psi[n] (h, l)
  // sites with their packed codes (0 without cell-0 rows)
  int2* occ = reinterpret_cast<int2*>(box + 2);    // carriers (nc)
  int2* tgt = occ + nc;                            // targets (nproc)
  int2* tt = tgt + nproc;                          // look-ahead (nproc z)
  int* over = reinterpret_cast<int*>(tt + (kLook ? nproc * z : 0));

  // A[x, y]: the full table's row x, or (compact) the cell-0 row of x's
  // sublattice at y moved by -cell(x)
  auto entry = [&](int2 x, int2 y) __attribute__((always_inline)) -> double {
    if constexpr (kCompact) {
      const uint32_t xk = uint32_t(x.y);
      const uint32_t off =
          (xk >> 24) * a.row_bytes + rel_col(xk, uint32_t(y.y), a.gp) * 8u;
      return *(gmem<double>)(a.tab + off);
    } else {
      const uint64_t off = uint64_t(uint32_t(x.x)) * a.row_bytes +
                           uint64_t(uint32_t(y.x)) * 8u;
      return *(gmem<double>)(a.tab + off);
    }
  };
  // a barrier for what passes through LDS: loads in flight stay in flight
  auto lds_barrier = [] {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  // the same site in every lane, in scalar registers
  auto uniform = [](int2 v) {
    return make_int2(__builtin_amdgcn_readfirstlane(v.x),
                     __builtin_amdgcn_readfirstlane(v.y));
  };

  if (tid < 64) ext[tid] = __builtin_bit_cast(double, kExp2J64[tid]);
  if (tid == 0) *over = 0;
  for (int c = tid; c < nc; c += kT) {
    const int s = dv->occ[c];
    occ[c] = make_int2(s, kCompact ? int(dv->pk[s]) : 0);
    cqs[c] = dv->cq[c];
  }
  // (the rates past the last process stay zero)
  for (int k = tid; k < per * HopLds::kStride; k += kT) kks[k] = 0.0;
  __syncthreads();
  // every process's look-ahead: the z targets of its target
  if constexpr (kLook)
    for (int u = tid; u < nproc * z; u += kT) {
      const int p = u / z, k = u - p * z;
      const int c = p / z, j = p - c * z;
      const int n = a.nbr2[int64_t(occ[c].x) * a.mz + j].x;
      tt[u] = a.nbr2[int64_t(n) * a.mz + k];
    }

  // ---- hops made, the last selection
  const KmcScalars sc0 = *dv->sc;
  // hops that this call may make
  int64_t due = a.n_pairs;
  if (a.max_hops > 0)
    due = min(due, max(a.max_hops - sc0.hops, int64_t(0)));
  if (sc0.finished) due = 0;
  int64_t h = 0;
  int m = -1;  // the last hop's carrier (-1: none made yet)
  int sel = 0, noselect = sc0.no_select;
  double k_tot = 0.0, u1c = 0.0;
  // sel / z = sel z_inv >> 16 for sel < 1024, z <= 64
  const int z_inv = (65536 + z - 1) / z;
  // lane l keeps the first uniform of hop (h & ~63) + l
  auto take_u1 = [&]() __attribute__((always_inline)) {
    if ((h & 63) == 0 && h + lane < a.n_pairs) u1c = a.U[2 * (h + lane)];
  };
  // k_tot and the selection: the first process whose cumulative rate
  // exceeds u1 k_tot; lane l sums the processes l per .. l per + per - 1
  // (the reference compares the cumulative sum of k / k_tot with u1: the
  // same choice but where u1 lies within an ulp of a boundary)
  auto select = [&]() __attribute__((always_inline)) {
    sel = nproc - 1;  // rounding left no cum > u1: the last one
    with_count_up<1, 10>(per, [&](auto n_per) __attribute__((always_inline)) {
      constexpr int kP = decltype(n_per)::value;
      double x[kP], ksum = 0.0;
#pragma unroll
      for (int i = 0; i < kP; ++i) {
        x[i] = kks[i * HopLds::kStride + lane];
        ksum = i == 0 ? x[0] : ksum + x[i];
      }
      const double incl = wave_incl_scan(ksum);
      k_tot = read_lane(incl, 63);
      const double thr = read_lane(u1c, int(h & 63)) * k_tot;
      double cum = dpp_f64<kDppWaveShr1, 0xf, true>(incl);
      // rates are not negative: a lane's running sums do not decrease, and
      // the count of those <= thr is the index of its first crossing
      int nb = 0;
#pragma unroll
      for (int i = 0; i < kP; ++i) {
        cum += x[i];
        nb += cum > thr ? 0 : 1;
      }
      const unsigned long long mask =
          __ballot(nb < kP && lane * kP + nb < nproc);
      if (mask) {
        const int src = __ffsll(static_cast<long long>(mask)) - 1;
        sel = src * kP + __builtin_amdgcn_readlane(nb, src);
      } else {
        ++noselect;
      }
    });
    m = (sel * z_inv) >> 16;
  };
  // target k of the mover's new site
  auto target = [&](int k) __attribute__((always_inline)) {
    if constexpr (kLook) return tt[sel * z + k];
    else return a.nbr2[int64_t(tgt[sel].x) * a.mz + k];
  };
  // the full sum of row x
  auto row_sum = [&](int2 x) __attribute__((always_inline)) {
    Dd r;
    int c = 0;
    for (; c + 8 <= nc; c += 8) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = entry(x, occ[c + u]);
#pragma unroll
      for (int u = 0; u < 8; ++u) dd_add_prod(r, cqs[c + u], v[u]);
    }
    for (; c < nc; ++c) dd_add_prod(r, cqs[c], entry(x, occ[c]));
    dd_norm(r);
    return r;
  };
  // a row's update by the hop: its entries at the mover's new and old site
  auto move = [](Dd& r, double q, double in, double out)
                  __attribute__((always_inline)) {
    dd_add_prod(r, q, in);
    dd_add_prod(r, -q, out);
    dd_norm(r);
  };

  if (wave < roles.process) {
    // ================================================ process wavefronts
    const bool pv = tid < nproc;
    const int pp = pv ? tid : 0;
    const int pk_at = (pp % per) * HopLds::kStride + pp / per;
    const int pc = pp / z, pj = pp - pc * z;
    const double pq = cqs[pc];
    // the site-dependent part of the process's rate: slot j of site s,
    // whose target is n.  Kept as loaded, so that nothing waits for these
    // loads before the next hop's rates need them.
    SlotRec r;
    double En, Es;
    auto load_inputs = [&](int s, int n) {
      r = a.rec[int64_t(s) * a.mz + pj];
      Es = a.pe[s].y;
      En = a.pe[n].y;
    };
    auto post = [&](int2 x) {  // what a selected process is read by
      tgt[pp] = x;
      pv3[3 * pp] = r.v[0];
      pv3[3 * pp + 1] = r.v[1];
      pv3[3 * pp + 2] = r.v[2];
    };
    const int s0 = occ[pc].x;
    int2 px = a.nbr2[int64_t(s0) * a.mz + pj];
    load_inputs(s0, px.x);
    Dd psi = row_sum(px);
    if (pv) post(px);
    __syncthreads();
    for (; h < due;) {
      take_u1();
      // ---- the rate; the mover's rows are new
      const bool mine = pc == m;
      const double fh = fresh[2 * pj], fl = fresh[2 * pj + 1];
      const double ps = psis[pc];
      psi.h = mine ? fh : psi.h;
      psi.l = mine ? fl : psi.l;
      {
        // products and sums rounded one by one, as NumPy forms them
#pragma clang fp contract(off)
        const double term01 = r.dphi + (psi.h - ps);
        const double g0 = 2 * pq * (term01 + pq * r.tself) + (En - Es);
        const double k = marcus_rate(g0, r.lam, r.i4l, r.vs, a.nkt, a.nu, ext);
        if (pv) {
          kks[pk_at] = k;
          dgs[pp] = g0;
        }
      }
      if (pv && mine) post(px);
      const int last = *over;
      lds_barrier();
      if (last) break;
      select();
      // ---- one round of loads
      int2 n = tgt[sel], s = occ[m];
      const double qm = cqs[m];
      const int2 tx = target(pj);
      n = uniform(n);
      s = uniform(s);
      const double an = entry(px, n), as = entry(px, s);
      // the mover's new process (its row comes with the next hop)
      if (pc == m) {
        px = tx;
        load_inputs(n.x, px.x);
      }
      move(psi, qm, an, as);
      if (pv && pp == sel) {
        box[0] = psi.h;
        box[1] = psi.l;
        psis[m] = psi.h;
      }
      ++h;
      lds_barrier();
    }
    return;
  }

  if (wave >= roles.process + roles.site) {
    // ================================================ helpers
    const int hw = wave - roles.process - roles.site;
    const int fc = lane & 15;
    // look-ahead load of this lane: target lk of the mover's new target lj
    const int lu = 64 * hw + lane;
    const bool la_on = kLook && lu < z * z;
    const int lj = la_on ? lu / z : 0;
    const int lk = la_on ? lu - lj * z : 0;
    int2 la = make_int2(0, 0);
    // a helper has the longest way from the selection to the barrier
    __builtin_amdgcn_s_setprio(3);
    // kF: carriers per lane whose sites and charges are kept here (the rest,
    // past 128, read from LDS)
    auto help = [&](auto n_f) __attribute__((always_inline)) {
      constexpr int kF = decltype(n_f)::value;
      int2 fo[kF];
      double fq[kF];
#pragma unroll
      for (int u = 0; u < kF; ++u) {
        const int c = fc + 16 * u;
        fo[u] = occ[c < nc ? c : 0];
        fq[u] = c < nc ? cqs[c] : 0.0;
      }
      __syncthreads();
      while (h < due) {
        take_u1();
        if (la_on && m >= 0) tt[(m * z + lj) * z + lk] = la;
        const int last = *over;
        lds_barrier();
        if (last) break;
        select();
        int2 n = tgt[sel];
        const int2 lx = kLook ? target(lj) : n;
        int k0 = 4 * hw;
        int2 fx = target(k0 + (lane >> 4) < z ? k0 + (lane >> 4) : 0);
        n = uniform(n);
#pragma unroll
        for (int u = 0; u < kF; ++u)
          if (fc + 16 * u == m) fo[u] = n;
        for (;;) {
          const int k = k0 + (lane >> 4);
          double e[kF];
#pragma unroll
          for (int u = 0; u < kF; ++u) e[u] = entry(fx, fo[u]);
          if (la_on && k0 == 4 * hw) la = a.nbr2[int64_t(lx.x) * a.mz + lk];
          Dd v;
#pragma unroll
          for (int u = 0; u < kF; ++u) dd_add_prod(v, fq[u], e[u]);
          if constexpr (kF == 8)
            for (int c = fc + 16 * kF; c < nc; c += 16)
              dd_add_prod(v, cqs[c], entry(fx, c == m ? n : occ[c]));
          dd_row_sum(v);
          if (fc == 0 && k < z) {
            fresh[2 * k] = v.h;
            fresh[2 * k + 1] = v.l;
          }
          k0 += 4 * roles.helper;
          if (k0 >= z) break;
          fx = target(k0 + (lane >> 4) < z ? k0 + (lane >> 4) : 0);
        }
        ++h;
        lds_barrier();
      }
    };
    if (nc <= 16)
      help(std::integral_constant<int, 1>{});
    else if (nc <= 32)
      help(std::integral_constant<int, 2>{});
    else if (nc <= 64)
      help(std::integral_constant<int, 4>{});
    else
      help(std::integral_constant<int, 8>{});
    return;
  }

  // ================================================== site wavefronts
  __builtin_amdgcn_s_setprio(1);
  const int sw = wave - roles.process;
  const int c = 64 * sw + lane;
  const bool own = c < nc;  // (lanes past n_c keep carrier 0's row)
  int2 sx = occ[own ? c : 0];
  Dd psi = row_sum(sx);
  double dsp[3] = {0.0, 0.0, 0.0}, bse[3] = {0.0, 0.0, 0.0},
         drf[3] = {0.0, 0.0, 0.0};
  if (own) {
    psis[c] = psi.h;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      dsp[k] = dv->disp[3 * c + k];
      bse[k] = dv->base[3 * c + k];
      drf[k] = dv->drift[3 * c + k];
    }
  }
  double t = sc0.t, energy = sc0.energy;
  int64_t start = sc0.start;
  bool stop = sc0.finished != 0;
  const double inv_dt = 1.0 / a.dt;
  double u2c = 0.0, luc = 0.0;  // second uniforms, as u1c
  // hop log of a block of 64 hops: lane l holds hop (h & ~63) + l
  double tlog = 0.0;
  int32_t plog = 0;
  auto flush_log = [&](int64_t block, int count) {
    if (sw == 0 && lane < count) {
      if (a.hop_time) a.hop_time[block + lane] = tlog;
      if (a.hop_proc) a.hop_proc[block + lane] = plog;
    }
  };
  // A hop that spans several path rows: with up to 32 carriers lane l writes
  // carrier l mod n_c's entries of every (64 / n_c)-th of them.  (With each
  // lane writing its own carrier's alone, 1 carrier with 16 slots and 301 rows
  // in 3 hops took 10.5 us a hop, the 256 threads of the kernel before 6.6,
  // now 6.7; 4 slots and 67000 rows a hop 6500 us, now 297.)
  const int copies = nc <= 32 ? 64 / nc : 1;
  const int copy = lane / (nc <= 32 ? nc : 64), cc = lane - copy * nc;
  // clock, energy, log and path rows of hop h
  auto tick = [&](double g_sel) {
    const int hl = int(h & 63);
    int64_t end;
    if (read_lane(u2c, hl) > 0.0) {
      t -= read_lane(luc, hl) / k_tot;
      // path step int(t / dt) of the correctly rounded quotient: below 1e6,
      // t (1/dt) is within 4e-10 of it, so more than 1e-9 away from an
      // integer its integer part is the quotient's; otherwise divide
      const double qf = t * inv_dt, fl = floor(qf), fr = qf - fl;
      if (fr > 1e-9 && fr < 1.0 - 1e-9 && qf < 1.0e6) {
        end = int(fl);
      } else {
        const double qd = t / a.dt;
        end = qd < 9.0e18 ? int64_t(qd) : a.P;
      }
    } else {
      t = INFINITY;
      end = a.P;
    }
    energy += g_sel;
    tlog = lane == hl ? t : tlog;
    plog = lane == hl ? sel : plog;
    if (hl == 63) flush_log(h - 63, 64);
    if (end < start + 1) return;
    const int64_t dp_hi = min(end, a.P);
    if (end >= a.P) end = a.P;
    if (sw == 0) {
      for (int64_t r = start + lane; r < dp_hi; r += 64) a.dpath[r] = g_sel;
      for (int64_t r = start + lane; r < end; r += 64) a.epath[r] = energy;
    }
    const int w = 3 * nc;
    if (copies > 1 && end - start >= 4) {
      double v[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double x = bse[k] + dsp[k];
        v[k] = from32(__builtin_amdgcn_ds_bpermute(4 * cc, lo32(x)),
                      __builtin_amdgcn_ds_bpermute(4 * cc, hi32(x)));
      }
      if (copy < copies)
        for (int64_t r = start + copy; r < end; r += copies)
#pragma unroll
          for (int k = 0; k < 3; ++k) a.rows[r * w + 3 * cc + k] = v[k];
    } else if (own) {
      for (int64_t r = start; r < end; ++r)
#pragma unroll
        for (int k = 0; k < 3; ++k)
          a.rows[r * w + 3 * c + k] = bse[k] + dsp[k];
    }
    if (own) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        bse[k] += dsp[k];
        dsp[k] = 0.0;
      }
    }
    start = end;
    // loop condition of the reference: continue while end < P
    stop = end >= a.P;
    if (stop && c == 0) *over = 1;
  };
  __syncthreads();
  while (h < due) {
    take_u1();
    if ((h & 63) == 0 && h + lane < a.n_pairs) {
      u2c = a.U[2 * (h + lane) + 1];
      luc = a.LU[h + lane];
    }
    // ---- what the last hop left
    if (c == m) {
      psi.h = box[0];
      psi.l = box[1];
      occ[m] = sx;
    }
    lds_barrier();
    if (stop) break;
    select();
    int2 n = tgt[sel], s = occ[m];
    const double qm = cqs[m];
    const double g_sel = dgs[sel];
    const double k_sel = kks[(sel % per) * HopLds::kStride + sel / per];
    double v[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] = pv3[3 * sel + k];
    n = uniform(n);
    s = uniform(s);
    const double bn = entry(sx, n), bs = entry(sx, s);
    if (c == m) {
#pragma clang fp contract(off)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        dsp[k] = dsp[k] + v[k];
        if (a.field_on) drf[k] = drf[k] + v[k] * k_sel;
      }
    }
    tick(g_sel);  // while the gathers are in flight
    move(psi, qm, bn, bs);
    if (c == m)  // continued from the row of n, see box
      sx = n;
    else if (own)
      psis[c] = psi.h;
    ++h;
    lds_barrier();
  }
  // ---- write the state back
  flush_log(h & ~int64_t(63), int(h & 63));
  if (own) {
    dv->occ[c] = sx.x;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      dv->disp[3 * c + k] = dsp[k];
      dv->base[3 * c + k] = bse[k];
      dv->drift[3 * c + k] = drf[k];
    }
  }
  if (c == 0) {
    KmcScalars o = sc0;
    o.t = t;
    o.energy = energy;
    o.start = start;
    o.hops = sc0.hops + h;
    o.no_select = noselect;
    if (stop) o.finished = 1;
    *dv->sc = o;
    // ended by its path or its hop count, or more uniforms are needed
    status[0] = stop || (a.max_hops > 0 && o.hops >= a.max_hops) ? 0 : 1;
    status[1] = int32_t(h);
  }
}

// Scratch of pycd_kmc_advance_static: log(u2) of up to kStaticPairs uniform
// pairs, then the hop loop's two status words.  One copy per device (every
// device the library runs on holds it until the process ends); host code
// reaches it only through the address hipGetSymbolAddress returns for the
// device (pycd_ctx_create resolves it once per device).  Calls that overlap
// on one device share it and race.
constexpr int64_t kStaticPairs = int64_t(1) << 20;
__device__ __align__(256) double scratch[kStaticPairs + 32];

__global__ void reset_status(int32_t* __restrict__ status) {
  status[0] = -1;
  status[1] = 0;
}

// phi_L[i] = sum_j A[i, j] q_L[j]: one wavefront per row.
__global__ void __launch_bounds__(256)
row_dot_kernel(const double* __restrict__ A, const double* __restrict__ q,
               int64_t N, double* __restrict__ out) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int64_t i = int64_t(blockIdx.x) * 4 + wave; i < N;
       i += int64_t(gridDim.x) * 4) {
    const double* row = A + i * N;
    double acc = 0.0;
    for (int64_t j = lane; j < N; j += 64) acc = fma(row[j], q[j], acc);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
    if (lane == 0) out[i] = acc;
  }
}

// tself[s, j] = A[s, s] - A[s, nbr(s, j)] for valid slots.
__global__ void self_term_kernel(const double* __restrict__ A,
                                 const int32_t* __restrict__ nbr, int64_t N,
                                 int max_z, double* __restrict__ tself) {
  const int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= N * max_z) return;
  const int64_t s = idx / max_z;
  const int n = nbr[idx];
  tself[idx] = n >= 0 ? A[s * N + s] - A[s * N + n] : 0.0;
}

// Lattice part of the potential difference of each hop, the reference's
// q . (A[n, :] - A[s, :]) restricted to the lattice charges: every product
// q_L[y] (A[n, y] - A[s, y]) rounded as NumPy forms it, their sum kept as
// an unevaluated pair (hi, lo) (Knuth's TwoSum) and rounded once at the
// end.  Forming it as phi_L[n] - phi_L[s] instead would carry about an ulp
// of phi_L, a sum of order 10 Ha, into every rate.  One wavefront per
// (site, slot); 0 for empty slots.
__device__ inline void two_sum(double a, double b, double& s, double& e) {
#pragma clang fp contract(off)
  s = a + b;
  const double bb = s - a;
  e = (a - (s - bb)) + (b - bb);
}

__global__ void __launch_bounds__(256)
slot_dphi_kernel(const double* __restrict__ A, const double* __restrict__ q,
                 const int32_t* __restrict__ nbr, int64_t N, int max_z,
                 double* __restrict__ dphi) {
#pragma clang fp contract(off)
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t NM = N * max_z;
  for (int64_t k = int64_t(blockIdx.x) * 4 + wave; k < NM;
       k += int64_t(gridDim.x) * 4) {
    const int n = nbr[k];
    if (n < 0) {
      if (lane == 0) dphi[k] = 0.0;
      continue;
    }
    const double* rs = A + (k / max_z) * N;
    const double* rn = A + int64_t(n) * N;
    double hi = 0.0, lo = 0.0;
    for (int64_t y = lane; y < N; y += 64) {
      const double p = q[y] * (rn[y] - rs[y]);
      double e;
      two_sum(hi, p, hi, e);
      lo += e;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const double h2 = __shfl_xor(hi, off, 64);
      const double l2 = __shfl_xor(lo, off, 64);
      double e;
      two_sum(hi, h2, hi, e);
      lo = lo + l2 + e;
    }
    if (lane == 0) dphi[k] = hi + lo;
  }
}

// Initial energy pieces: e[0] = q_L . phi_L is precomputed on the host side
// of the session; this kernel adds the carrier terms
// 2 sum_c q_c phi_L[occ_c] + sum_{c,c'} q_c q_c' A[occ_c, occ_c'].
__global__ void carrier_energy_kernel(const double* __restrict__ A,
                                      const double* __restrict__ phiL,
                                      const double* __restrict__ cq,
                                      const int32_t* __restrict__ occ,
                                      int nc, int64_t N,
                                      double* __restrict__ out) {
  __shared__ double part[256];
  double acc = 0.0;
  for (int c = threadIdx.x; c < nc; c += blockDim.x) {
    const double* row = A + int64_t(occ[c]) * N;
    double inner = 0.0;
    for (int c2 = 0; c2 < nc; ++c2) inner = fma(cq[c2], row[occ[c2]], inner);
    acc += cq[c] * (2.0 * phiL[occ[c]] + inner);
  }
  part[threadIdx.x] = acc;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if (int(threadIdx.x) < w) part[threadIdx.x] += part[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = part[0];
}

__global__ void dot_kernel(const double* __restrict__ a,
                           const double* __restrict__ b, int64_t n,
                           double* __restrict__ out) {
  __shared__ double part[256];
  double acc = 0.0;
  for (int64_t k = threadIdx.x; k < n; k += blockDim.x)
    acc = fma(a[k], b[k], acc);
  part[threadIdx.x] = acc;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if (int(threadIdx.x) < w) part[threadIdx.x] += part[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = part[0];
}

}  // namespace pycd

using namespace pycd;

struct pycd_kmc {
  pycd_ctx* ctx = nullptr;
  pycd_kmc_problem pb{};
  DevBuf<double> A, phiL, dphi, vec, lam, vab, tself, E, cq, qL;
  DevBuf<int32_t> nbr, occ, status;
  DevBuf<double> disp, base, drift, rows, epath, dpath, tmp;
  DevBuf<KmcScalars> sc;
  DevBuf<double> ubuf, tbuf, lubuf;
  DevBuf<int32_t> pbuf;
  // periodic supercell: cell-0 rows of the table and packed site codes
  bool compact = false;
  Geo geo{};
  DevBuf<double> Ac;
  DevBuf<uint32_t> pk, nbr_pk;
  // slot records, (phi_L, E) per site, targets with their codes, the device
  // copy of the kernel's state pointers
  DevBuf<SlotRec> rec;
  DevBuf<double2> pe;
  DevBuf<int2> nbr2;
  DevBuf<KmcDev> dev;
  double qLAqL = 0.0;
  // the hop loop's roles, its look-ahead and its LDS
  HopRoles hop_roles{};
  int hop_look = 0;
  size_t hop_smem = 0;
  // PYCD_KMC_WAVE may be named, and what was named
  bool wave_ok = false;
  size_t wave_bytes = 0;
  int32_t variant = PYCD_KMC_AUTO;
  bool begun = false;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  double last_ms = 0.0;
  ~pycd_kmc() {
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
  }
};

namespace {

int check_problem(pycd_ctx* ctx, const pycd_kmc_problem* pb) {
  if (!pb) return fail(ctx, PYCD_ERR_ARG, "null problem");
  if (pb->n_sites <= 0 || pb->n_sites > (int64_t(1) << 31) - 1)
    return fail(ctx, PYCD_ERR_ARG, "bad n_sites");
  if (pb->n_carriers <= 0 || pb->z <= 0 || pb->z > 64 || pb->max_z < pb->z)
    return fail(ctx, PYCD_ERR_ARG, "bad carrier/slot counts (z <= 64)");
  if (!pb->table || !pb->lattice_q || !pb->nbr_site || !pb->nbr_vec ||
      !pb->nbr_lambda || !pb->nbr_vab || !pb->site_energy || !pb->carrier_q)
    return fail(ctx, PYCD_ERR_ARG, "null table pointer");
  if (!(pb->time_interval > 0) || pb->n_path < 1 || !(pb->kT > 0))
    return fail(ctx, PYCD_ERR_ARG, "bad time grid or temperature");
  return PYCD_OK;
}

// phi_lattice = A q_lattice, the lattice part of every hop's potential
// difference and q_lattice^T A q_lattice from the resident table and
// lattice charges.
hipError_t lattice_terms(pycd_kmc* s) {
  hipStream_t st = s->ctx->stream;
  const int64_t N = s->pb.n_sites;
  const int blocks = int(std::min<int64_t>((N + 3) / 4, 8192));
  row_dot_kernel<<<blocks, 256, 0, st>>>(s->A.ptr, s->qL.ptr, N, s->phiL.ptr);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t NM = N * s->pb.max_z;
  slot_dphi_kernel<<<int(std::min<int64_t>((NM + 3) / 4, 16384)), 256, 0,
                     st>>>(s->A.ptr, s->qL.ptr, s->nbr.ptr, N, s->pb.max_z,
                           s->dphi.ptr);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  dot_kernel<<<1, 256, 0, st>>>(s->qL.ptr, s->phiL.ptr, N, s->tmp.ptr);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  e = hipMemcpyAsync(&s->qLAqL, s->tmp.ptr, sizeof(double),
                     hipMemcpyDeviceToHost, st);
  if (e != hipSuccess) return e;
  return hipStreamSynchronize(st);
}

// Largest |A[i, j] - Ac[sub(i), rel(i, j)]| over the full table, as the bit
// pattern of a non-negative double (ordered like the values).  One
// workgroup of 256 per 4 rows.
__global__ void __launch_bounds__(256)
periodic_gap(const double* __restrict__ A, const double* __restrict__ Ac,
             int64_t N, Geo g, unsigned long long* __restrict__ worst) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const GeoPk gp = geo_pk(g);
  double m = 0.0;
  for (int64_t i = int64_t(blockIdx.x) * 4 + wave; i < N;
       i += int64_t(gridDim.x) * 4) {
    const uint32_t a = site_pack(uint32_t(i), g);
    const RowKey key = row_key(a, gp);
    const double* row = A + i * N;
    const double* crow = Ac + int64_t(a >> 24) * N;
    for (int64_t j = lane; j < N; j += 64)
      m = nan_max(m, fabs(row[j] - crow[rel_col(key, site_pack(uint32_t(j), g),
                                                 gp)]));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    m = nan_max(m, __shfl_xor(m, off, 64));
  if (lane == 0)
    atomicMax(worst, static_cast<unsigned long long>(__double_as_longlong(m)));
}

// A periodic supercell's table is translation-invariant: the hop loop can
// read the n_unit rows of cell 0 (L2-resident) instead of the full table.
// Used only when the cell shape is given, fits the packed site codes, the
// full table is above kCellRowsFrom bytes, and every entry of the full
// table equals its cell-0 translate to kTranslationTol of the table's
// scale (a NaN anywhere fails);
// otherwise the loop reads the full table.  Smaller tables stay in the
// caches whole, and there the two are near each other (768 sites, 8 and 32
// carriers: 1.12 and 1.28 us per hop on the full table, 1.07 and 1.29 on
// cell-0 rows); above, the full table's misses show (2592 sites, 16
// carriers: 1.26 and 1.07; 6144 sites: 1.39 and 1.08).
constexpr int64_t kCellRowsFrom = int64_t(32) << 20;
hipError_t compact_setup(pycd_kmc* s, const std::vector<int32_t>& nb) {
  const pycd_kmc_problem& pb = s->pb;
  const int64_t N = pb.n_sites;
  const int mz = pb.max_z;
  const Geo g{pb.cells[0], pb.cells[1], pb.cells[2], pb.n_unit};
  s->compact = false;
  if (g.nx < 1 || g.ny < 1 || g.nz < 1 || g.nu < 1 || g.nx > 255 ||
      g.ny > 255 || g.nz > 255 || g.nu > 255 ||
      int64_t(g.nx) * g.ny * g.nz * g.nu != N || N >= (int64_t(1) << 24) ||
      int64_t(g.ny) * g.nz * g.nu >= 65536 ||
      N * N * int64_t(sizeof(double)) <= kCellRowsFrom)
    return hipSuccess;
  hipStream_t st = s->ctx->stream;
  std::vector<uint32_t> pk(N), npk(size_t(N) * mz, 0u);
  for (int64_t i = 0; i < N; ++i) pk[i] = site_pack(uint32_t(i), g);
  for (size_t k = 0; k < npk.size(); ++k)
    if (nb[k] >= 0) npk[k] = pk[nb[k]];
  const size_t rows = size_t(g.nu) * size_t(N);
  hipError_t e;
  if ((e = s->pk.alloc(N)) != hipSuccess) return e;
  if ((e = s->nbr_pk.alloc(npk.size())) != hipSuccess) return e;
  if ((e = s->Ac.alloc(rows)) != hipSuccess) return e;
  if ((e = upload(s->pk.ptr, pk.data(), pk.size(), st)) != hipSuccess) return e;
  if ((e = upload(s->nbr_pk.ptr, npk.data(), npk.size(), st)) != hipSuccess)
    return e;
  if ((e = hipMemcpyAsync(s->Ac.ptr, s->A.ptr, rows * sizeof(double),
                          hipMemcpyDeviceToDevice, st)) != hipSuccess)
    return e;
  DevBuf<unsigned long long> worst;
  if ((e = worst.alloc(1)) != hipSuccess) return e;
  const unsigned long long zero = 0;
  if ((e = upload(worst.ptr, &zero, 1, st)) != hipSuccess) return e;
  periodic_gap<<<int(std::min<int64_t>((N + 3) / 4, 8192)), 256, 0, st>>>(
      s->A.ptr, s->Ac.ptr, N, g, worst.ptr);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  unsigned long long bits = 0;
  std::vector<double> c0(rows);
  if ((e = hipMemcpyAsync(&bits, worst.ptr, 8, hipMemcpyDeviceToHost, st)) !=
      hipSuccess)
    return e;
  if ((e = hipMemcpyAsync(c0.data(), s->Ac.ptr, rows * sizeof(double),
                          hipMemcpyDeviceToHost, st)) != hipSuccess)
    return e;
  if ((e = hipStreamSynchronize(st)) != hipSuccess) return e;
  double gap, scale = 0.0;
  std::memcpy(&gap, &bits, 8);
  for (double v : c0) scale = std::max(scale, std::fabs(v));
  if (gap <= kTranslationTol * scale) {
    s->compact = true;
    s->geo = g;
  } else {
    s->Ac.release();
    s->pk.release();
    s->nbr_pk.release();
  }
  return hipSuccess;
}

// Slot records, targets and (phi_L, E) pairs of every site, from the slot
// tables and the lattice terms.
hipError_t pack_hop_inputs(pycd_kmc* s) {
  hipStream_t st = s->ctx->stream;
  const int64_t N = s->pb.n_sites;
  const int64_t NM = N * s->pb.max_z;
  const double* f = s->pb.field;
  const bool field_on = f[0] != 0.0 || f[1] != 0.0 || f[2] != 0.0;
  pack_slot_records<<<int((NM + 255) / 256), 256, 0, st>>>(
      NM, s->tself.ptr, s->dphi.ptr, s->lam.ptr, s->vab.ptr, s->vec.ptr,
      s->nbr.ptr, s->compact ? s->nbr_pk.ptr : nullptr, f[0], f[1], f[2],
      field_on ? 1 : 0, s->rec.ptr, s->nbr2.ptr);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  pack_site_pe<<<int((N + 255) / 256), 256, 0, st>>>(N, s->phiL.ptr,
                                                     s->E.ptr, s->pe.ptr);
  return hipGetLastError();
}

// The sessions for which PYCD_KMC_WAVE can be named, a line of the interface:
// few carriers, and the bytes of every table entry that their rates read
// (those of carrier pairs in groups of 4 for n_c z + n_c rows, psi and
// charges, sites with codes, z z targets per carrier) within a workgroup's
// LDS.  0 for the others.  Both names run the same kernel.
size_t rate_entry_bytes(int nc, int z) {
  const int nproc = nc * z;
  if (nc > 64 || nproc > 256 || z > 8) return 0;
  const size_t ncp = (((size_t(nc) + 1) / 2) + 3) & ~size_t(3);
  return 16 * ncp * (nproc + nc) + sizeof(double) * (size_t(nc) + 2 * ncp) +
         sizeof(int32_t) * (2 * size_t(nc) + 2 * size_t(nproc) * z);
}

}  // namespace

extern "C" int pycd_kmc_create(pycd_ctx* ctx, const pycd_kmc_problem* pb,
                               pycd_kmc** out) {
  if (!ctx || !out) return PYCD_ERR_ARG;
  *out = nullptr;
  int rc = check_problem(ctx, pb);
  if (rc) return rc;
  DeviceGuard guard(ctx->device);
  const int64_t N = pb->n_sites;
  const int nc = pb->n_carriers, z = pb->z, mz = pb->max_z;
  if (!session_fits(nc, z))
    return fail(ctx, PYCD_ERR_ARG,
                "n_c=%d, z=%d: a session takes n_c (104 z + 88) up to %lld",
                nc, z, (long long)kSessionMost);
  // Host-side validation of the slot table (every index the kernel reads).
  std::vector<int32_t> nb(size_t(N) * mz);
  {
    if (is_device_ptr(pb->nbr_site)) {
      PYCD_HIP(ctx, hipMemcpy(nb.data(), pb->nbr_site, nb.size() * 4,
                              hipMemcpyDeviceToHost));
    } else {
      std::memcpy(nb.data(), pb->nbr_site, nb.size() * 4);
    }
    for (size_t k = 0; k < nb.size(); ++k)
      if (nb[k] < -1 || nb[k] >= N)
        return fail(ctx, PYCD_ERR_ARG, "nbr_site[%zu]=%d out of range", k,
                    nb[k]);
    // Closure: a hopping site (slot 0 valid) has z valid slots and every
    // target is itself a hopping site, so a carrier never reaches a site
    // whose slot rows the kernel cannot read.
    for (int64_t s = 0; s < N; ++s) {
      const int32_t* row = nb.data() + size_t(s) * mz;
      if (row[0] < 0) continue;
      for (int j = 0; j < z; ++j) {
        if (row[j] < 0)
          return fail(ctx, PYCD_ERR_ARG, "site %lld has fewer than %d slots",
                      (long long)s, z);
        if (nb[size_t(row[j]) * mz] < 0)
          return fail(ctx, PYCD_ERR_ARG,
                      "slot %d of site %lld targets non-hopping site %d", j,
                      (long long)s, row[j]);
      }
    }
  }
  pycd_kmc* s = new (std::nothrow) pycd_kmc();
  if (!s) return PYCD_ERR_NOMEM;
  s->ctx = ctx;
  s->pb = *pb;
  hipStream_t st = ctx->stream;
  auto bail = [&](int code) {
    delete s;
    return code;
  };
#define S_HIP(expr)                                                         \
  do {                                                                      \
    hipError_t e_ = (expr);                                                 \
    if (e_ != hipSuccess)                                                   \
      return bail(fail(ctx, PYCD_ERR_HIP, "%s: %s", #expr,                  \
                       hipGetErrorString(e_)));                             \
  } while (0)
  const size_t NM = size_t(N) * mz;
  const int64_t P = pb->n_path;
  S_HIP(s->A.alloc(size_t(N) * N));
  S_HIP(s->phiL.alloc(N));
  S_HIP(s->dphi.alloc(NM));
  S_HIP(s->qL.alloc(N));
  S_HIP(s->nbr.alloc(NM));
  S_HIP(s->vec.alloc(NM * 3));
  S_HIP(s->lam.alloc(NM));
  S_HIP(s->vab.alloc(NM));
  S_HIP(s->tself.alloc(NM));
  S_HIP(s->E.alloc(N));
  S_HIP(s->cq.alloc(nc));
  S_HIP(s->occ.alloc(nc));
  S_HIP(s->status.alloc(2));
  S_HIP(s->disp.alloc(3 * nc));
  S_HIP(s->base.alloc(3 * nc));
  S_HIP(s->drift.alloc(3 * nc));
  S_HIP(s->rows.alloc(size_t(P) * 3 * nc));
  S_HIP(s->epath.alloc(P));
  S_HIP(s->dpath.alloc(P));
  S_HIP(s->tmp.alloc(2));
  S_HIP(s->sc.alloc(1));
  S_HIP(upload(s->A.ptr, pb->table, size_t(N) * N, st));
  S_HIP(upload(s->qL.ptr, pb->lattice_q, N, st));
  S_HIP(upload(s->nbr.ptr, pb->nbr_site, NM, st));
  S_HIP(upload(s->vec.ptr, pb->nbr_vec, NM * 3, st));
  S_HIP(upload(s->lam.ptr, pb->nbr_lambda, NM, st));
  S_HIP(upload(s->vab.ptr, pb->nbr_vab, NM, st));
  S_HIP(upload(s->E.ptr, pb->site_energy, N, st));
  S_HIP(upload(s->cq.ptr, pb->carrier_q, nc, st));
  self_term_kernel<<<int((NM + 255) / 256), 256, 0, st>>>(s->A.ptr, s->nbr.ptr,
                                                         N, mz, s->tself.ptr);
  S_HIP(hipGetLastError());
  S_HIP(lattice_terms(s));
  S_HIP(compact_setup(s, nb));
  S_HIP(s->rec.alloc(NM));
  S_HIP(s->nbr2.alloc(NM));
  S_HIP(s->pe.alloc(size_t(N)));
  S_HIP(s->dev.alloc(1));
  S_HIP(pack_hop_inputs(s));
  {
    int lds_max = 0;
    S_HIP(hipDeviceGetAttribute(&lds_max,
                                hipDeviceAttributeMaxSharedMemoryPerBlock,
                                ctx->device));
    s->wave_bytes = rate_entry_bytes(nc, z);
    s->hop_roles = HopRoles(nc, z);
    HopLds hl{nc, z, z * z <= 64 * s->hop_roles.helper ? 1 : 0};
    if (hl.bytes() + 512 > size_t(lds_max)) hl.look = 0;
    s->hop_look = hl.look;
    s->hop_smem = hl.bytes();
    // (512 bytes of 2^(j/64) are beside the dynamic part)
    const double tab_bytes = 8.0 * double(s->compact ? s->geo.nu : N) * N;
    s->wave_ok = s->wave_bytes > 0 && s->wave_bytes + 512 <= size_t(lds_max) &&
                 tab_bytes < 4294967296.0;
  }
#undef S_HIP
  *out = s;
  return PYCD_OK;
}

extern "C" int pycd_kmc_set_variant(pycd_kmc* s, int32_t variant) {
  if (!s) return PYCD_ERR_ARG;
  if (variant != PYCD_KMC_AUTO && variant != PYCD_KMC_WORKGROUP &&
      variant != PYCD_KMC_WAVE)
    return fail(s->ctx, PYCD_ERR_ARG, "unknown kernel variant %d", variant);
  if (variant == PYCD_KMC_WAVE && !s->wave_ok)
    return fail(s->ctx, PYCD_ERR_ARG,
                "PYCD_KMC_WAVE is for n_c <= 64, n_c z <= 256, z <= 8, the "
                "entries its rates read (%zu B) within a workgroup's LDS and "
                "a table below 4 GiB (n_c=%d, z=%d)",
                s->wave_bytes, s->pb.n_carriers, s->pb.z);
  s->variant = variant;
  return PYCD_OK;
}

extern "C" int pycd_kmc_variant(const pycd_kmc* s, int32_t* variant) {
  if (!s || !variant) return PYCD_ERR_ARG;
  const bool wave = s->variant == PYCD_KMC_WAVE ||
                    (s->variant == PYCD_KMC_AUTO && s->wave_ok);
  *variant = wave ? PYCD_KMC_WAVE : PYCD_KMC_WORKGROUP;
  return PYCD_OK;
}

extern "C" int pycd_kmc_table_rows(const pycd_kmc* s, int64_t* rows) {
  if (!s || !rows) return PYCD_ERR_ARG;
  *rows = s->compact ? int64_t(s->geo.nu) : s->pb.n_sites;
  return PYCD_OK;
}

extern "C" int pycd_kmc_set_sites(pycd_kmc* s, const double* lattice_q,
                                  const double* site_energy) {
  if (!s) return PYCD_ERR_ARG;
  pycd_ctx* ctx = s->ctx;
  if (!lattice_q || !site_energy)
    return fail(ctx, PYCD_ERR_ARG, "null lattice_q or site_energy");
  DeviceGuard guard(ctx->device);
  hipStream_t st = ctx->stream;
  const int64_t N = s->pb.n_sites;
  // the next trajectory starts from these sites: a running one is ended
  s->begun = false;
  PYCD_HIP(ctx, upload(s->qL.ptr, lattice_q, N, st));
  PYCD_HIP(ctx, upload(s->E.ptr, site_energy, N, st));
  PYCD_HIP(ctx, lattice_terms(s));
  PYCD_HIP(ctx, pack_hop_inputs(s));
  return PYCD_OK;
}

extern "C" void pycd_kmc_destroy(pycd_kmc* s) {
  if (!s) return;
  DeviceGuard guard(s->ctx->device);
  (void)hipStreamSynchronize(s->ctx->stream);
  delete s;
}

extern "C" int pycd_kmc_begin(pycd_kmc* s, const int64_t* occupancy,
                              double ewald_neut) {
  if (!s || !occupancy) return PYCD_ERR_ARG;
  pycd_ctx* ctx = s->ctx;
  DeviceGuard guard(ctx->device);
  const pycd_kmc_problem& pb = s->pb;
  const int nc = pb.n_carriers;
  std::vector<int32_t> occ(nc);
  {
    // occupancy comes from the host API; validate every site.
    std::vector<int32_t> nb(size_t(pb.n_sites) * pb.max_z);
    PYCD_HIP(ctx, hipMemcpy(nb.data(), s->nbr.ptr, nb.size() * 4,
                            hipMemcpyDeviceToHost));
    for (int c = 0; c < nc; ++c) {
      const int64_t v = occupancy[c];
      if (v < 0 || v >= pb.n_sites)
        return fail(ctx, PYCD_ERR_ARG, "occupancy[%d]=%lld out of range", c,
                    (long long)v);
      for (int j = 0; j < pb.z; ++j)
        if (nb[size_t(v) * pb.max_z + j] < 0)
          return fail(ctx, PYCD_ERR_ARG,
                      "carrier %d sits on site %lld with fewer than z=%d hop "
                      "slots",
                      c, (long long)v, pb.z);
      occ[c] = int32_t(v);
    }
  }
  hipStream_t st = ctx->stream;
  const int64_t P = pb.n_path;
  PYCD_HIP(ctx, hipMemcpyAsync(s->occ.ptr, occ.data(), 4 * nc,
                               hipMemcpyHostToDevice, st));
  PYCD_HIP(ctx, hipMemsetAsync(s->disp.ptr, 0, 24 * nc, st));
  PYCD_HIP(ctx, hipMemsetAsync(s->base.ptr, 0, 24 * nc, st));
  PYCD_HIP(ctx, hipMemsetAsync(s->drift.ptr, 0, 24 * nc, st));
  PYCD_HIP(ctx, hipMemsetAsync(s->rows.ptr, 0, 24 * size_t(nc) * P, st));
  PYCD_HIP(ctx, hipMemsetAsync(s->epath.ptr, 0, 8 * size_t(P), st));
  PYCD_HIP(ctx, hipMemsetAsync(s->dpath.ptr, 0, 8 * size_t(P), st));
  carrier_energy_kernel<<<1, 256, 0, st>>>(s->A.ptr, s->phiL.ptr, s->cq.ptr,
                                          s->occ.ptr, nc, pb.n_sites,
                                          s->tmp.ptr);
  PYCD_HIP(ctx, hipGetLastError());
  double carrier_part = 0.0;
  PYCD_HIP(ctx, hipMemcpyAsync(&carrier_part, s->tmp.ptr, sizeof(double),
                               hipMemcpyDeviceToHost, st));
  PYCD_HIP(ctx, hipStreamSynchronize(st));
  KmcScalars sc{};
  sc.t = 0.0;
  sc.energy = ewald_neut + (s->qLAqL + carrier_part);
  sc.start = 1;
  sc.hops = 0;
  sc.finished = P <= 1 ? 1 : 0;
  sc.no_select = 0;
  PYCD_HIP(ctx, hipMemcpyAsync(s->sc.ptr, &sc, sizeof(sc),
                               hipMemcpyHostToDevice, st));
  PYCD_HIP(ctx, hipMemcpyAsync(s->epath.ptr, &sc.energy, sizeof(double),
                               hipMemcpyHostToDevice, st));
  PYCD_HIP(ctx, hipStreamSynchronize(st));
  s->begun = true;
  return PYCD_OK;
}

namespace {

template <bool kCompact, bool kLook>
hipError_t launch_hop_t(const pycd_kmc* s, hipStream_t st, const HopArgs& args,
                        int32_t* status) {
  if (s->hop_smem > 65536) {
    hipError_t e = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&kmc_hop_kernel<kCompact, kLook>),
        hipFuncAttributeMaxDynamicSharedMemorySize, int(s->hop_smem));
    if (e != hipSuccess) return e;
  }
  kmc_hop_kernel<kCompact, kLook>
      <<<1, s->hop_roles.threads(), s->hop_smem, st>>>(args, s->dev.ptr,
                                                       s->hop_roles, status);
  return hipGetLastError();
}

hipError_t launch_hop(const pycd_kmc* s, hipStream_t st, const HopArgs& args,
                      int32_t* status) {
  if (!s->hop_roles.fit(s->pb.n_carriers, s->pb.z)) return hipErrorInvalidValue;
  if (s->compact)
    return s->hop_look ? launch_hop_t<true, true>(s, st, args, status)
                       : launch_hop_t<true, false>(s, st, args, status);
  return s->hop_look ? launch_hop_t<false, true>(s, st, args, status)
                     : launch_hop_t<false, false>(s, st, args, status);
}

}  // namespace

namespace pycd {

int hop_loop(pycd_kmc* s, const double* dU, double* LU, int32_t* status_dev,
             int64_t n_pairs, int64_t max_hops, double* dT, int32_t* dP,
             bool timed, int64_t* made);

// Device address of `scratch` on `device` (made current by the caller),
// resolved once per device and kept.
int kmc_static_scratch(int device, double** out) {
  static std::mutex mu;
  static std::vector<double*> addr;
  std::lock_guard<std::mutex> lock(mu);
  if (device < 0) return PYCD_ERR_ARG;
  if (addr.size() <= size_t(device)) addr.resize(size_t(device) + 1, nullptr);
  if (!addr[device]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p)
      return PYCD_ERR_HIP;
    addr[device] = static_cast<double*>(p);
  }
  *out = addr[device];
  return PYCD_OK;
}

}  // namespace pycd

extern "C" int pycd_kmc_advance(pycd_kmc* s, const double* uniforms,
                                int64_t n_pairs, int64_t max_hops,
                                double* hop_time, int32_t* hop_proc,
                                int64_t* hops_out) {
  if (!s) return PYCD_ERR_ARG;
  pycd_ctx* ctx = s->ctx;
  if (!s->begun) return fail(ctx, PYCD_ERR_STATE, "pycd_kmc_begin not called");
  if (n_pairs < 0 || (n_pairs > 0 && !uniforms))
    return fail(ctx, PYCD_ERR_ARG, "bad uniform buffer");
  if (n_pairs > (int64_t(1) << 30))
    return fail(ctx, PYCD_ERR_ARG, "at most 2^30 uniform pairs per call");
  DeviceGuard guard(ctx->device);
  hipStream_t st = ctx->stream;
  const double* dU = uniforms;
  if (n_pairs > 0 && !is_device_ptr(uniforms)) {
    if (s->ubuf.count < size_t(2 * n_pairs))
      PYCD_HIP(ctx, s->ubuf.alloc(size_t(2 * n_pairs)));
    PYCD_HIP(ctx, hipMemcpyAsync(s->ubuf.ptr, uniforms, 16 * size_t(n_pairs),
                                 hipMemcpyHostToDevice, st));
    dU = s->ubuf.ptr;
  }
  double* dT = hop_time;
  int32_t* dP = hop_proc;
  const bool t_host = hop_time && !is_device_ptr(hop_time);
  const bool p_host = hop_proc && !is_device_ptr(hop_proc);
  if (t_host) {
    if (s->tbuf.count < size_t(n_pairs))
      PYCD_HIP(ctx, s->tbuf.alloc(size_t(std::max<int64_t>(n_pairs, 1))));
    dT = s->tbuf.ptr;
  }
  if (p_host) {
    if (s->pbuf.count < size_t(n_pairs))
      PYCD_HIP(ctx, s->pbuf.alloc(size_t(std::max<int64_t>(n_pairs, 1))));
    dP = s->pbuf.ptr;
  }
  if (s->lubuf.count < size_t(std::max<int64_t>(n_pairs, 1)))
    PYCD_HIP(ctx, s->lubuf.alloc(size_t(std::max<int64_t>(n_pairs, 1))));
  if (!s->ev0) {
    PYCD_HIP(ctx, hipEventCreate(&s->ev0));
    PYCD_HIP(ctx, hipEventCreate(&s->ev1));
  }
  int64_t made = 0;
  const int rc = hop_loop(s, dU, s->lubuf.ptr, s->status.ptr, n_pairs,
                          max_hops, dT, dP, true, &made);
  if (t_host && made > 0)
    PYCD_HIP(ctx, hipMemcpy(hop_time, dT, 8 * size_t(made),
                            hipMemcpyDeviceToHost));
  if (p_host && made > 0)
    PYCD_HIP(ctx, hipMemcpy(hop_proc, dP, 4 * size_t(made),
                            hipMemcpyDeviceToHost));
  if (hops_out) *hops_out = made;
  return rc;
}

namespace pycd {

// The hop loop of pycd_kmc_advance and pycd_kmc_advance_static: log(u2) of
// the chunk into LU, the kernel, its status into `status` (device) and back.
// Allocates nothing.  `timed`: HIP events around it (created beforehand).
int hop_loop(pycd_kmc* s, const double* dU, double* LU, int32_t* status_dev,
             int64_t n_pairs, int64_t max_hops, double* dT, int32_t* dP,
             bool timed, int64_t* made) {
  pycd_ctx* ctx = s->ctx;
  hipStream_t st = ctx->stream;
  const pycd_kmc_problem& pb = s->pb;
  const KmcDev d{s->pk.ptr,    s->cq.ptr,    s->occ.ptr, s->disp.ptr,
                 s->base.ptr, s->drift.ptr, s->sc.ptr};
  HopArgs args;
  args.tab = reinterpret_cast<const char*>(s->compact ? s->Ac.ptr : s->A.ptr);
  args.row_bytes = uint32_t(pb.n_sites) * uint32_t(sizeof(double));
  args.gp = geo_pk(s->compact ? s->geo : Geo{1, 1, 1, 1});
  args.rec = s->rec.ptr;
  args.pe = s->pe.ptr;
  args.nbr2 = s->nbr2.ptr;
  args.rows = s->rows.ptr;
  args.epath = s->epath.ptr;
  args.dpath = s->dpath.ptr;
  args.U = dU;
  args.LU = LU;
  args.hop_time = dT;
  args.hop_proc = dP;
  args.nc = pb.n_carriers;
  args.z = pb.z;
  args.mz = pb.max_z;
  args.field_on =
      pb.field[0] != 0.0 || pb.field[1] != 0.0 || pb.field[2] != 0.0;
  args.nu = pb.nu;
  args.nkt = -1.0 / pb.kT;
  args.dt = pb.time_interval;
  args.P = pb.n_path;
  args.n_pairs = n_pairs;
  args.max_hops = max_hops;
  if (timed) PYCD_HIP(ctx, hipEventRecord(s->ev0, st));
  reset_status<<<1, 1, 0, st>>>(status_dev);
  if (n_pairs > 0)
    log_u2_kernel<<<int(std::min<int64_t>((n_pairs + 255) / 256, 4096)), 256,
                    0, st>>>(dU, n_pairs, LU);
  PYCD_HIP(ctx, hipMemcpyAsync(s->dev.ptr, &d, sizeof(KmcDev),
                               hipMemcpyHostToDevice, st));
  PYCD_HIP(ctx, launch_hop(s, st, args, status_dev));
  PYCD_HIP(ctx, hipGetLastError());
  if (timed) PYCD_HIP(ctx, hipEventRecord(s->ev1, st));
  int32_t status[2] = {-1, 0};
  PYCD_HIP(ctx, hipMemcpyAsync(status, status_dev, sizeof(status),
                               hipMemcpyDeviceToHost, st));
  PYCD_HIP(ctx, hipStreamSynchronize(st));
  if (timed) {
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, s->ev0, s->ev1);
    s->last_ms = ms;
  }
  *made = status[1];
  if (status[0] < 0) return fail(ctx, PYCD_ERR_STATE, "kernel did not report");
  return status[0] == 1 ? PYCD_NEED_UNIFORMS : PYCD_OK;
}

}  // namespace pycd

extern "C" int pycd_kmc_advance_static(pycd_kmc* s, const double* uniforms,
                                       int64_t n_pairs, int64_t max_hops,
                                       double* hop_time, int32_t* hop_proc,
                                       int64_t* hops_out) {
  if (!s) return PYCD_ERR_ARG;
  pycd_ctx* ctx = s->ctx;
  if (!s->begun) return fail(ctx, PYCD_ERR_STATE, "pycd_kmc_begin not called");
  if (n_pairs < 0 || (n_pairs > 0 && !uniforms))
    return fail(ctx, PYCD_ERR_ARG, "bad uniform buffer");
  if (n_pairs > kStaticPairs)
    return fail(ctx, PYCD_ERR_ARG,
                "pycd_kmc_advance_static takes at most %lld uniform pairs "
                "per call (its log(u2) scratch is a fixed device array); got "
                "%lld",
                (long long)kStaticPairs, (long long)n_pairs);
  if (!ctx->static_scratch)
    return fail(ctx, PYCD_ERR_STATE, "static scratch of the device unresolved");
  DeviceGuard guard(ctx->device);
  if ((n_pairs > 0 && !is_device_ptr(uniforms)) ||
      (hop_time && !is_device_ptr(hop_time)) ||
      (hop_proc && !is_device_ptr(hop_proc)))
    return fail(ctx, PYCD_ERR_ARG,
                "pycd_kmc_advance_static takes device buffers only");
  double* LU = ctx->static_scratch;
  int32_t* status = reinterpret_cast<int32_t*>(LU + kStaticPairs);
  int64_t made = 0;
  const int rc = hop_loop(s, uniforms, LU, status, n_pairs, max_hops,
                          hop_time, hop_proc, false, &made);
  if (hops_out) *hops_out = made;
  return rc;
}

extern "C" int pycd_kmc_read(pycd_kmc* s, double* unwrapped, double* energy,
                             double* delg_0, double* drift, int64_t* occupancy,
                             double scalars[4]) {
  if (!s) return PYCD_ERR_ARG;
  pycd_ctx* ctx = s->ctx;
  DeviceGuard guard(ctx->device);
  hipStream_t st = ctx->stream;
  const pycd_kmc_problem& pb = s->pb;
  const int nc = pb.n_carriers;
  const int64_t P = pb.n_path;
  if (unwrapped)
    PYCD_HIP(ctx, download(unwrapped, s->rows.ptr, size_t(P) * 3 * nc, st));
  if (energy) PYCD_HIP(ctx, download(energy, s->epath.ptr, size_t(P), st));
  if (delg_0) PYCD_HIP(ctx, download(delg_0, s->dpath.ptr, size_t(P), st));
  if (drift) PYCD_HIP(ctx, download(drift, s->drift.ptr, 3 * size_t(nc), st));
  KmcScalars sc{};
  PYCD_HIP(ctx, hipMemcpyAsync(&sc, s->sc.ptr, sizeof(sc),
                               hipMemcpyDeviceToHost, st));
  std::vector<int32_t> occ(nc);
  PYCD_HIP(ctx, hipMemcpyAsync(occ.data(), s->occ.ptr, 4 * nc,
                               hipMemcpyDeviceToHost, st));
  PYCD_HIP(ctx, hipStreamSynchronize(st));
  if (occupancy)
    for (int c = 0; c < nc; ++c) occupancy[c] = occ[c];
  if (scalars) {
    scalars[0] = sc.t;
    scalars[1] = sc.energy;
    scalars[2] = double(sc.start);
    scalars[3] = double(sc.hops);
  }
  return PYCD_OK;
}

extern "C" double pycd_kmc_last_ms(const pycd_kmc* s) {
  return s ? s->last_ms : -1.0;
}
