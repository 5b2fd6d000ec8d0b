// Ewald pair table of PyCD's System.get_precomputed_array on gfx950.
//
//   A[i,j] = erfc(sqrt(alpha) r_ij) / (2 r_ij) / eps      (r_ij < r_cut)
//          + 2/eps * sum_{k in half space, |k|^2 < k_cut^2}
//                    (2 pi / V) exp(-k^2 / (4 alpha)) / k^2 cos(k . r_ij)
//          - sqrt(alpha / pi) / eps * delta_ij
// with the real-space diagonal equal to 0.5/eps (PyCD/core.py:799-814,
// 853-878, 1594-1661).
//
// The reciprocal sum is recast as a symmetric rank-2K product of per-site
// structure factors Y[i, m] = sqrt(w_m) cos(k_m . r_i),
// Y[i, K + m] = sqrt(w_m) sin(k_m . r_i): A_recip = 2/eps * Y Y^T, because
// cos(k.(r_j - r_i)) = cos(k.r_i) cos(k.r_j) + sin(k.r_i) sin(k.r_j).  The
// contraction writes the upper triangle of tiles; finish_table adds the
// real-space term (minimum image + erfc) and the self term and writes the
// mirror.
#include "common.hpp"
#include "ewald_common.hpp"

#include <cmath>

namespace pycd {

// --------------------------------------------------------- structure factors
// Y[i, m] = sqrt(w_m) cos, Y[i, K + m] = sqrt(w_m) sin for i < n, m < K; the
// columns from 2 K to Kp and the rows from n to n_pad are zero.  A thread
// keeps one k vector and walks kSfRows rows, so a wavefront's stores are 512
// contiguous bytes and no index is divided.  Bound by sincos and by the
// write of Y.
constexpr int kSfRows = 16;

__global__ void __launch_bounds__(256)
structure_factor_f64(const double* __restrict__ pos, int n, int n_pad,
                     const double* __restrict__ kv, const double* __restrict__ sw,
                     int K, int Kp, double* __restrict__ Y) {
  const int m = blockIdx.x * 256 + threadIdx.x;
  if (m >= Kp - K) return;
  const bool real = m < K;
  const double kx = real ? kv[3 * m] : 0.0, ky = real ? kv[3 * m + 1] : 0.0,
               kz = real ? kv[3 * m + 2] : 0.0, w = real ? sw[m] : 0.0;
  const int i0 = blockIdx.y * kSfRows, i1 = min(i0 + kSfRows, n_pad);
  for (int i = i0; i < i1; ++i) {
    double vc = 0.0, vs = 0.0;
    if (real && i < n) {
      const double ph = kx * pos[3 * i] + ky * pos[3 * i + 1] +
                        kz * pos[3 * i + 2];
      double s, c;
      sincos(ph, &s, &c);
      vc = w * c;
      vs = w * s;
    }
    double* row = Y + int64_t(i) * Kp;
    if (real) row[m] = vc;
    row[K + m] = vs;
  }
}

// ------------------------------------------------- FP64 contraction + epilogue
// One (32 kB) x (32 kB) tile of A per 256-thread workgroup, each wavefront
// one quarter of it in kB x kB blocks of v_mfma_f64_16x16x4: lane l gives
// row (column) l mod 16 at k + l / 16 and holds rows l / 16 + 4 v of column
// l mod 16.  The instruction adds its four products one after another in
// ascending k, each rounded as an FMA (checked against that chain on random
// operands), so an entry is the chain over k whatever the tile, and tiles
// give the same table bit for bit.
//
// Bound by the FP64 matrix rate, 78.6 TF/s (77 measured with operands in
// registers).  A wavefront reads 2 kB doubles of LDS per lane and k step for
// kB^2 instructions of 64 cycles: 32 cycles of LDS per 1024 at kB = 4.  On
// the vector units, where every FMA takes its operands from two LDS reads
// shared by 8, the LDS was the limit (8 x 8 entries per thread, 2 bytes per
// FMA).  At 12000 sites and 2 K = 9836: 34.0 -> 21.3 ms (66 TF/s over whole
// tiles, two workgroups per CU); at 2592 sites and 2 K = 2142, fewer tiles
// than CUs: 611 -> 275 us.
//
// K goes through LDS in slices of 16 in two stages, one barrier per slice
// without a memory fence (only this wavefront's LDS operations are waited
// for), global loads two slices ahead.  Y holds whole tiles of rows and Kp
// whole pairs of slices (zero past n and 2 K), so loads are unconditional.  Rows
// of 16 + 2 doubles put the 16 rows and two k of half a wavefront's read on
// distinct banks.
constexpr int kSlice = 16;
typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));

template <int kB>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2)))
table_f64(const double* __restrict__ Y, int n, int Kp, int chunk,
          EwaldScalars es, double* __restrict__ A) {
  constexpr int kTile = 32 * kB;
  constexpr int kRow = kSlice + 2;
  constexpr int kArr = kTile * kRow;
  // stage s, operand a at S + (2 s + a) kArr
  __shared__ __attribute__((aligned(16))) double S[4 * kArr];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int bi, bj;
  tile_coords_upper(n, kTile, bi, bj);
  const int i0 = bi * kTile, j0 = bj * kTile;
  const bool mirror = bi != bj;
  const int wr = (wave >> 1) * (kTile / 2), wc = (wave & 1) * (kTile / 2);

  v4d acc[kB][kB];
#pragma unroll
  for (int x = 0; x < kB; ++x)
#pragma unroll
    for (int y = 0; y < kB; ++y) acc[x][y] = v4d{0.0, 0.0, 0.0, 0.0};

  // loader: a thread takes 2 consecutive k of every 32nd row, 8 threads
  // the 128 bytes of a row
  const int lrow = t >> 3, lk = (t & 7) * 2;
  typedef const __attribute__((address_space(1))) v2d* gp;
  // this workgroup's columns of Y: part blockIdx.y, `chunk` wide
  const int kb = int(blockIdx.y) * chunk, kn = min(chunk, Kp - kb);
  const double* ya = Y + int64_t(i0 + lrow) * Kp + kb + lk;
  const double* yb = Y + int64_t(j0 + lrow) * Kp + kb + lk;
  v2d ra[kB], rb[kB];
  auto gload = [&](int k0) {
#pragma unroll
    for (int q = 0; q < kB; ++q) {
      ra[q] = *(gp)(ya + int64_t(32 * q) * Kp + k0);
      rb[q] = *(gp)(yb + int64_t(32 * q) * Kp + k0);
    }
  };
  auto sstore = [&](int stage) {
    double* a = S + 2 * stage * kArr + lrow * kRow + lk;
#pragma unroll
    for (int q = 0; q < kB; ++q) {
      *reinterpret_cast<v2d*>(a + 32 * q * kRow) = ra[q];
      *reinterpret_cast<v2d*>(a + kArr + 32 * q * kRow) = rb[q];
    }
  };
  auto lds_barrier = [] {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  // fragments of k step u of the slice in `stage`: one double per block,
  // two sets so that a step's reads are in flight behind the last step's
  // instructions
  double fa[2][kB], fb[2][kB];
  auto fetch = [&](int set, int stage, int u) {
    const double* a = S + 2 * stage * kArr + (wr + (lane & 15)) * kRow +
                      (lane >> 4) + 4 * u;
    const double* b = S + (2 * stage + 1) * kArr + (wc + (lane & 15)) * kRow +
                      (lane >> 4) + 4 * u;
#pragma unroll
    for (int x = 0; x < kB; ++x) {
      fa[set][x] = a[16 * x * kRow];
      fb[set][x] = b[16 * x * kRow];
    }
  };
  auto multiply = [&](int set) {
#pragma unroll
    for (int x = 0; x < kB; ++x)
#pragma unroll
      for (int y = 0; y < kB; ++y)
        acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(
            fa[set][x], fb[set][y], acc[x][y], 0, 0, 0);
  };
  // One k step: the fragments of the next step (and `more`, if any) issued
  // between this step's instructions, one read per kB / 2 of them, so that
  // neither the matrix core nor the LDS waits for a burst of the other.
  auto k_step = [&](int set, int next_stage, int next_u, auto&& more) {
    fetch(set ^ 1, next_stage, next_u);
    more();
    multiply(set);
#pragma unroll
    for (int q = 0; q < 2 * kB; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, kB / 2, 0);  // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);       // LDS read
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);       // LDS write
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);       // global load
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // Step for the slice at k0, in `stage`, its first fragments read: the next
  // slice goes from registers to the other stage, the one after it is
  // loaded; the barrier comes once this slice's last fragments are read, a k
  // step before the slice is done, and the next slice's first fragments are
  // read behind that k step.  (The last steps load and store the last slice
  // again, into a stage that no step reads.)
  auto step = [&](int stage, int k0) {
    k_step(0, stage, 1, [] {});
    k_step(1, stage, 2, [&] { sstore(stage ^ 1); });
    k_step(0, stage, 3, [&] { gload(min(k0 + 2 * kSlice, kn - kSlice)); });
    lds_barrier();
    k_step(1, stage ^ 1, 0, [] {});
  };
  gload(0);
  sstore(0);
  gload(min(kSlice, kn - kSlice));
  lds_barrier();
  fetch(0, 0, 0);
  for (int k0 = 0; k0 < kn; k0 += 2 * kSlice) {
    step(0, k0);
    step(1, k0 + kSlice);
  }

  // the reciprocal part alone (of several parts: the sum itself, each part
  // its own table), no mirror: finish_table does the rest
  const bool whole = gridDim.y == 1;
  A += int64_t(blockIdx.y) * n * n;
#pragma unroll
  for (int x = 0; x < kB; ++x)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = i0 + wr + 16 * x + (lane >> 4) + 4 * v;
      double* row = A + int64_t(i) * n + j0 + wc + (lane & 15);
#pragma unroll
      for (int y = 0; y < kB; ++y)
        if (i < n && j0 + wc + 16 * y + (lane & 15) < n)
          row[16 * y] =
              whole ? recip_part(es, acc[x][y][v]) : acc[x][y][v];
    }
}

// Parts of the columns of Y.  A small table has few tiles, and a tile is a
// serial chain of K steps: 120 sites, 3 tiles of 64 x 64 and 2 K = 6914,
// took 197 us on 3 of 256 CUs.  The columns are split so that tiles times parts
// come to about two workgroups per CU, each part of at least 8 slices; the
// parts are added in order (reduce_parts): 10 + 5 us.  Against sums in
// 80 bits the parts' error is a quarter of the chain's (7e-16 and 3e-15 of
// the table there).  From 23 tiles a side (a workgroup per CU) there is one
// part.  The count is by n and K alone, not by the tile, so that tile
// variants keep giving the same table.
int k_parts(int n, int Kp) {
  const int nb = (n + 63) / 64, tiles = nb * (nb + 1) / 2;
  return std::max(1, std::min(512 / tiles, Kp / (8 * kSlice)));
}

// Sum of the parts of every entry in the upper triangle of tiles (the
// others hold nothing and are written by finish_table).
__global__ void __launch_bounds__(256)
reduce_parts(const double* __restrict__ P, int n, int parts, int tile,
             EwaldScalars es, double* __restrict__ A) {
  const int j = blockIdx.x * 64 + (threadIdx.x & 63);
  const int i = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= n || j >= n || i / tile > j / tile) return;
  const int64_t o = int64_t(i) * n + j, step = int64_t(n) * n;
  double acc = P[o];
  int k = 1;
  for (; k + 8 <= parts; k += 8) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = P[o + (k + u) * step];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc += v[u];
  }
  for (; k < parts; ++k) acc += P[o + k * step];
  A[o] = recip_part(es, acc);
}

// The rest of each entry after the contraction, and its mirror, one 64 x 64
// block of the upper triangle per 256-thread workgroup: a wavefront takes
// every 4th row, a lane a column, so that rows are read and written 512
// bytes at a time and row positions come through scalar loads; the mirror
// goes through LDS and is written the same way.  (In the contraction's
// epilogue these were 64 minimum images and erfcs of straight-line code per
// thread at two wavefronts per SIMD, and 8-byte mirror stores: 378 us in
// one kernel at 2592 sites, 275 + 59 us apart.)  Off the diagonal tiles (j, i) is the same
// number as (i, j): the same products in the same order, and squared
// distances from negated differences: fractional coordinates, the
// round-half-even wrap and the candidate images (the kept offsets come in
// +/- pairs) of (j, i) are the negatives of those of (i, j).  A tile on the
// diagonal has both as formed, so its blocks write no mirror.
//
// kRows: rows of a block.  16 instead of 64 below 128 blocks of 64, where a
// block's rows one after another take longer than there is to do beside them;
// above, 64 write whole lines of the mirror.  Device time of this kernel with
// 16 and 64 rows: 3 tiles 9.6 and 20.5 us, 45 17 and 22, 78 25 and 23, 120 33
// and 26 (without order among the sites 16 rows are the faster ones there),
// 190 46 and 30, 435 91 and 41.
template <int kTile, int kRows>
__global__ void __launch_bounds__(256)
finish_table(const double* __restrict__ pos, int n, MicGeometry g,
             EwaldScalars es, double* __restrict__ A,
             unsigned long long* __restrict__ pairs) {
  constexpr int kCol = kTile / 64, kSub = kCol * (kTile / kRows);
  __shared__ double T[kRows][65];
  int bi, bj;
  tile_coords_upper_at(n, kTile, int(blockIdx.x) / kSub, bi, bj);
  const int sub = int(blockIdx.x) % kSub;
  const int i0 = bi * kTile + sub / kCol * kRows;
  const int j0 = bj * kTile + sub % kCol * 64;
  const bool mirror = bi != bj;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = j0 + lane;
  const bool j_ok = j < n;
  const double pjx = j_ok ? pos[3 * j] : 0.0;
  const double pjy = j_ok ? pos[3 * j + 1] : 0.0;
  const double pjz = j_ok ? pos[3 * j + 2] : 0.0;
  const int i_end = min(kRows, n - i0);
  unsigned cnt = 0;
  for (int k = wave; k < i_end; k += 4) {
    const int i = i0 + k;
    if (j_ok) {
      const int64_t o = int64_t(i) * n + j;
      const double recip = A[o];
      double v = real_part_d(i, j, pjx - pos[3 * i], pjy - pos[3 * i + 1],
                             pjz - pos[3 * i + 2], g, es, cnt) +
                 recip;
      if (i == j) v += es.self_term;
      A[o] = v;
      T[k][lane] = v;
    }
  }
  count_pairs(mirror ? 2 * cnt : cnt, pairs);
  if (!mirror) return;
  __syncthreads();
  // rows of the mirror, kRows entries each
  constexpr int kPer = 64 / kRows;
  const int j_end = min(64, n - j0), r = lane % kRows;
  if (r < i_end)
    for (int k = kPer * wave + lane / kRows; k < j_end; k += 4 * kPer)
      A[int64_t(j0 + k) * n + i0 + r] = T[r][k];
}

void launch_finish(hipStream_t s, int tile, const double* pos, int n,
                   const MicGeometry& geo, const EwaldScalars& es, double* A,
                   unsigned long long* pairs) {
  const int nb = (n + tile - 1) / tile, tiles = nb * (nb + 1) / 2;
  if (tile != 64)
    finish_table<128, 64><<<4 * tiles, 256, 0, s>>>(pos, n, geo, es, A, pairs);
  else if (tiles >= 128)
    finish_table<64, 64><<<tiles, 256, 0, s>>>(pos, n, geo, es, A, pairs);
  else
    finish_table<64, 16><<<4 * tiles, 256, 0, s>>>(pos, n, geo, es, A, pairs);
}

// ------------------------------------------------------------------ launch
int launch_table_mfma(pycd_ctx* ctx, int precision, const double* pos, int n,
                      const double* kv, const double* sw, int K,
                      const MicGeometry& geo, const EwaldScalars& es,
                      double* out, unsigned long long* pairs,
                      hipEvent_t after_sf, hipEvent_t (&real)[2]);

int launch_table(pycd_ctx* ctx, int precision, const double* pos, int n,
                 const double* kv, const double* sw, int K,
                 const MicGeometry& geo, const EwaldScalars& es, double* out,
                 unsigned long long* pairs, hipEvent_t after_sf,
                 hipEvent_t (&real)[2]) {
  if (precision != PYCD_PREC_F64)
    return launch_table_mfma(ctx, precision, pos, n, kv, sw, K, geo, es, out,
                             pairs, after_sf, real);
  hipStream_t s = ctx->stream;
  // tile variant: 1 = 64 x 64, 2 = 128 x 128; 0 picks (wide_tiles)
  int v = ctx->table_variant[PYCD_PREC_F64];
  if (v == 0) v = wide_tiles(n, ctx->cu_count) ? 2 : 1;
  const int tile = v == 2 ? 128 : 64;
  const int nb = (n + tile - 1) / tile;
  // K in whole pairs of slices, rows in whole tiles
  const int pair = 2 * kSlice;
  const int Kp = std::max(pair, (2 * K + pair - 1) / pair * pair);
  const int n_pad = nb * tile;
  WorkBuf<double> Y;
  PYCD_HIP(ctx, Y.alloc(ctx, size_t(n_pad) * Kp));
  structure_factor_f64<<<dim3((Kp - K + 255) / 256,
                              (n_pad + kSfRows - 1) / kSfRows),
                         256, 0, s>>>(pos, n, n_pad, kv, sw, K, Kp, Y.ptr);
  PYCD_HIP(ctx, hipGetLastError());
  PYCD_HIP(ctx, hipEventRecord(after_sf, s));
  // (parts of whole pairs of slices, none empty)
  const int want = k_parts(n, Kp);
  const int chunk = (Kp / pair + want - 1) / want * pair;
  const int parts = (Kp + chunk - 1) / chunk;
  WorkBuf<double> P;
  if (parts > 1) PYCD_HIP(ctx, P.alloc(ctx, size_t(parts) * n * n));
  double* sums = parts > 1 ? P.ptr : out;
  const dim3 grid(nb * (nb + 1) / 2, parts);
  if (v == 2)
    table_f64<4><<<grid, 256, 0, s>>>(Y.ptr, n, Kp, chunk, es, sums);
  else
    table_f64<2><<<grid, 256, 0, s>>>(Y.ptr, n, Kp, chunk, es, sums);
  PYCD_HIP(ctx, hipGetLastError());
  if (parts > 1) {
    reduce_parts<<<dim3((n + 63) / 64, (n + 3) / 4), 256, 0, s>>>(
        P.ptr, n, parts, tile, es, out);
    PYCD_HIP(ctx, hipGetLastError());
  }
  PYCD_HIP(ctx, hipEventRecord(real[0], s));
  launch_finish(s, tile, pos, n, geo, es, out, pairs);
  PYCD_HIP(ctx, hipEventRecord(real[1], s));
  PYCD_HIP(ctx, hipGetLastError());
  return PYCD_OK;
}

// -------------------------------------------------------------------- host
int build_ewald_setup(pycd_ctx* ctx, const double* trans, const double* cell,
                      const int32_t* pbc, double alpha, double k_cut,
                      EwaldSetup& st) {
  // Volume and reciprocal lattice from the translational matrix, with the
  // operation order of PyCD/core.py:711-722.
  const double* T = trans;
  auto cross = [](const double* a, const double* b, double* o) {
    o[0] = a[1] * b[2] - a[2] * b[1];
    o[1] = a[2] * b[0] - a[0] * b[2];
    o[2] = a[0] * b[1] - a[1] * b[0];
  };
  double c12[3], c20[3], c01[3];
  cross(T + 3, T + 6, c12);
  cross(T + 6, T + 0, c20);
  cross(T + 0, T + 3, c01);
  st.volume = std::fabs(T[0] * c12[0] + T[1] * c12[1] + T[2] * c12[2]);
  if (!(st.volume > 0))
    return fail(ctx, PYCD_ERR_ARG, "degenerate translational matrix");
  const double pref = 2 * M_PI / st.volume;
  double B[9];
  for (int d = 0; d < 3; ++d) {
    B[d] = pref * c12[d];
    B[3 + d] = pref * c20[d];
    B[6 + d] = pref * c01[d];
  }
  for (int a = 0; a < 3; ++a) {
    const double len = std::sqrt(B[3 * a] * B[3 * a] + B[3 * a + 1] * B[3 * a + 1] +
                                 B[3 * a + 2] * B[3 * a + 2]);
    st.k_max[a] = int(std::ceil(k_cut / len));
  }
  // Half space in mgrid (C) order: keep v unless -v came earlier, i.e. keep
  // v whose first non-zero component is negative (PyCD/core.py:816-838).
  const double k_cut_2 = k_cut * k_cut;
  const double alpha4 = 4 * alpha;
  st.kv.clear();
  st.sw.clear();
  for (int a = -st.k_max[0]; a <= st.k_max[0]; ++a)
    for (int b = -st.k_max[1]; b <= st.k_max[1]; ++b)
      for (int c = -st.k_max[2]; c <= st.k_max[2]; ++c) {
        const bool keep = a < 0 || (a == 0 && (b < 0 || (b == 0 && c < 0)));
        if (!keep) continue;
        const double k[3] = {a * B[0] + b * B[3] + c * B[6],
                             a * B[1] + b * B[4] + c * B[7],
                             a * B[2] + b * B[5] + c * B[8]};
        const double k2 = k[0] * k[0] + k[1] * k[1] + k[2] * k[2];
        if (!(k2 < k_cut_2)) continue;
        st.kv.insert(st.kv.end(), k, k + 3);
        st.sw.push_back(std::sqrt(pref * std::exp(-k2 / alpha4) / k2));
      }
  st.K = int(st.sw.size());
  // minimum-image geometry
  fill_mic_geometry(cell, pbc, st.geo, /*distance_only=*/true);
  return PYCD_OK;
}

}  // namespace pycd

using namespace pycd;

extern "C" int pycd_pair_table(pycd_ctx* ctx, const double* pos, int64_t n,
                               const double cell[9], const double trans[9],
                               const int32_t pbc[3], double alpha,
                               double r_cut, double k_cut, double eps_r,
                               int32_t precision, double* table_out,
                               pycd_ewald_report* report) {
  if (!ctx) return PYCD_ERR_ARG;
  if (!pos || !cell || !trans || !pbc || !table_out)
    return fail(ctx, PYCD_ERR_ARG, "null argument");
  if (n <= 0 || n > (int64_t(1) << 17))
    return fail(ctx, PYCD_ERR_ARG, "site count %lld outside [1, 131072]",
                (long long)n);
  if (!(alpha > 0) || !(r_cut >= 0) || !(k_cut >= 0) || !(eps_r > 0))
    return fail(ctx, PYCD_ERR_ARG, "invalid Ewald parameters");
  if (precision != PYCD_PREC_F64 && precision != PYCD_PREC_F32 &&
      precision != PYCD_PREC_BF16X3)
    return fail(ctx, PYCD_ERR_ARG, "unknown precision %d", precision);
  DeviceGuard guard(ctx->device);
  EwaldSetup st;
  int rc = build_ewald_setup(ctx, trans, cell, pbc, alpha, k_cut, st);
  if (rc) return rc;
  const int N = int(n);
  const int K = st.K;
  EwaldScalars es;
  es.sqrt_alpha = std::sqrt(alpha);
  es.r_cut = r_cut;
  // fl(r_cut^2) is within half an ulp of the exact square; 2^-50 above it
  // is above the exact square, so r^2 >= r_cut2 gives sqrt(r^2) >= r_cut
  es.r_cut2 = r_cut * r_cut * (1.0 + 0x1p-50);
  es.eps = eps_r;
  es.self_term = -1.0 * std::sqrt(alpha / M_PI) / eps_r;
  es.unit_eps = eps_r == 1.0;
  // (the margins are far above the rounding of f)
  for (int k = 0; k < 3; ++k) {
    const double* c = st.geo.inv + k;
    es.far[k] = r_cut * std::sqrt(c[0] * c[0] + c[3] * c[3] + c[6] * c[6]) *
                    (1.0 + 1e-9) + 1e-9;
  }

  WorkBuf<double> d_pos, d_kv, d_sw, d_A;
  WorkBuf<unsigned long long> d_pairs;
  PYCD_HIP(ctx, d_pos.alloc(ctx, size_t(N) * 3));
  PYCD_HIP(ctx, d_kv.alloc(ctx, size_t(K) * 3 + 3));
  PYCD_HIP(ctx, d_sw.alloc(ctx, size_t(K) + 1));
  PYCD_HIP(ctx, d_pairs.alloc(ctx, 1));
  hipStream_t s = ctx->stream;
  Staging stage(ctx);
  PYCD_HIP(ctx, stage_up(stage, d_pos.ptr, pos, size_t(N) * 3, s));
  PYCD_HIP(ctx, stage_up(stage, d_kv.ptr, st.kv.data(), 3 * size_t(K), s));
  PYCD_HIP(ctx, stage_up(stage, d_sw.ptr, st.sw.data(), size_t(K), s));
  PYCD_HIP(ctx, hipMemsetAsync(d_pairs.ptr, 0, sizeof(unsigned long long), s));
  double* out = table_out;
  const bool out_dev = is_device_ptr(table_out);
  if (!out_dev) {
    PYCD_HIP(ctx, d_A.alloc(ctx, size_t(N) * N));
    out = d_A.ptr;
  }

  // the whole table around the structure factors; the real-space kernel
  hipEvent_t ev[3], real[2];
  for (auto& e : ev) PYCD_HIP(ctx, hipEventCreate(&e));
  for (auto& e : real) PYCD_HIP(ctx, hipEventCreate(&e));
  PYCD_HIP(ctx, hipEventRecord(ev[0], s));
  rc = launch_table(ctx, precision, d_pos.ptr, N, d_kv.ptr, d_sw.ptr, K, st.geo,
                    es, out, d_pairs.ptr, ev[1], real);
  if (rc) {
    for (auto& e : ev) (void)hipEventDestroy(e);
    for (auto& e : real) (void)hipEventDestroy(e);
    return rc;
  }
  PYCD_HIP(ctx, hipEventRecord(ev[2], s));
  unsigned long long pairs = 0;
  hipError_t e = hipSuccess;
  if (!stage.get(&pairs, d_pairs.ptr, sizeof(pairs), &e))
    e = hipMemcpyAsync(&pairs, d_pairs.ptr, sizeof(pairs),
                       hipMemcpyDeviceToHost, s);
  PYCD_HIP(ctx, e);
  if (!out_dev) {
    const size_t bytes = sizeof(double) * N * size_t(N);
    if (!stage.get(table_out, out, bytes, &e))
      e = hipMemcpyAsync(table_out, out, bytes, hipMemcpyDeviceToHost, s);
    PYCD_HIP(ctx, e);
  }
  PYCD_HIP(ctx, stage.finish());
  float ms_sf = 0, ms_rest = 0, ms_real = 0;
  (void)hipEventElapsedTime(&ms_sf, ev[0], ev[1]);
  (void)hipEventElapsedTime(&ms_rest, ev[1], ev[2]);
  (void)hipEventElapsedTime(&ms_real, real[0], real[1]);
  for (auto& e : ev) (void)hipEventDestroy(e);
  for (auto& e : real) (void)hipEventDestroy(e);
  if (report) {
    report->n_kvec = K;
    report->n_real_pairs = int64_t(pairs);
    for (int a = 0; a < 3; ++a) report->k_max[a] = st.k_max[a];
    report->precision = precision;
    report->volume = st.volume;
    report->ms_sf = ms_sf;
    report->ms_real = ms_real;
    report->ms_recip = ms_rest;
    report->ms_total = double(ms_sf) + ms_rest;
  }
  return PYCD_OK;
}
