// Reduced-precision reciprocal contraction of the Ewald table on MFMA.
//
// A_recip = 2/eps * Y Y^T with the structure factors Y (N x 2K) is computed
// on the matrix cores in one of two modes:
//   F32     Y in FP32, v_mfma_f32_16x16x4f32, FP32 accumulation;
//   BF16X3  Y = hi + lo with hi = bf16(Y), lo = bf16(Y - hi) (both from the
//           FP64 structure factor), Y Y^T ~ hi hi^T + hi lo^T + lo hi^T on
//           v_mfma_f32_16x16x32_bf16, FP32 accumulation.
// The real-space term (minimum image, erfc) and the self term are added in
// FP64 by finish_table, as for the FP64 kernel, so only the reciprocal sum
// carries the reduced precision.
//
// Tiling: 256 threads = 4 wavefronts per 128 x 128 output tile; each
// wavefront owns 64 x 64 = 4 x 4 MFMA blocks of 16 x 16.  K is staged
// through LDS in slices (row-major, padded rows); the global loads of the
// next slice are in flight while the current one is multiplied.  The F32
// mode has two stages; the BF16X3 mode also has two-stage kernels (one barrier per slice, loads two
// or three slices ahead) on 128 x 128 tiles and on 256 x 256 tiles of 8
// wavefronts; the latter is the default from 4096 sites on.
#include "ewald_common.hpp"

#include <hip/hip_bf16.h>

namespace pycd {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr int kMTile = 128;

// 16-byte load through a global (address-space-1) pointer.  A generic
// pointer would compile to a flat load, which also counts against the LDS
// wait counter and would make every LDS read wait for the prefetch.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__device__ inline uint4 load16_global(const void* p) {
  const u32x4 v = *(const __attribute__((address_space(1))) u32x4*)(p);
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ inline float4 load16f_global(const void* p) {
  const uint4 v = load16_global(p);
  return make_float4(__uint_as_float(v.x), __uint_as_float(v.y),
                     __uint_as_float(v.z), __uint_as_float(v.w));
}

// Structure factors in reduced precision from the FP64 values, a thread one
// k column of kLowRows rows, its k vector in registers; columns past 2 K and
// rows past n are written as zeros here rather than by fills of the whole
// array ahead (which, with a division per element for its row, took 0.29 +
// 0.07 ms at 12000 sites and 2 K = 9834, now 0.23).
constexpr int kLowRows = 16;
template <int kMode>
__global__ void __launch_bounds__(256)
structure_factor_lowp(const double* __restrict__ pos, int n, int n_pad,
                      const double* __restrict__ kv,
                      const double* __restrict__ sw, int K, int Kp,
                      float* __restrict__ y32, __bf16* __restrict__ yhi,
                      __bf16* __restrict__ ylo) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= Kp - K) return;
  const bool real = m < K;
  const double kx = real ? kv[3 * m] : 0.0, ky = real ? kv[3 * m + 1] : 0.0,
               kz = real ? kv[3 * m + 2] : 0.0, w = real ? sw[m] : 0.0;
  // w v and, in two parts, its rounding to BF16 and what that leaves.  A
  // cosine is rounded by way of FP32, a sine at once: 8.5e-6 of the cosines
  // go to the other neighbour for that (an FP32 value lies halfway between
  // two BF16 ones once in 65536), and the low part holds the difference.
  // Tables of this mode have had these bits from the start.
  auto put = [&](int64_t o, double v, bool by_f32) {
#pragma clang fp contract(off)
    const double y = w * v;
    if constexpr (kMode == PYCD_PREC_F32) {
      y32[o] = float(y);
    } else {
      float f = float(y);
      asm volatile("" : "+v"(f));  // (rounded here, not folded)
      const __bf16 h = by_f32 ? __bf16(f) : __bf16(y);
      yhi[o] = h;
      ylo[o] = __bf16(y - double(float(h)));
    }
  };
  const int i0 = blockIdx.y * kLowRows, i1 = min(i0 + kLowRows, n_pad);
  for (int i = i0; i < i1; ++i) {
    double s = 0.0, c = 0.0;
    if (real && i < n) {
      const double ph = kx * pos[3 * i] + ky * pos[3 * i + 1] +
                        kz * pos[3 * i + 2];
      sincos(ph, &s, &c);
    }
    const int64_t row = int64_t(i) * Kp;
    if (real) put(row + m, c, true);
    put(row + K + m, s, false);
  }
}

// The reciprocal part of a wavefront's kX x kY blocks of 16 x 16, at
// (i0, j0), into the table; finish_table does the rest.
template <int kX, int kY>
__device__ __forceinline__ void store_recip(const v4f (&acc)[kX][kY],
                                            double* __restrict__ A, int n,
                                            int i0, int j0,
                                            const EwaldScalars& es) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int x = 0; x < kX; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + 16 * x + (lane >> 4) * 4 + r;
      double* row = A + int64_t(i) * n + j0 + (lane & 15);
#pragma unroll
      for (int y = 0; y < kY; ++y)
        if (i < n && j0 + 16 * y + (lane & 15) < n)
          row[16 * y] = recip_part(es, double(acc[x][y][r]));
    }
}

// One (32 kB) x (32 kB) tile per workgroup, each wavefront a quarter of it
// in kB x kB blocks of v_mfma_f32_16x16x4: lane l gives row (column) l mod 16
// at k + l / 16.  Bound by the FP32 matrix rate.  K goes through LDS in
// slices of 16 in two stages, one barrier per slice, global loads two slices
// ahead and each k step's fragments read behind the last step's products
// (see table_f64, which this mirrors); rows of 16 + 4 floats put a
// wavefront's 64 reads on distinct banks, and the 40 KB of a 128 x 128
// workgroup let four share a CU, so that the few tiles per CU of a table
// (4.6 at 6144 sites) are worked on side by side.  With one stage, two
// barriers a slice and the rest of the entries in the epilogue: 2.07 ms at
// 6144 sites and 2 K = 5036 (1.3 at the matrix rate); now 1.65 and 0.15 for
// finish_table.  64 x 64 or 128 x 128 tiles as for table_f64 (wide_tiles).  Every
// entry is the chain over k whatever the tile.
constexpr int kFSlice = 16;
template <int kB>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(4)))
table_mfma_f32(const float* __restrict__ Y, int n, int Kp, EwaldScalars es,
               double* __restrict__ A) {
  constexpr int kTile = 32 * kB;
  constexpr int kRow = kFSlice + 4;
  constexpr int kArr = kTile * kRow;
  constexpr int kQ = kTile / 64;  // 16-byte chunks per thread and operand
  // stage s, operand a at S + (2 s + a) kArr
  __shared__ __attribute__((aligned(16))) float S[4 * kArr];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int bi, bj;
  tile_coords_upper(n, kTile, bi, bj);
  const int i0 = bi * kTile, j0 = bj * kTile;
  const int wr = (wave >> 1) * (kTile / 2), wc = (wave & 1) * (kTile / 2);
  v4f acc[kB][kB];
#pragma unroll
  for (int x = 0; x < kB; ++x)
#pragma unroll
    for (int y = 0; y < kB; ++y) acc[x][y] = v4f{0.f, 0.f, 0.f, 0.f};
  // loader: a thread takes 4 consecutive k of every 64th row
  const int lrow = t >> 2, lk = (t & 3) * 4;
  const float* ya = Y + int64_t(i0 + lrow) * Kp + lk;
  const float* yb = Y + int64_t(j0 + lrow) * Kp + lk;
  float4 ra[kQ], rb[kQ];
  auto gload = [&](int k0) {
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      ra[q] = load16f_global(ya + int64_t(64 * q) * Kp + k0);
      rb[q] = load16f_global(yb + int64_t(64 * q) * Kp + k0);
    }
  };
  auto sstore = [&](int stage) {
    float* a = S + 2 * stage * kArr + lrow * kRow + lk;
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      *reinterpret_cast<float4*>(a + 64 * q * kRow) = ra[q];
      *reinterpret_cast<float4*>(a + kArr + 64 * q * kRow) = rb[q];
    }
  };
  auto lds_barrier = [] {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  float fa[2][kB], fb[2][kB];
  auto fetch = [&](int set, int stage, int u) {
    const float* a = S + 2 * stage * kArr + (wr + (lane & 15)) * kRow +
                     (lane >> 4) + 4 * u;
    const float* b = S + (2 * stage + 1) * kArr + (wc + (lane & 15)) * kRow +
                     (lane >> 4) + 4 * u;
#pragma unroll
    for (int x = 0; x < kB; ++x) {
      fa[set][x] = a[16 * x * kRow];
      fb[set][x] = b[16 * x * kRow];
    }
  };
  auto k_step = [&](int set, int next_stage, int next_u, auto&& more) {
    fetch(set ^ 1, next_stage, next_u);
    more();
#pragma unroll
    for (int x = 0; x < kB; ++x)
#pragma unroll
      for (int y = 0; y < kB; ++y)
        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(
            fa[set][x], fb[set][y], acc[x][y], 0, 0, 0);
#pragma unroll
    for (int q = 0; q < 2 * kB; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, kB / 2, 0);  // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);       // LDS read
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);       // LDS write
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);       // global load
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto step = [&](int stage, int k0) {
    k_step(0, stage, 1, [] {});
    k_step(1, stage, 2, [&] { sstore(stage ^ 1); });
    k_step(0, stage, 3, [&] { gload(min(k0 + 2 * kFSlice, Kp - kFSlice)); });
    lds_barrier();
    k_step(1, stage ^ 1, 0, [] {});
  };
  gload(0);
  sstore(0);
  gload(min(kFSlice, Kp - kFSlice));
  lds_barrier();
  fetch(0, 0, 0);
  for (int k0 = 0; k0 < Kp; k0 += 2 * kFSlice) {
    step(0, k0);
    step(1, k0 + kFSlice);
  }
  store_recip<kB, kB>(acc, A, n, i0 + wr, j0 + wc, es);
}

// K is staged in slices of kBSlice = 32 or 64: a 64-deep slice makes two
// 32-deep MFMA steps per pair of barriers, and its global loads (in
// registers while the previous slice is multiplied) have twice the matrix
// work to arrive in.  Padded rows of kBSlice + 8 bf16 put the 8 rows one
// 16-byte LDS read serves on distinct banks.  The sums over k run in the
// same order for both, so they give the same table bit for bit.
template <int kBSlice>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2, 2)))
table_mfma_bf16x3(const __bf16* __restrict__ Yhi,
                  const __bf16* __restrict__ Ylo, int n, int Kp,
                  EwaldScalars es, double* __restrict__ A) {
  constexpr int kRow = kBSlice + 8;  // padded row (bf16 elements)
  __shared__ __attribute__((aligned(16))) __bf16 Ah[kMTile * kRow];
  __shared__ __attribute__((aligned(16))) __bf16 Al[kMTile * kRow];
  __shared__ __attribute__((aligned(16))) __bf16 Bh[kMTile * kRow];
  __shared__ __attribute__((aligned(16))) __bf16 Bl[kMTile * kRow];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int bi, bj;
  tile_coords_upper(n, kMTile, bi, bj);
  const int i0 = bi * kMTile, j0 = bj * kMTile;
  const int wr = (wave >> 1) * 64, wc = (wave & 1) * 64;
  v4f acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
  // loader: 128 rows x kBSlice bf16 = 256 threads x kBSlice / 2 bf16
  // (16-byte chunks) per array
  constexpr int kQ = kBSlice / 16;  // chunks per thread and array
  const int lrow = t >> 1, lk = (t & 1) * (kBSlice / 2);
  const bool a_ok = i0 + lrow < n, b_ok = j0 + lrow < n;
  const int64_t aoff = int64_t(i0 + lrow) * Kp + lk;
  const int64_t boff = int64_t(j0 + lrow) * Kp + lk;
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  uint4 ah[kQ], al[kQ], bh[kQ], bl[kQ];
  auto gload = [&](int k0) {
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      ah[q] = a_ok ? load16_global(Yhi + aoff + k0 + 8 * q) : zero;
      al[q] = a_ok ? load16_global(Ylo + aoff + k0 + 8 * q) : zero;
      bh[q] = b_ok ? load16_global(Yhi + boff + k0 + 8 * q) : zero;
      bl[q] = b_ok ? load16_global(Ylo + boff + k0 + 8 * q) : zero;
    }
  };
  auto sstore = [&]() {
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      *reinterpret_cast<uint4*>(Ah + lrow * kRow + lk + 8 * q) = ah[q];
      *reinterpret_cast<uint4*>(Al + lrow * kRow + lk + 8 * q) = al[q];
      *reinterpret_cast<uint4*>(Bh + lrow * kRow + lk + 8 * q) = bh[q];
      *reinterpret_cast<uint4*>(Bl + lrow * kRow + lk + 8 * q) = bl[q];
    }
  };
  gload(0);
  sstore();
  __syncthreads();
  for (int k0 = 0; k0 < Kp; k0 += kBSlice) {
    const bool more = k0 + kBSlice < Kp;
    if (more) gload(k0 + kBSlice);
#pragma unroll
    for (int h = 0; h < kBSlice / 32; ++h) {
      // this wavefront's column blocks once, then one row block at a time
      const int kof = (lane >> 4) * 8 + 32 * h;
      v8bf b_h[4], b_l[4];
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        const int rb = (wc + 16 * y + (lane & 15)) * kRow + kof;
        b_h[y] = *reinterpret_cast<const v8bf*>(Bh + rb);
        b_l[y] = *reinterpret_cast<const v8bf*>(Bl + rb);
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int ra = (wr + 16 * x + (lane & 15)) * kRow + kof;
        const v8bf a_h = *reinterpret_cast<const v8bf*>(Ah + ra);
        const v8bf a_l = *reinterpret_cast<const v8bf*>(Al + ra);
#pragma unroll
        for (int y = 0; y < 4; ++y) {
          acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a_l, b_h[y], acc[x][y], 0, 0, 0);
          acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a_h, b_l[y], acc[x][y], 0, 0, 0);
          acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a_h, b_h[y], acc[x][y], 0, 0, 0);
        }
      }
    }
    __syncthreads();  // every wavefront is done with this slice
    if (more) sstore();
    __syncthreads();
  }
  store_recip<4, 4>(acc, A, n, i0 + wr, j0 + wc, es);
}

// K slices of 32 in two LDS stages and three register sets: while slice t
// is multiplied out of one stage, slice t + 1 (in registers since two steps
// before) goes to the other stage and slice t + 3 is loaded into the
// registers slice t left, so a global load has three steps to arrive.  One barrier per slice, without a
// memory fence: it waits for this wavefront's LDS operations only, and the
// loads in flight stay in flight.  Two workgroups fill a CU's 160 KB of LDS.
// The sums over k run in the same order as the one-stage kernels, so the
// table is the same bit for bit.  Y holds whole 128-row tiles (rows past n
// are zero) and Kp is a multiple of 6 kB (zero columns), so every load and
// LDS store is made unconditionally: a branch around them would make the
// compiler wait for all loads in flight.
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2, 2)))
table_mfma_bf16x3_2stage(const __bf16* __restrict__ Yhi,
                         const __bf16* __restrict__ Ylo, int n, int Kp,
                         EwaldScalars es, double* __restrict__ A) {
  constexpr int kB = 32;
  constexpr int kRow = kB + 8;  // padded row (bf16 elements)
  constexpr int kArr = kMTile * kRow;
  // stage s, array a (hi A, lo A, hi B, lo B) at S + (4 s + a) kArr
  __shared__ __attribute__((aligned(16))) __bf16 S[2 * 4 * kArr];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int bi, bj;
  tile_coords_upper(n, kMTile, bi, bj);
  const int i0 = bi * kMTile, j0 = bj * kMTile;
  const int wr = (wave >> 1) * 64, wc = (wave & 1) * 64;
  v4f acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
  // loader: 128 rows x 32 bf16 per array = 256 threads x one 16-byte chunk
  // of each of hi/lo at two k offsets
  constexpr int kQ = kB / 16;
  const int lrow = t >> 1, lk = (t & 1) * (kB / 2);
  const int64_t aoff = int64_t(i0 + lrow) * Kp + lk;
  const int64_t boff = int64_t(j0 + lrow) * Kp + lk;
  struct Regs { uint4 v[4][kQ]; };
  auto gload = [&](Regs& r, int k0) {
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      r.v[0][q] = load16_global(Yhi + aoff + k0 + 8 * q);
      r.v[1][q] = load16_global(Ylo + aoff + k0 + 8 * q);
      r.v[2][q] = load16_global(Yhi + boff + k0 + 8 * q);
      r.v[3][q] = load16_global(Ylo + boff + k0 + 8 * q);
    }
  };
  auto sstore = [&](int stage, const Regs& r) {
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int q = 0; q < kQ; ++q)
        *reinterpret_cast<uint4*>(S + (4 * stage + a) * kArr + lrow * kRow +
                                  lk + 8 * q) = r.v[a][q];
  };
  // all of this wavefront's LDS operations done, then the barrier
  auto lds_barrier = [] {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  auto multiply = [&](int stage) {
    const __bf16* Ah = S + (4 * stage + 0) * kArr;
    const __bf16* Al = S + (4 * stage + 1) * kArr;
    const __bf16* Bh = S + (4 * stage + 2) * kArr;
    const __bf16* Bl = S + (4 * stage + 3) * kArr;
    const int kof = (lane >> 4) * 8;
    v8bf b_h[4], b_l[4];
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const int rb = (wc + 16 * y + (lane & 15)) * kRow + kof;
      b_h[y] = *reinterpret_cast<const v8bf*>(Bh + rb);
      b_l[y] = *reinterpret_cast<const v8bf*>(Bl + rb);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int ra = (wr + 16 * x + (lane & 15)) * kRow + kof;
      const v8bf a_h = *reinterpret_cast<const v8bf*>(Ah + ra);
      const v8bf a_l = *reinterpret_cast<const v8bf*>(Al + ra);
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            a_l, b_h[y], acc[x][y], 0, 0, 0);
        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            a_h, b_l[y], acc[x][y], 0, 0, 0);
        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            a_h, b_h[y], acc[x][y], 0, 0, 0);
      }
    }
  };
  // step for slice k0 (in stage `stage`): `next` holds slice k0 + kB,
  // `spare` takes slice k0 + 3 kB; at the end of K they load and store the
  // last slice again (into a stage no step reads)
  // (scheduling barriers keep the loads at the start of the step and the
  // LDS stores at its end, which the scheduler would otherwise swap)
  auto step = [&](int stage, int k0, Regs& next, Regs& spare) {
    gload(spare, min(k0 + 3 * kB, Kp - kB));
    __builtin_amdgcn_sched_barrier(0);
    multiply(stage);
    __builtin_amdgcn_sched_barrier(0);
    sstore(stage ^ 1, next);
    lds_barrier();
  };
  Regs r0, r1, r2;
  gload(r0, 0);
  sstore(0, r0);
  gload(r1, kB);
  gload(r2, 2 * kB);
  lds_barrier();
  for (int k0 = 0; k0 < Kp; k0 += 6 * kB) {
    step(0, k0, r1, r0);
    step(1, k0 + kB, r2, r1);
    step(0, k0 + 2 * kB, r0, r2);
    step(1, k0 + 3 * kB, r1, r0);
    step(0, k0 + 4 * kB, r2, r1);
    step(1, k0 + 5 * kB, r0, r2);
  }
  store_recip<4, 4>(acc, A, n, i0 + wr, j0 + wc, es);
}

// 256 x 256 output tiles on 8 wavefronts (512 threads), each wavefront
// 128 x 64 = 8 x 4 MFMA blocks: a step loads half the bytes per product of
// the 128 x 128 tiles, and a wavefront reads a quarter less LDS per
// product.  K slices of 32 in two LDS stages (160 KB, one workgroup per CU):
// a step loads the next slice into registers as it starts and stores it to
// the other stage as it ends, with the step's 96 MFMAs per wavefront in
// between (one register set: the accumulators take half the registers).  For the table to equal
// the 128 x 128 kernels' bit for bit, every entry is formed with the same
// operands in the same roles: in a diagonal 256-tile the lower-left 128 x 128
// block is not stored, its upper mirror writes it (as a 128 x 128 tile off
// the diagonal does), and the two diagonal 128-blocks store both (i, j) and
// (j, i) as formed.  Y holds whole 256-row tiles and Kp is a multiple of
// 2 kB, so loads and LDS stores are unconditional.
constexpr int kMTile2 = 256;

// Two 128 x 128 tiles in one 512-thread workgroup of the 256 x 256 kernel,
// one per half (4 wavefronts of 64 x 64, as in the 128 x 128 kernels), each
// half in its own 80 KB of the LDS, the two in step at the shared
// barriers.  `sub` lists the tiles (tile row, tile column); workgroup k
// takes entries 2k and 2k + 1 (a missing second one repeats the first and
// stores nothing).
__device__ __forceinline__ void bf16x3_tile_pair(
    __bf16* S, const __bf16* __restrict__ Yhi, const __bf16* __restrict__ Ylo,
    int n, int Kp, const EwaldScalars& es, double* __restrict__ A,
    const int2* __restrict__ sub, int n_sub, int k) {
  constexpr int kB = 32;
  constexpr int kRow = kB + 8;
  constexpr int kArr = kMTile * kRow;
  const int t = threadIdx.x, th = t & 255, lane = t & 63;
  const int half = __builtin_amdgcn_readfirstlane(t >> 8);
  const int wave = __builtin_amdgcn_readfirstlane((t >> 6) & 3);
  int idx = 2 * k + half;
  const bool dummy = idx >= n_sub;
  if (dummy) idx = 2 * k;
  const int2 tl = sub[idx];
  const int i0 = tl.x * kMTile, j0 = tl.y * kMTile;
  const int wr = (wave >> 1) * 64, wc = (wave & 1) * 64;
  __bf16* Sh = S + half * (2 * 4 * kArr);
  v4f acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
  constexpr int kQ = kB / 16;
  const int lrow = th >> 1, lk = (th & 1) * (kB / 2);
  const int64_t aoff = int64_t(i0 + lrow) * Kp + lk;
  const int64_t boff = int64_t(j0 + lrow) * Kp + lk;
  struct Regs { uint4 v[4][kQ]; };
  auto gload = [&](Regs& r, int k0) {
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      r.v[0][q] = load16_global(Yhi + aoff + k0 + 8 * q);
      r.v[1][q] = load16_global(Ylo + aoff + k0 + 8 * q);
      r.v[2][q] = load16_global(Yhi + boff + k0 + 8 * q);
      r.v[3][q] = load16_global(Ylo + boff + k0 + 8 * q);
    }
  };
  auto sstore = [&](int stage, const Regs& r) {
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int q = 0; q < kQ; ++q)
        *reinterpret_cast<uint4*>(Sh + (4 * stage + a) * kArr + lrow * kRow +
                                  lk + 8 * q) = r.v[a][q];
  };
  auto lds_barrier = [] {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  auto multiply = [&](int stage) {
    const __bf16* Ah = Sh + (4 * stage + 0) * kArr;
    const __bf16* Al = Sh + (4 * stage + 1) * kArr;
    const __bf16* Bh = Sh + (4 * stage + 2) * kArr;
    const __bf16* Bl = Sh + (4 * stage + 3) * kArr;
    const int kof = (lane >> 4) * 8;
    v8bf b_h[4], b_l[4];
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const int rb = (wc + 16 * y + (lane & 15)) * kRow + kof;
      b_h[y] = *reinterpret_cast<const v8bf*>(Bh + rb);
      b_l[y] = *reinterpret_cast<const v8bf*>(Bl + rb);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int ra = (wr + 16 * x + (lane & 15)) * kRow + kof;
      const v8bf a_h = *reinterpret_cast<const v8bf*>(Ah + ra);
      const v8bf a_l = *reinterpret_cast<const v8bf*>(Al + ra);
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            a_l, b_h[y], acc[x][y], 0, 0, 0);
        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            a_h, b_l[y], acc[x][y], 0, 0, 0);
        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            a_h, b_h[y], acc[x][y], 0, 0, 0);
      }
    }
  };
  Regs r;
  auto step = [&](int stage, int k0) {
    gload(r, min(k0 + kB, Kp - kB));
    __builtin_amdgcn_sched_barrier(0);
    multiply(stage);
    __builtin_amdgcn_sched_barrier(0);
    sstore(stage ^ 1, r);
    lds_barrier();
  };
  gload(r, 0);
  sstore(0, r);
  lds_barrier();
  for (int k0 = 0; k0 < Kp; k0 += 2 * kB) {
    step(0, k0);
    step(1, k0 + kB);
  }
  if (dummy) return;
  store_recip<4, 4>(acc, A, n, i0 + wr, j0 + wc, es);
}

__global__ void __launch_bounds__(512)
__attribute__((amdgpu_waves_per_eu(2, 2)))
table_mfma_bf16x3_256(const __bf16* __restrict__ Yhi,
                      const __bf16* __restrict__ Ylo, int n, int Kp,
                      EwaldScalars es, double* __restrict__ A,
                      int main_tiles, const int2* __restrict__ sub,
                      int n_sub) {
  constexpr int kB = 32;
  constexpr int kRow = kB + 8;  // padded row (bf16 elements)
  constexpr int kArr = kMTile2 * kRow;
  // stage s, array a (hi A, lo A, hi B, lo B) at S + (4 s + a) kArr
  __shared__ __attribute__((aligned(16))) __bf16 S[2 * 4 * kArr];
  // the tiles past the last whole round of 256 x 256 tiles, as pairs of
  // 128 x 128 tiles (the last round takes about half as long)
  if (int(blockIdx.x) >= main_tiles) {
    bf16x3_tile_pair(S, Yhi, Ylo, n, Kp, es, A, sub, n_sub,
                     int(blockIdx.x) - main_tiles);
    return;
  }
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int bi, bj;
  tile_coords_upper(n, kMTile2, bi, bj);
  const int i0 = bi * kMTile2, j0 = bj * kMTile2;
  const int wr = (wave >> 2) * 128, wc = (wave & 3) * 64;
  // in a diagonal tile the lower-left 128-block is not stored
  const bool skip = bi == bj && wr == 128 && wc < 128;
  v4f acc[8][4];
#pragma unroll
  for (int a = 0; a < 8; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
  // loader: 256 rows x 32 bf16 per array = 512 threads x two 16-byte chunks
  constexpr int kQ = kB / 16;
  const int lrow = t >> 1, lk = (t & 1) * (kB / 2);
  const int64_t aoff = int64_t(i0 + lrow) * Kp + lk;
  const int64_t boff = int64_t(j0 + lrow) * Kp + lk;
  struct Regs { uint4 v[4][kQ]; };
  auto gload = [&](Regs& r, int k0) {
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      r.v[0][q] = load16_global(Yhi + aoff + k0 + 8 * q);
      r.v[1][q] = load16_global(Ylo + aoff + k0 + 8 * q);
      r.v[2][q] = load16_global(Yhi + boff + k0 + 8 * q);
      r.v[3][q] = load16_global(Ylo + boff + k0 + 8 * q);
    }
  };
  auto sstore = [&](int stage, const Regs& r) {
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int q = 0; q < kQ; ++q)
        *reinterpret_cast<uint4*>(S + (4 * stage + a) * kArr + lrow * kRow +
                                  lk + 8 * q) = r.v[a][q];
  };
  auto lds_barrier = [] {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  auto multiply = [&](int stage) {
    const __bf16* Ah = S + (4 * stage + 0) * kArr;
    const __bf16* Al = S + (4 * stage + 1) * kArr;
    const __bf16* Bh = S + (4 * stage + 2) * kArr;
    const __bf16* Bl = S + (4 * stage + 3) * kArr;
    const int kof = (lane >> 4) * 8;
    v8bf b_h[4], b_l[4];
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const int rb = (wc + 16 * y + (lane & 15)) * kRow + kof;
      b_h[y] = *reinterpret_cast<const v8bf*>(Bh + rb);
      b_l[y] = *reinterpret_cast<const v8bf*>(Bl + rb);
    }
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const int ra = (wr + 16 * x + (lane & 15)) * kRow + kof;
      const v8bf a_h = *reinterpret_cast<const v8bf*>(Ah + ra);
      const v8bf a_l = *reinterpret_cast<const v8bf*>(Al + ra);
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            a_l, b_h[y], acc[x][y], 0, 0, 0);
        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            a_h, b_l[y], acc[x][y], 0, 0, 0);
        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            a_h, b_h[y], acc[x][y], 0, 0, 0);
      }
    }
  };
  // step for slice k0 (in stage `stage`): slice k0 + kB is loaded and
  // goes to the other stage; the last step loads and stores the last slice
  // again (into a stage no step reads); scheduling barriers keep the loads
  // at the start of the step and the LDS stores at its end
  Regs r;
  auto step = [&](int stage, int k0) {
    gload(r, min(k0 + kB, Kp - kB));
    __builtin_amdgcn_sched_barrier(0);
    multiply(stage);
    __builtin_amdgcn_sched_barrier(0);
    sstore(stage ^ 1, r);
    lds_barrier();
  };
  gload(r, 0);
  sstore(0, r);
  lds_barrier();
  for (int k0 = 0; k0 < Kp; k0 += 2 * kB) {
    step(0, k0);
    step(1, k0 + kB);
  }
  if (skip) return;
  store_recip<8, 4>(acc, A, n, i0 + wr, j0 + wc, es);
}

int launch_table_mfma(pycd_ctx* ctx, int precision, const double* pos, int n,
                      const double* kv, const double* sw, int K,
                      const MicGeometry& geo, const EwaldScalars& es,
                      double* out, unsigned long long* pairs,
                      hipEvent_t after_sf, hipEvent_t (&real)[2]) {
  hipStream_t s = ctx->stream;
  // K padded to whole slices of the mode's kernel (zero columns add nothing)
  // BF16x3 default: 256 x 256 tiles from 4096 sites on, K slices of 64
  // below (a few large tiles would leave most CUs idle)
  int bvar = ctx->table_variant[PYCD_PREC_BF16X3];
  if (bvar == 0) bvar = n >= 4096 ? 4 : 2;
  const int bslice = bvar == 1 || bvar >= 3 ? 32 : 64;
  // (the two-stage kernels take K in groups of six and of two 32-slices)
  const int slice = precision == PYCD_PREC_F32 ? 2 * kFSlice
                    : bvar == 3              ? 6 * bslice
                    : bvar == 4              ? 2 * bslice
                                             : bslice;
  const int Kp = std::max(slice, ((2 * K + slice - 1) / slice) * slice);
  // rows in whole tiles: the rows past n stay zero
  const int tile =
      precision == PYCD_PREC_F32
          ? (wide_tiles(n, ctx->cu_count) ? kMTile : 64)
          : (bvar == 4 ? kMTile2 : kMTile);
  const int nb = (n + tile - 1) / tile;
  const int n_pad = nb * tile;
  const size_t elems = size_t(n_pad) * Kp;
  WorkBuf<float> y32;
  WorkBuf<__bf16> yhi, ylo;
  WorkBuf<int2> d_sub;
  std::vector<int2> sub;
  const dim3 sf_grid((Kp - K + 255) / 256, (n_pad + kLowRows - 1) / kLowRows);
  if (precision == PYCD_PREC_F32) {
    PYCD_HIP(ctx, y32.alloc(ctx, elems));
    structure_factor_lowp<PYCD_PREC_F32><<<sf_grid, 256, 0, s>>>(
        pos, n, n_pad, kv, sw, K, Kp, y32.ptr, nullptr, nullptr);
  } else {
    PYCD_HIP(ctx, yhi.alloc(ctx, elems));
    PYCD_HIP(ctx, ylo.alloc(ctx, elems));
    structure_factor_lowp<PYCD_PREC_BF16X3><<<sf_grid, 256, 0, s>>>(
        pos, n, n_pad, kv, sw, K, Kp, nullptr, yhi.ptr, ylo.ptr);
  }
  PYCD_HIP(ctx, hipGetLastError());
  PYCD_HIP(ctx, hipEventRecord(after_sf, s));
  const int tiles = nb * (nb + 1) / 2;
  if (precision == PYCD_PREC_F32 && tile == 64)
    table_mfma_f32<2><<<tiles, 256, 0, s>>>(y32.ptr, n, Kp, es, out);
  else if (precision == PYCD_PREC_F32)
    table_mfma_f32<4><<<tiles, 256, 0, s>>>(y32.ptr, n, Kp, es, out);
  else if (bvar == 3)
    table_mfma_bf16x3_2stage<<<tiles, 256, 0, s>>>(yhi.ptr, ylo.ptr, n, Kp,
                                                   es, out);
  else if (bvar == 4) {
    // whole rounds of 256 x 256 tiles (one workgroup per CU), the rest as
    // pairs of 128 x 128 tiles; fewer tiles than one round all go whole
    int dev_cus = 0;
    PYCD_HIP(ctx, hipDeviceGetAttribute(&dev_cus,
                                        hipDeviceAttributeMultiprocessorCount,
                                        ctx->device));
    const int round = std::max(dev_cus, 1);
    const int main_tiles = tiles >= round ? (tiles / round) * round : tiles;
    for (int w = main_tiles; w < tiles; ++w) {
      int bi = 0, bj = 0;
      tile_coords_upper_at(n, kMTile2, w, bi, bj);
      for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b) {
          const int si = 2 * bi + a, sj = 2 * bj + b;
          if (si > sj || si * kMTile >= n || sj * kMTile >= n) continue;
          sub.push_back(make_int2(si, sj));
        }
    }
    if (!sub.empty()) {
      PYCD_HIP(ctx, d_sub.alloc(ctx, sub.size()));
      PYCD_HIP(ctx, hipMemcpyAsync(d_sub.ptr, sub.data(),
                                   sizeof(int2) * sub.size(),
                                   hipMemcpyHostToDevice, s));
    }
    const int grid = main_tiles + int((sub.size() + 1) / 2);
    table_mfma_bf16x3_256<<<grid, 512, 0, s>>>(yhi.ptr, ylo.ptr, n, Kp, es,
                                               out, main_tiles, d_sub.ptr,
                                               int(sub.size()));
  }
  else if (bslice == 32)
    table_mfma_bf16x3<32><<<tiles, 256, 0, s>>>(yhi.ptr, ylo.ptr, n, Kp,
                                                es, out);
  else
    table_mfma_bf16x3<64><<<tiles, 256, 0, s>>>(yhi.ptr, ylo.ptr, n, Kp,
                                                es, out);
  PYCD_HIP(ctx, hipGetLastError());
  PYCD_HIP(ctx, hipEventRecord(real[0], s));
  launch_finish(s, std::min(tile, kMTile), pos, n, geo, es, out, pairs);
  PYCD_HIP(ctx, hipGetLastError());
  PYCD_HIP(ctx, hipEventRecord(real[1], s));
  PYCD_HIP(ctx, hipStreamSynchronize(s));
  return PYCD_OK;
}

}  // namespace pycd
