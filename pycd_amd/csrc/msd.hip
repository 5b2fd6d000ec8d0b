// Windowed-origin squared displacement of Analysis.compute_msd on gfx950.
//
//   sd[t, tau, c] = mean_{t0 < P - tau} |r(t0 + tau) - r(t0)|^2
// for every trajectory t, lag tau in [1, M) and carrier c
// (PyCD/core.py:2996-3007); sd[t, 0, c] = 0.
//
// The sums over origins of one carrier's path come from msd_unit (msd.hpp),
// one workgroup per (trajectory, carrier) or, when those are too few to fill
// the chip, several that share its lags and origins (msd_split); the sums of
// shared origins are then added in order by msd_scale_kernel.  Reading every
// pair's two positions from L2, 32 trajectories of 16 carriers, 10001 rows
// and 501 lags took 13.2 ms; from the LDS windows 0.60 ms, 33 TF/s of its 8
// operations per distance (FP64 issue allows 0.42 ms at the same clock).  The
// smallest calls still read from L2 (msd_short_kernel).
#include "common.hpp"
#include "msd.hpp"

#include <algorithm>

namespace pycd {

// Unit u = ((traj parts + part) passes + pass) nc + c; with one pass a
// workgroup takes every lag, else those of its pass.  Workgroup b runs on XCD
// b mod 8; each XCD takes a consecutive range of units, so the carriers of a
// trajectory, which share cache lines of its rows, read them through one L2.
// With one part the means go to sd, else the sums to `sums`.
template <int kQ>
__global__ void __launch_bounds__(kMsdThreads)
__attribute__((amdgpu_waves_per_eu(4, 4)))
msd_kernel(const double* __restrict__ pos, uint32_t units, int64_t P,
           uint32_t nc, int64_t M, uint32_t parts, uint32_t passes, int seg,
           double* __restrict__ sums, double* __restrict__ sd) {
  const uint32_t b = blockIdx.x, per = units / kMsdXcds;
  const uint32_t u =
      b < per * kMsdXcds ? b % kMsdXcds * per + b / kMsdXcds : b;
  uint32_t traj = u / nc, part = 0, pass = 0;
  const uint32_t c = u - traj * nc;
  if (passes > 1) {
    pass = traj % passes;
    traj /= passes;
  }
  if (parts > 1) {
    part = traj % parts;
    traj /= parts;
  }
  const int64_t w3 = 3 * int64_t(nc);
  const double* path = pos + int64_t(traj) * P * w3 + 3 * c;
  msd_unit<kQ>(
      (const __attribute__((address_space(1))) double*)path, w3, P,
      int64_t(pass) * msd_pass(kQ), M, passes > 1, int(part), int(parts), seg,
      [&](int64_t tau, double v) {
        if (parts > 1)
          sums[((int64_t(traj) * nc + c) * parts + part) * M + tau] = v;
        else
          sd[(int64_t(traj) * M + tau) * nc + c] =
              tau > 0 ? v / double(P - tau) : 0.0;
      });
}

// A block of 8 lags of one path per workgroup: a thread takes every 256th
// origin, for all 8 lags, from L2.
constexpr int kLagBlock = 8;
__global__ void __launch_bounds__(256)
msd_short_kernel(const double* __restrict__ pos, int64_t P, int nc, int64_t M,
                 double* __restrict__ sd) {
  const int64_t nlb = (M + kLagBlock - 1) / kLagBlock;
  const int64_t b = blockIdx.x;
  const int64_t tau0 = b % nlb * kLagBlock;
  const int c = int(b / nlb % nc);
  const int64_t traj = b / nlb / nc;
  const double* base = pos + (traj * P * nc + c) * 3;
  const int64_t stride = int64_t(nc) * 3;
  double acc[kLagBlock];
#pragma unroll
  for (int l = 0; l < kLagBlock; ++l) acc[l] = 0.0;
  for (int64_t t0 = threadIdx.x; t0 < P; t0 += blockDim.x) {
    const double x0 = base[t0 * stride];
    const double y0 = base[t0 * stride + 1];
    const double z0 = base[t0 * stride + 2];
#pragma unroll
    for (int l = 0; l < kLagBlock; ++l) {
      const int64_t tau = tau0 + l;
      if (tau >= 1 && tau < M && t0 + tau < P) {
        const double* q = base + (t0 + tau) * stride;
        const double dx = q[0] - x0, dy = q[1] - y0, dz = q[2] - z0;
        acc[l] += dx * dx + dy * dy + dz * dz;
      }
    }
  }
  __shared__ double part[kLagBlock][256];
#pragma unroll
  for (int l = 0; l < kLagBlock; ++l) part[l][threadIdx.x] = acc[l];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (int(threadIdx.x) < w)
#pragma unroll
      for (int l = 0; l < kLagBlock; ++l)
        part[l][threadIdx.x] += part[l][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < kLagBlock) {
    const int64_t tau = tau0 + threadIdx.x;
    if (tau < M)
      sd[(traj * M + tau) * nc + c] =
          tau >= 1 ? part[threadIdx.x][0] / double(P - tau) : 0.0;
  }
}

// sd[t, tau, c] from the parts' sums, added in order; eight are read before
// the first is added.
__global__ void __launch_bounds__(256)
msd_scale_kernel(const double* __restrict__ sums, int64_t paths, int64_t P,
                 int nc, int64_t M, int parts, double* __restrict__ sd) {
  const int64_t k = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (k >= paths * M) return;
  const int64_t tau = k % M, path = k / M;
  const int64_t traj = path / nc, c = path % nc;
  const double* from = sums + path * parts * M + tau;
  double v = 0.0;
  if (tau > 0) {
    ExactSum s;
    int p = 0;
    for (; p + 8 <= parts; p += 8) {
      double x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = from[(p + i) * M];
#pragma unroll
      for (int i = 0; i < 8; ++i) s.add(x[i]);
    }
    for (; p < parts; ++p) s.add(from[p * M]);
    v = s.value() / double(P - tau);
  }
  sd[(traj * M + tau) * nc + c] = v;
}

}  // namespace pycd

using namespace pycd;

namespace {

// How a call is shared out: lanes per group (0: msd_short_kernel), workgroups
// per path over its origins and over its lags (one a pass, or one for all),
// the origins of a segment.
struct MsdSplit {
  int kq, seg;
  int64_t parts, passes;
};

// Few paths leave CUs idle with one workgroup each.  Up to kFill of them, the
// passes go to workgroups of their own and the origins to as many parts as
// come to kFill workgroups (8 per CU), of at least kLeast distances each (a
// part costs its window and its sums) and at most kMaxParts, the sums within
// 1 GiB; below 64 paths in the narrowest passes, which there are most of.  In
// origin parts alone, of segments as long as the window allows, 1 path of
// 10001 rows and 5001 lags took 226 us and 20000 x 20000 643; now 44 and 119.
// kFill = 1024: 16 x 16 paths, 2001 rows and lags 193 us, 2048: 186; 16 paths
// of 1001 rows and lags 26 and 30.
//
// The smallest calls are bound by launches and latency: a second kernel that
// adds the parts costs 4 us, and a workgroup's windows and runs 2, so up to
// two workgroups of 8 lags per CU (one where the lags are one pass, which a
// workgroup takes without parts) and 2048 rows take the short kernel: 1 path
// of 1001 rows and 1000 lags 19.6 us against 25.2, 4 x 3 paths of 301 rows
// and 300 lags 18.4 against 23.9, 8 paths of 100 rows and 8 lags 16.5 against
// 18.0; past the lines 8 paths of 1000 rows and 500 lags 29.8 against 26.1,
// 1 path of 2500 rows 25.2 against 24.3, of 50 rows 16.5 against 16.2.
constexpr int64_t kFill = 2048, kLeast = 16384, kMaxParts = 64;

MsdSplit msd_split(int64_t paths, int64_t P, int64_t M) {
  MsdSplit s{0, kMsdWin, 1, 1};
  const int64_t blocks = paths * ((M + kLagBlock - 1) / kLagBlock);
  if (P > 64 && P <= 2048 && blocks <= (M > msd_pass(16) ? 512 : 256) &&
      blocks * P <= 450000)
    return s;
  s.kq = paths < 64 ? 16 : msd_lanes(1, [&](int64_t) {
    return MsdCase{P, M, 1.0};
  });
  const int64_t pass = msd_pass(s.kq);
  if (paths < kFill) s.passes = (M + pass - 1) / pass;
  s.parts = std::max<int64_t>(
      1, std::min({P / (kLeast / std::min(M, pass)),
                   kFill / (paths * s.passes), kMaxParts,
                   (int64_t(1) << 27) / paths / M}));
  if (s.parts > 1) {
    // equal segments, the same number for every part
    const int64_t most =
        s.parts * msd_segment(s.kq, s.passes > 1 ? pass : 0, M);
    const int64_t all = (P + most - 1) / most * s.parts;
    s.seg = int(((P + all - 1) / all + 3) & ~3);
  }
  return s;
}

}  // namespace

extern "C" int pycd_msd(pycd_ctx* ctx, const double* pos, int64_t n_traj,
                        int64_t n_path, int64_t n_carriers, int64_t n_lags,
                        double* sd) {
  if (!ctx) return PYCD_ERR_ARG;
  if (!pos || !sd || n_traj <= 0 || n_path <= 0 || n_carriers <= 0 ||
      n_lags <= 0)
    return fail(ctx, PYCD_ERR_ARG, "bad MSD arguments");
  if (n_lags > n_path)
    return fail(ctx, PYCD_ERR_ARG, "n_lags %lld exceeds n_path %lld",
                (long long)n_lags, (long long)n_path);
  DeviceGuard guard(ctx->device);
  hipStream_t st = ctx->stream;
  const size_t npos = size_t(n_traj) * n_path * n_carriers * 3;
  const size_t nsd = size_t(n_traj) * n_lags * n_carriers;
  WorkBuf<double> dpos, dsd;
  const double* p = pos;
  double* o = sd;
  if (!is_device_ptr(pos)) {
    PYCD_HIP(ctx, dpos.alloc(ctx, npos));
    PYCD_HIP(ctx, hipMemcpyAsync(dpos.ptr, pos, 8 * npos, hipMemcpyHostToDevice,
                                 st));
    p = dpos.ptr;
  }
  const bool out_dev = is_device_ptr(sd);
  if (!out_dev) {
    PYCD_HIP(ctx, dsd.alloc(ctx, nsd));
    o = dsd.ptr;
  }
  const int64_t paths = n_traj * n_carriers;
  const MsdSplit split = msd_split(paths, n_path, n_lags);
  const int64_t parts = split.parts, passes = split.passes;
  const int64_t units = paths * parts * passes;
  if (units > (int64_t(1) << 31) - 1)
    return fail(ctx, PYCD_ERR_ARG, "MSD problem too large for one launch");
  WorkBuf<double> sums;
  if (parts > 1) PYCD_HIP(ctx, sums.alloc(ctx, size_t(paths) * parts * n_lags));
  auto go = [&](auto* kernel) {
    kernel<<<unsigned(units), kMsdThreads, 0, st>>>(
        p, uint32_t(units), n_path, uint32_t(n_carriers), n_lags,
        uint32_t(parts), uint32_t(passes), split.seg, sums.ptr, o);
  };
  if (split.kq == 0)
    msd_short_kernel<<<unsigned(paths * ((n_lags + kLagBlock - 1) / kLagBlock)),
                       256, 0, st>>>(p, n_path, int(n_carriers), n_lags, o);
  else if (split.kq == 64) go(msd_kernel<64>);
  else if (split.kq == 32) go(msd_kernel<32>);
  else go(msd_kernel<16>);
  PYCD_HIP(ctx, hipGetLastError());
  if (parts > 1)
    msd_scale_kernel<<<unsigned((paths * n_lags + 255) / 256), 256, 0, st>>>(
        sums.ptr, paths, n_path, int(n_carriers), n_lags, int(parts), o);
  PYCD_HIP(ctx, hipGetLastError());
  if (!out_dev)
    PYCD_HIP(ctx, hipMemcpyAsync(sd, o, 8 * nsd, hipMemcpyDeviceToHost, st));
  PYCD_HIP(ctx, hipStreamSynchronize(st));
  return PYCD_OK;
}
