// Windowed-origin squared displacement of Analysis.compute_msd on gfx950.
//
//   sd[t, tau, c] = mean_{t0 < P - tau} |r(t0 + tau) - r(t0)|^2
// for every trajectory t, lag tau in [1, M) and carrier c
// (PyCD/core.py:2996-3007); sd[t, 0, c] = 0.
//
// The sums over origins of one carrier's path come from msd_unit (msd.hpp),
// one workgroup per (trajectory, carrier) or, when those are too few to fill
// the chip, several that share its origin segments; their sums are then
// added in order by msd_scale_kernel.  Reading every pair's two positions
// from L2, 32 trajectories of 16 carriers, 10001 rows and 501 lags took
// 13.2 ms; from the LDS windows 0.60 ms, 33 TF/s of its 8 operations per
// distance (FP64 issue allows 0.42 ms at the same clock).
#include "common.hpp"
#include "msd.hpp"

#include <algorithm>

namespace pycd {

// Unit u = (traj parts + part) nc + c.  Workgroup b runs on XCD b mod 8;
// each XCD takes a consecutive range of units, so the carriers of a
// trajectory, which share cache lines of its rows, read them through one L2.
// With one part the means go to sd, else the sums to `sums`.
template <int kQ>
__global__ void __launch_bounds__(kMsdThreads)
__attribute__((amdgpu_waves_per_eu(4, 4)))
msd_kernel(const double* __restrict__ pos, int64_t units, int64_t P, int nc,
           int64_t M, int parts, double* __restrict__ sums,
           double* __restrict__ sd) {
  const int64_t b = blockIdx.x, per = units / kMsdXcds;
  const int64_t u = b < per * kMsdXcds ? b % kMsdXcds * per + b / kMsdXcds : b;
  const int c = int(u % nc);
  const int part = int(u / nc % parts);
  const int64_t traj = u / nc / parts;
  const int64_t w3 = 3 * int64_t(nc);
  msd_unit<kQ>(
      (const __attribute__((address_space(1))) double*)(pos + traj * P * w3 +
                                                        3 * c),
      w3, P, M, part, parts, [&](int64_t tau, double v) {
        if (parts > 1)
          sums[u * M + tau] = v;
        else
          sd[(traj * M + tau) * nc + c] = tau > 0 ? v / double(P - tau) : 0.0;
      });
}

// sd[t, tau, c] from the parts' sums, added in order.
__global__ void __launch_bounds__(256)
msd_scale_kernel(const double* __restrict__ sums, int64_t paths, int64_t P,
                 int nc, int64_t M, int parts, double* __restrict__ sd) {
  const int64_t k = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (k >= paths * M) return;
  const int64_t tau = k % M, path = k / M;
  const int64_t traj = path / nc, c = path % nc;
  double v = 0.0;
  if (tau > 0) {
    ExactSum s;
    for (int p = 0; p < parts; ++p)
      s.add(sums[((traj * parts + p) * nc + c) * M + tau]);
    v = s.value() / double(P - tau);
  }
  sd[(traj * M + tau) * nc + c] = v;
}

}  // namespace pycd

using namespace pycd;

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
  // origin segments shared by `parts` workgroups, so that about 2048 (8 per
  // CU) are there where the paths allow, the sums within 1 GiB
  const int kq = msd_lanes(1, [&](int64_t) {
    return std::make_pair(n_lags, 1.0);
  });
  const int64_t paths = n_traj * n_carriers;
  const int64_t S = msd_segment(kq, 0, n_lags);
  const int64_t parts = std::max<int64_t>(
      1, std::min({(n_path + S - 1) / S, int64_t(2048) / paths,
                   (int64_t(1) << 27) / paths / n_lags}));
  const int64_t units = paths * parts;
  if (units > (int64_t(1) << 31) - 1)
    return fail(ctx, PYCD_ERR_ARG, "MSD problem too large for one launch");
  WorkBuf<double> sums;
  if (parts > 1) PYCD_HIP(ctx, sums.alloc(ctx, size_t(units) * n_lags));
  auto go = [&](auto* kernel) {
    kernel<<<unsigned(units), kMsdThreads, 0, st>>>(
        p, units, n_path, int(n_carriers), n_lags, int(parts), sums.ptr, o);
  };
  if (kq == 64) go(msd_kernel<64>);
  else if (kq == 32) go(msd_kernel<32>);
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
