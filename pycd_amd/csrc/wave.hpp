// Wavefront-wide reductions and scans of FP64 values on gfx950: DPP row
// moves and row broadcasts, no LDS.  Every lane of the wavefront must be
// active.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pycd {

// Cross-lane moves through DPP (rows of 16 lanes): a lane whose source is
// outside its row (bound_ctrl) or whose row is masked off reads 0.
template <int kCtrl, int kRowMask, bool kBound>
__device__ inline double dpp_f64(double v) {
  const int64_t b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, int(b), kCtrl, kRowMask, 0xf,
                                             kBound);
  const int hi = __builtin_amdgcn_update_dpp(0, int(b >> 32), kCtrl, kRowMask,
                                             0xf, kBound);
  return __longlong_as_double((int64_t(uint32_t(hi)) << 32) | uint32_t(lo));
}

constexpr int kDppRowShr = 0x110;     // + n: lane i reads lane i - n of its row
constexpr int kDppWaveShr1 = 0x138;   // lane i reads lane i - 1
constexpr int kDppRowBcast15 = 0x142; // lane 15 of a row to the next row
constexpr int kDppRowBcast31 = 0x143; // lane 31 to rows 2 and 3

// Inclusive prefix sum over the 64 lanes: Hillis-Steele within each row of
// 16, then the row totals carried across rows.
__device__ inline double wave_incl_scan(double v) {
  v += dpp_f64<kDppRowShr + 1, 0xf, true>(v);
  v += dpp_f64<kDppRowShr + 2, 0xf, true>(v);
  v += dpp_f64<kDppRowShr + 4, 0xf, true>(v);
  v += dpp_f64<kDppRowShr + 8, 0xf, true>(v);
  v += dpp_f64<kDppRowBcast15, 0xa, false>(v);
  v += dpp_f64<kDppRowBcast31, 0xc, false>(v);
  return v;
}

__device__ inline double read_lane(double v, int lane) {
  const int64_t b = __double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_readlane(int(b), lane);
  const uint32_t hi = __builtin_amdgcn_readlane(int(b >> 32), lane);
  return __longlong_as_double((int64_t(hi) << 32) | lo);
}

// Sum over the wavefront, returned in a scalar register.
__device__ inline double wave_sum(double v) {
  return read_lane(wave_incl_scan(v), 63);
}

constexpr int kDppRowRor = 0x120;  // + n: rotate each row of 16 by n lanes

__device__ inline uint32_t lo32(double x) {
  return uint32_t(__double_as_longlong(x));
}
__device__ inline uint32_t hi32(double x) {
  return uint32_t(uint64_t(__double_as_longlong(x)) >> 32);
}
__device__ inline double from32(uint32_t lo, uint32_t hi) {
  return __longlong_as_double(int64_t((uint64_t(hi) << 32) | lo));
}

__device__ inline double wave_excl_scan(double v) {
  return dpp_f64<kDppWaveShr1, 0xf, true>(wave_incl_scan(v));
}

}  // namespace pycd
