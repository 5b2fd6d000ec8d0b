// Shared host-side plumbing of libpycd_hip.so: context, errors, buffers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/pycd_hip.h"

namespace pycd {

// hipMalloc on the current device, tried again with nothing kept there by
// the workspaces where the device is full.  Every allocation of the library
// goes through it.
inline hipError_t device_malloc(void** out, size_t bytes);

// Memory that the one-shot calls (tables, neighbour lists, displacements)
// of a context work in.  Device blocks are kept from call to call up to
// kMaxKept bytes, oldest given back first, and a page-locked staging buffer
// for small transfers is made with the context; both go with it.  A block
// is free again only when the call that took it is done with the context's
// stream, on which every call works, so that a later call's use is ordered
// after it; any number of threads may take at once.  Kept memory stands in
// no other allocation's way: the library's allocations that find the device
// full are tried again with nothing kept on it (device_malloc).
// (hipFree of a block of 240 MB takes 0.27 ms, hipMalloc 0.04, and copies of
// pageable host memory 0.02-0.09 each: the 12000-site BF16x3 table 5.65 ->
// 4.70 ms, the 6144-site FP32 one 2.20 -> 1.83, the 120-site FP64 one 262 ->
// 177 us.)
class Workspace {
 public:
  static constexpr size_t kMaxKept = size_t(512) << 20;
  static constexpr int kMaxBlocks = 32;
  static constexpr size_t kStaging = size_t(2) << 20;
  // Device blocks are for work on `stream` of `device`.
  hipError_t open(int device, hipStream_t stream) {
    device_ = device;
    stream_ = stream;
    const hipError_t e =
        hipHostMalloc(&staging_, kStaging, hipHostMallocDefault);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lock(open_mu_);
    next_ = open_;
    open_ = this;
    return hipSuccess;
  }
  void close() {
    {
      std::lock_guard<std::mutex> lock(open_mu_);
      for (Workspace** w = &open_; *w; w = &(*w)->next_)
        if (*w == this) {
          *w = next_;
          break;
        }
    }
    clear();
    if (staging_) (void)hipHostFree(staging_);
    staging_ = nullptr;
  }
  // Frees what the open workspaces of `device` keep.  (Not one whose stream
  // is being captured: that stream cannot be waited for.)
  static void give_back(int device) {
    std::lock_guard<std::mutex> lock(open_mu_);
    for (Workspace* w = open_; w; w = w->next_) {
      hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
      if (w->device_ == device &&
          hipStreamIsCapturing(w->stream_, &capture) == hipSuccess &&
          capture == hipStreamCaptureStatusNone)
        w->clear();
    }
  }
  // The smallest kept block of at least `bytes` and at most twice that,
  // else a new one; *got: its size.
  hipError_t take(size_t bytes, void** out, size_t* got) {
    const size_t need = (bytes + 4095) & ~size_t(4095);
    {
      std::lock_guard<std::mutex> lock(mu_);
      int best = -1;
      for (int k = 0; k < n_; ++k)
        if (kept_[k].bytes >= need && kept_[k].bytes / 2 <= need &&
            (best < 0 || kept_[k].bytes < kept_[best].bytes))
          best = k;
      if (best >= 0) {
        const Block b = remove(best);
        *out = b.ptr;
        *got = b.bytes;
        return hipSuccess;
      }
    }
    const hipError_t e = device_malloc(out, need);
    *got = e == hipSuccess ? need : 0;
    return e;
  }
  void give(void* p, size_t bytes) {
    void* out = p;  // what is not kept: a block too large, or the oldest one
    if (bytes <= kMaxKept) {
      std::lock_guard<std::mutex> lock(mu_);
      out = n_ == kMaxBlocks ? remove(0).ptr : nullptr;
      kept_[n_++] = {p, bytes};
      held_ += bytes;
    }
    if (out) release(out);
    while (release_oldest(kMaxKept)) {
    }
  }
  void clear() {
    while (release_oldest(0)) {
    }
  }
  // The staging buffer, or NULL while another call has it.
  void* take_staging() {
    std::lock_guard<std::mutex> lock(mu_);
    if (staging_busy_) return nullptr;
    staging_busy_ = true;
    return staging_;
  }
  void give_staging() {
    std::lock_guard<std::mutex> lock(mu_);
    staging_busy_ = false;
  }

 private:
  struct Block {
    void* ptr;
    size_t bytes;
  };
  Block remove(int k) {  // the lock held
    const Block b = kept_[k];
    held_ -= b.bytes;
    --n_;
    for (; k < n_; ++k) kept_[k] = kept_[k + 1];
    return b;
  }
  bool release_oldest(size_t above) {
    void* p = nullptr;
    {
      std::lock_guard<std::mutex> lock(mu_);
      if (n_ == 0 || held_ <= above) return false;
      p = remove(0).ptr;
    }
    release(p);
    return true;
  }
  void release(void* p) {
    (void)hipStreamSynchronize(stream_);
    (void)hipFree(p);
  }
  // the open workspaces of the process
  static inline std::mutex open_mu_;
  static inline Workspace* open_ = nullptr;
  Workspace* next_ = nullptr;
  std::mutex mu_;
  int device_ = 0;
  hipStream_t stream_ = nullptr;
  Block kept_[kMaxBlocks];  // oldest first
  int n_ = 0;
  size_t held_ = 0;
  void* staging_ = nullptr;
  bool staging_busy_ = false;
};

inline hipError_t device_malloc(void** out, size_t bytes) {
  const hipError_t e = hipMalloc(out, bytes);
  if (e != hipErrorOutOfMemory) return e;
  (void)hipGetLastError();
  int device = 0;
  (void)hipGetDevice(&device);
  Workspace::give_back(device);
  return hipMalloc(out, bytes);
}

}  // namespace pycd

struct pycd_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string error;
  int cu_count = 0;
  double wall_clock_hz = 1e8;  // rate of the kernels' wall_clock64()
  std::vector<uint32_t> simd_keys;  // hardware keys of the SIMDs (probed once)
  // device address of the static scratch of pycd_kmc_advance_static
  double* static_scratch = nullptr;
  // table kernel variant per PYCD_PREC_* (0: the default choice)
  int table_variant[3] = {0, 0, 0};
  pycd::Workspace work;
};

namespace pycd {

// Device address of the plain hop loop's static scratch on `device` (the
// current device), resolved once per device (kmc_plain.hip).
int kmc_static_scratch(int device, double** out);

inline int fail(pycd_ctx* ctx, int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  std::vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  if (ctx) ctx->error = buf;
  return code;
}

#define PYCD_HIP(ctx, expr)                                                   \
  do {                                                                        \
    hipError_t e_ = (expr);                                                   \
    if (e_ != hipSuccess)                                                     \
      return ::pycd::fail((ctx), PYCD_ERR_HIP, "%s failed: %s (%s:%d)", #expr, \
                          hipGetErrorString(e_), __FILE__, __LINE__);         \
  } while (0)

// True when `p` is device (or managed) memory visible to the current device.
inline bool is_device_ptr(const void* p) {
  if (!p) return false;
  hipPointerAttribute_t attr;
  if (hipPointerGetAttributes(&attr, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return attr.type == hipMemoryTypeDevice || attr.type == hipMemoryTypeManaged;
}

// Owned device allocation.
template <typename T>
struct DevBuf {
  T* ptr = nullptr;
  size_t count = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { release(); }
  void release() {
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    count = 0;
  }
  hipError_t alloc(size_t n) {
    release();
    if (n == 0) return hipSuccess;
    void* p = nullptr;
    const hipError_t e = device_malloc(&p, n * sizeof(T));
    if (e == hipSuccess) {
      ptr = static_cast<T*>(p);
      count = n;
    }
    return e;
  }
};

// Device memory of one call, from the context's workspace.  On the way out
// of a call that failed the stream may still hold work on it; the next user
// works on the same stream.
template <typename T>
struct WorkBuf {
  T* ptr = nullptr;
  WorkBuf() = default;
  WorkBuf(const WorkBuf&) = delete;
  WorkBuf& operator=(const WorkBuf&) = delete;
  ~WorkBuf() {
    if (ptr) work_->give(ptr, bytes_);
  }
  // (once per buffer)
  hipError_t alloc(pycd_ctx* ctx, size_t n) {
    if (n == 0) return hipSuccess;
    work_ = &ctx->work;
    void* p = nullptr;
    const hipError_t e = work_->take(n * sizeof(T), &p, &bytes_);
    if (e == hipSuccess) ptr = static_cast<T*>(p);
    return e;
  }

 private:
  Workspace* work_ = nullptr;
  size_t bytes_ = 0;
};

// The context's staging buffer for one call: host data of a few small
// copies side by side.  put()/get() return false when it does not fit (or
// another call has the buffer); the caller then copies from its own memory.
// Results arrive at finish(), after the stream is done.
class Staging {
 public:
  explicit Staging(pycd_ctx* ctx)
      : ctx_(ctx), base_(static_cast<char*>(ctx->work.take_staging())) {}
  ~Staging() {
    if (!base_) return;
    // (no copy of a call that failed is left on the buffer)
    if (pending_) (void)hipStreamSynchronize(ctx_->stream);
    ctx_->work.give_staging();
  }
  Staging(const Staging&) = delete;
  Staging& operator=(const Staging&) = delete;
  bool put(void* dst, const void* src, size_t bytes, hipError_t* e) {
    char* at = room(bytes);
    if (!at) return false;
    std::memcpy(at, src, bytes);
    pending_ = true;
    *e = hipMemcpyAsync(dst, at, bytes, hipMemcpyHostToDevice, ctx_->stream);
    return true;
  }
  bool get(void* dst, const void* src, size_t bytes, hipError_t* e) {
    char* at = n_results_ < kResults ? room(bytes) : nullptr;
    if (!at) return false;
    pending_ = true;
    *e = hipMemcpyAsync(at, src, bytes, hipMemcpyDeviceToHost, ctx_->stream);
    results_[n_results_++] = {dst, at, bytes};
    return true;
  }
  hipError_t finish() {
    const hipError_t e = hipStreamSynchronize(ctx_->stream);
    pending_ = false;
    if (e == hipSuccess)
      for (int k = 0; k < n_results_; ++k)
        std::memcpy(results_[k].dst, results_[k].src, results_[k].bytes);
    n_results_ = 0;
    return e;
  }

 private:
  struct Result {
    void* dst;
    const char* src;
    size_t bytes;
  };
  char* room(size_t bytes) {
    const size_t need = (bytes + 255) & ~size_t(255);
    if (!base_ || need > Workspace::kStaging - used_) return nullptr;
    char* at = base_ + used_;
    used_ += need;
    return at;
  }
  pycd_ctx* ctx_;
  char* base_;
  size_t used_ = 0;
  bool pending_ = false;
  static constexpr int kResults = 4;
  Result results_[kResults];
  int n_results_ = 0;
};

// Copies `n` elements from a host-or-device pointer into device memory.
template <typename T>
hipError_t upload(T* dst, const T* src, size_t n, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipMemcpyKind kind =
      is_device_ptr(src) ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
  return hipMemcpyAsync(dst, src, n * sizeof(T), kind, st);
}

// Copies `n` elements to the device, through the staging buffer where the
// source is host memory that fits it.
template <typename T>
hipError_t stage_up(Staging& stage, T* dst, const T* src, size_t n,
                    hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipError_t e = hipSuccess;
  if (!is_device_ptr(src) && stage.put(dst, src, n * sizeof(T), &e)) return e;
  return upload(dst, src, n, st);
}

template <typename T>
hipError_t download(T* dst, const T* src, size_t n, hipStream_t st) {
  if (n == 0) return hipSuccess;
  hipMemcpyKind kind =
      is_device_ptr(dst) ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost;
  return hipMemcpyAsync(dst, src, n * sizeof(T), kind, st);
}

// e**y with e = 2.718281828459045 (the double numpy's `np.e ** y` raises,
// PyCD/core.py:2047).  That double lies below Euler's number, so
// ln(e_double) = 1 - kLnEDefect and e_double**y = exp(y) exp(-y kLnEDefect)
// = exp(y) (1 - y kLnEDefect) to far below an ulp for any rate exponent
// (|y| < 1e6).  One exp and one FMA instead of an FP64 pow; measured
// against the exactly rounded power, within 3.3e-16 relative for
// y in [-60, 5] (the plain exp alone is off by up to 3.3e-15 there).
constexpr double kLnEDefect = 5.318237706605891e-17;

__host__ __device__ inline double numpy_e_pow(double y) {
  const double e = exp(y);
  return fma(-(y * kLnEDefect), e, e);
}

// e_double**y by Tang's table-driven method (P. T. P. Tang, ACM TOMS 15(2),
// 1989): y = (64 m + j) ln2 / 64 + r with |r| <= ln2 / 128, so
// e**y = 2^m 2^(j/64) e^r, with e^r - 1 by its Taylor polynomial to r^6
// (truncation below 4e-20 relative).  The reduction splits ln2 / 64 after
// Cody and Waite into a head of 36 bits, exact times any |64 m + j| < 2^17,
// and a tail; ln(e_double) = 1 - kLnEDefect enters r, whose ulp is far
// below y kLnEDefect.  Within 1.003 ulp of the exactly rounded e_double**y
// for |y| <= 700 (12 million random arguments, against a long-double
// power); 0 below about -745, inf above 709, NaN for NaN.  `T` holds
// 2^(j/64), j = 0..63, exactly rounded (kExp2J64: the bit patterns of the
// doubles nearest to 2^(j/64), from a 60-digit evaluation).
constexpr uint64_t kExp2J64[64] = {
    0x3ff0000000000000, 0x3ff02c9a3e778061, 0x3ff059b0d3158574, 0x3ff0874518759bc8,
    0x3ff0b5586cf9890f, 0x3ff0e3ec32d3d1a2, 0x3ff11301d0125b51, 0x3ff1429aaea92de0,
    0x3ff172b83c7d517b, 0x3ff1a35beb6fcb75, 0x3ff1d4873168b9aa, 0x3ff2063b88628cd6,
    0x3ff2387a6e756238, 0x3ff26b4565e27cdd, 0x3ff29e9df51fdee1, 0x3ff2d285a6e4030b,
    0x3ff306fe0a31b715, 0x3ff33c08b26416ff, 0x3ff371a7373aa9cb, 0x3ff3a7db34e59ff7,
    0x3ff3dea64c123422, 0x3ff4160a21f72e2a, 0x3ff44e086061892d, 0x3ff486a2b5c13cd0,
    0x3ff4bfdad5362a27, 0x3ff4f9b2769d2ca7, 0x3ff5342b569d4f82, 0x3ff56f4736b527da,
    0x3ff5ab07dd485429, 0x3ff5e76f15ad2148, 0x3ff6247eb03a5585, 0x3ff6623882552225,
    0x3ff6a09e667f3bcd, 0x3ff6dfb23c651a2f, 0x3ff71f75e8ec5f74, 0x3ff75feb564267c9,
    0x3ff7a11473eb0187, 0x3ff7e2f336cf4e62, 0x3ff82589994cce13, 0x3ff868d99b4492ed,
    0x3ff8ace5422aa0db, 0x3ff8f1ae99157736, 0x3ff93737b0cdc5e5, 0x3ff97d829fde4e50,
    0x3ff9c49182a3f090, 0x3ffa0c667b5de565, 0x3ffa5503b23e255d, 0x3ffa9e6b5579fdbf,
    0x3ffae89f995ad3ad, 0x3ffb33a2b84f15fb, 0x3ffb7f76f2fb5e47, 0x3ffbcc1e904bc1d2,
    0x3ffc199bdd85529c, 0x3ffc67f12e57d14b, 0x3ffcb720dcef9069, 0x3ffd072d4a07897c,
    0x3ffd5818dcfba487, 0x3ffda9e603db3285, 0x3ffdfc97337b9b5f, 0x3ffe502ee78b3ff6,
    0x3ffea4afa2a490da, 0x3ffefa1bee615a27, 0x3fff50765b6e4540, 0x3fffa7c1819e90d8};
constexpr double kExpInvL = 92.33248261689366;  // 64 / ln2
constexpr double kExpLhi = __builtin_bit_cast(double, 0x3f862e42fefa0000ull);
constexpr double kExpLlo = __builtin_bit_cast(double, 0x3d1cf79abc9e3b3aull);

__device__ inline double e_pow_tab(double y, const double* __restrict__ T) {
#pragma clang fp contract(off)
  const double kf = rint(y * kExpInvL);
  double r = fma(-kf, kExpLhi, y);
  r = fma(-kf, kExpLlo, r);
  r = fma(-y, kLnEDefect, r);
  const int k = int(kf);
  const double t = T[k & 63];
  double p = fma(1.0 / 720, r, 1.0 / 120);
  p = fma(p, r, 1.0 / 24);
  p = fma(p, r, 1.0 / 6);
  p = fma(p, r, 0.5);
  p = fma(p, r * r, r);
  return ldexp(fma(t, p, t), k >> 6);
}

// The reference's hop rate k = nu e**(-dGs / kT) with
// dGs = (lam + dG0)^2 / (4 lam) - V_ab - 0.5 F.d (PyCD/core.py:2040-2047),
// given i4l = 1 / (4 lam), vs = V_ab + 0.5 F.d and nkt = -1 / kT, each
// formed once and rounded once: the exponent moves by a few ulp, the rate
// by |exponent| 1e-16 relative at most.
__device__ inline double marcus_rate(double g0, double lam, double i4l,
                                     double vs, double nkt, double nu,
                                     const double* __restrict__ T) {
#pragma clang fp contract(off)
  const double t = lam + g0;
  const double gs = t * t * i4l - vs;
  return nu * e_pow_tab(gs * nkt, T);
}

// Scoped device selection.
struct DeviceGuard {
  int prev = 0;
  explicit DeviceGuard(int dev) {
    (void)hipGetDevice(&prev);
    if (prev != dev) (void)hipSetDevice(dev);
  }
  ~DeviceGuard() { (void)hipSetDevice(prev); }
};

}  // namespace pycd
