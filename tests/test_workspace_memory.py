"""Device memory that a context keeps between calls, on a simulated device:
the host code of the library (csrc/common.hpp, csrc/ctx.hip) compiled against
a HIP runtime of a few lines whose device holds 1000 MiB."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "pycd_amd" / "csrc"

RUNTIME = r"""
#pragma once
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#define __host__
#define __device__
#define __global__
#define __forceinline__ inline
#define __restrict__
using std::fma; using std::exp; using std::ldexp; using std::rint;
typedef int hipError_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
typedef struct fakeStream { int device; bool capturing; }* hipStream_t;
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone,
                              hipStreamCaptureStatusActive };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost,
                     hipMemcpyDeviceToDevice, hipMemcpyDefault };
enum hipMemoryType { hipMemoryTypeHost, hipMemoryTypeDevice,
                     hipMemoryTypeManaged };
struct hipPointerAttribute_t { hipMemoryType type; };
struct hipDeviceProp_t { int multiProcessorCount; };
enum { hipStreamNonBlocking = 1, hipHostMallocDefault = 0,
       hipDeviceAttributeWallClockRate = 0 };
namespace sim {
inline size_t used[2] = {0, 0};
inline int current = 0;
inline bool broken = false;  // a capturing stream was waited for
inline size_t mallocs = 0;
inline std::map<void*, std::pair<int, size_t>> blocks;
constexpr size_t kHolds = size_t(1000) << 20;
}
inline hipError_t hipMalloc(void** p, size_t n) {
  if (sim::used[sim::current] + n > sim::kHolds) return hipErrorOutOfMemory;
  *p = std::malloc(1);
  ++sim::mallocs;
  sim::used[sim::current] += n;
  sim::blocks[*p] = {sim::current, n};
  return hipSuccess;
}
inline hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  auto b = sim::blocks.find(p);
  if (b == sim::blocks.end()) return hipErrorInvalidValue;
  sim::used[b->second.first] -= b->second.second;
  sim::blocks.erase(b);
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, int) {
  return (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char* hipGetErrorString(hipError_t) { return "error"; }
inline hipError_t hipGetDevice(int* d) { *d = sim::current; return 0; }
inline hipError_t hipSetDevice(int d) { sim::current = d; return 0; }
inline hipError_t hipGetDeviceCount(int* n) { *n = 2; return hipSuccess; }
inline hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  p->multiProcessorCount = 256;
  return hipSuccess;
}
inline hipError_t hipDeviceGetAttribute(int* v, int, int) {
  *v = 100000;
  return hipSuccess;
}
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, int) {
  *s = new fakeStream{sim::current, false};
  return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s) { delete s; return 0; }
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  if (s->capturing) sim::broken = true;
  return hipSuccess;
}
inline hipError_t hipStreamIsCapturing(hipStream_t s,
                                       hipStreamCaptureStatus* c) {
  *c = s->capturing ? hipStreamCaptureStatusActive
                    : hipStreamCaptureStatusNone;
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind,
                                 hipStream_t) { return hipSuccess; }
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a,
                                          const void*) {
  a->type = hipMemoryTypeHost;
  return hipSuccess;
}
"""

MAIN = r"""
#include "common.hpp"
#include <cstdio>
namespace pycd {
int kmc_static_scratch(int, double** out) { *out = nullptr; return PYCD_OK; }
}
static const size_t kMiB = size_t(1) << 20;
static int failed = 0;
static void check(bool ok, const char* what) {
  if (!ok) { std::printf("FAILED: %s\n", what); ++failed; }
}
// a one-shot call that works in `mib` MiB
static void one_shot(pycd_ctx* ctx, size_t mib) {
  pycd::DeviceGuard g(ctx->device);
  pycd::WorkBuf<char> a;
  check(a.alloc(ctx, mib * kMiB) == hipSuccess, "workspace block");
}
int main() {
  pycd_ctx *a = nullptr, *b = nullptr, *other = nullptr;
  check(pycd_ctx_create(0, &a) == 0 && pycd_ctx_create(0, &b) == 0 &&
        pycd_ctx_create(1, &other) == 0, "contexts");
  void* p = nullptr;
  // what a session, batch or family allocates, from the kept memory of its
  // own context and of another on the device
  one_shot(a, 500);
  one_shot(b, 300);
  one_shot(other, 400);
  check(sim::used[0] == 800 * kMiB, "blocks are kept");
  {
    pycd::DevBuf<char> buf;
    check(buf.alloc(900 * kMiB) == hipSuccess, "a buffer of 900 MiB");
    check(sim::used[0] == 900 * kMiB, "kept memory given back");
    check(sim::used[1] == 400 * kMiB, "the other device's is not touched");
    check(pycd_dev_alloc(a, int64_t(200 * kMiB), &p) == PYCD_ERR_HIP,
          "what does not fit is refused");
  }
  // pycd_dev_alloc
  one_shot(a, 500);
  check(pycd_dev_alloc(b, int64_t(900 * kMiB), &p) == 0, "pycd_dev_alloc");
  check(pycd_dev_free(b, p) == 0, "pycd_dev_free");
  // a one-shot call of another context
  one_shot(a, 500);
  one_shot(b, 900);
  // a context whose stream is being captured keeps its blocks
  one_shot(a, 500);
  a->stream->capturing = true;
  check(pycd_dev_alloc(b, int64_t(900 * kMiB), &p) == PYCD_ERR_HIP,
        "refused while the memory is held by a capturing context");
  a->stream->capturing = false;
  check(!sim::broken, "no capturing stream is waited for");
  check(pycd_dev_alloc(b, int64_t(900 * kMiB), &p) == 0, "afterwards");
  check(pycd_dev_free(b, p) == 0, "pycd_dev_free");
  // calls of many sizes: the oldest blocks make room for the newest
  pycd_ctx_destroy(a);
  check(pycd_ctx_create(0, &a) == 0, "context");
  const size_t others = sim::blocks.size();
  for (int k = 0; k < 100; ++k) {
    pycd::DeviceGuard g(0);
    pycd::WorkBuf<char> one;
    check(one.alloc(a, (size_t(k) * 5 + 1) << 12) == hipSuccess, "block");
  }
  const size_t before = sim::mallocs;
  for (int k = 90; k < 100; ++k) {
    pycd::DeviceGuard g(0);
    pycd::WorkBuf<char> one;
    check(one.alloc(a, (size_t(k) * 5 + 1) << 12) == hipSuccess, "block");
  }
  check(sim::mallocs == before, "the newest sizes are kept");
  check(sim::blocks.size() == others + 32, "no more than 32 blocks are");
  pycd_ctx_destroy(a);
  check(pycd_ctx_create(0, &a) == 0, "context");
  // contexts that are gone
  one_shot(b, 400);
  pycd_ctx_destroy(b);
  check(sim::used[0] == 0, "a context's memory goes with it");
  one_shot(a, 500);
  check(pycd_dev_alloc(a, int64_t(900 * kMiB), &p) == 0, "after a destroy");
  check(pycd_dev_free(a, p) == 0, "pycd_dev_free");
  pycd_ctx_destroy(a);
  pycd_ctx_destroy(other);
  check(sim::blocks.empty(), "nothing is left");
  std::printf("%d failed\n", failed);
  return failed != 0;
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="needs g++")
def test_kept_memory_is_there_for_every_allocation(tmp_path):
    """Sessions, batches and pycd_dev_alloc get what one-shot calls of any
    context on the device keep, as if nothing were kept."""
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "sim"
    res = subprocess.run(
        ["g++", "-std=c++17", "-O1", "-w", "-I", str(tmp_path), "-I",
         str(CSRC), str(tmp_path / "main.cpp"), "-x", "c++",
         str(CSRC / "ctx.hip"), "-o", str(exe), "-lpthread"],
        capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    res = subprocess.run([str(exe)], capture_output=True, text=True,
                         timeout=60)
    assert res.returncode == 0, res.stdout
