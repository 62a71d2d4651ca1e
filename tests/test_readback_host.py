"""The read-back object on the CPU: its header compiled against a stand-in for
the runtime that counts device and pinned bytes and refuses them past a limit.
Small reads hold what they need and no more, planes go in few copies, a card with little memory left is
read in small pieces, and reads without pinned memory or threads still work."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lbmflow_amd", "csrc")

RUNTIME = r"""
#pragma once
#include <cstdlib>
#include <cstring>
#include <map>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
typedef void* hipStream_t;
typedef int* hipEvent_t;
enum { hipMemcpyDeviceToHost, hipEventDisableTiming = 2, hipEventReleaseToSystem = 4, hipHostMallocCoherent = 8 };
inline hipError_t last = hipSuccess;
struct Pool {
  size_t used = 0, limit = ~(size_t)0;
  std::map<void*, size_t> held;
  hipError_t get(void** p, size_t n) {
    if (used + n > limit) return last = hipErrorOutOfMemory;
    *p = malloc(n);
    held[*p] = n;
    used += n;
    return hipSuccess;
  }
  hipError_t put(void* p) {
    used -= held.at(p);
    held.erase(p);
    free(p);
    return hipSuccess;
  }
};
inline Pool dev, pinned;
inline int events = 0, copies = 0;
template <typename T> hipError_t hipMalloc(T** p, size_t n) { return dev.get((void**)p, n); }
inline hipError_t hipFree(void* p) { return dev.put(p); }
inline hipError_t hipHostMalloc(void** p, size_t n, int) { return pinned.get(p, n); }
inline hipError_t hipHostFree(void* p) { return pinned.put(p); }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
  ++copies;
  memcpy(d, s, n);
  return hipSuccess;
}
namespace lbm {
inline hipError_t launch_to_host(void* d, const void* s, size_t n, hipStream_t t) { return hipMemcpyAsync(d, s, n, 0, t); }
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) { ++events; *e = new int; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { --events; delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
"""

MAIN = r"""
#include "lbm_readback.hpp"
#include <cstdio>
using lbm::Readback;
static int pieces;
static bool read_ok(Readback& rb, uint32_t n, uint32_t planes) {
  std::vector<float> out((size_t)n * planes, -1.0f);
  pieces = copies = 0;
  const hipError_t e = rb.read_planes(0, nullptr, n, planes, [&](uint32_t k) { return out.data() + (size_t)k * n; },
                                      [&](uint32_t i0, uint32_t cnt, float* w) {
    ++pieces;
    for (uint32_t k = 0; k < planes; ++k)
      for (uint32_t j = 0; j < cnt; ++j) w[(size_t)k * cnt + j] = (float)((i0 + j) % 65521u) + 0.5f * k;
    return hipSuccess;
  });
  if (e != hipSuccess) return false;
  for (uint32_t k = 0; k < planes; ++k)
    for (uint32_t i = 0; i < n; ++i)
      if (out[(size_t)k * n + i] != (float)(i % 65521u) + 0.5f * k) return false;
  return true;
}
#define CHECK(c) if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; }
int main() {
  const size_t MiB = (size_t)1 << 20;
  {
    Readback rb;  // small reads hold little, larger ones grow to the bounds
    CHECK(read_ok(rb, 105, 4) && dev.used <= MiB / 8 && pinned.used <= 2 * MiB && pieces == 1);
    CHECK(read_ok(rb, 32768, 27) && dev.used <= 4 * MiB && pieces == 1);
    CHECK(copies == 2);  // planes that lie together go in one copy per slot
    CHECK(read_ok(rb, 9000001, 4) && dev.used == 64 * MiB && pinned.used == 48 * MiB && pieces == 3);
    CHECK(copies <= 69 + 3);
    CHECK(read_ok(rb, 105, 27) && dev.used == 64 * MiB && copies == 1);
  }
  CHECK(dev.used == 0 && pinned.used == 0 && events == 0);
  {
    Readback rb;  // a nearly full card
    dev.limit = 3 * MiB;
    CHECK(read_ok(rb, 1000003, 4) && dev.used <= 3 * MiB && pieces > 4);
    dev.limit = 100000;
    Readback tight;
    dev.limit = dev.used + 100000;
    CHECK(read_ok(tight, 100003, 27));
    dev.limit = 0;
    Readback none;
    CHECK(!read_ok(none, 105, 4) && pieces == 0);
    dev.limit = ~(size_t)0;
    CHECK(read_ok(none, 105, 4));
  }
  CHECK(dev.used == 0 && pinned.used == 0 && events == 0);
  {
    Readback rb;  // no pinned memory, then only a little
    pinned.limit = 0;
    CHECK(read_ok(rb, 105, 4) && read_ok(rb, 3000001, 4));
    pinned.limit = 2 * MiB;
    Readback few;
    CHECK(read_ok(few, 105, 4) && pinned.used > 0 && read_ok(few, 3000001, 4) && read_ok(few, 105, 4));
  }
  CHECK(dev.used == 0 && pinned.used == 0 && events == 0);
  {
    Readback rb;  // an allocation takes back what the read-back keeps; a refused one leaves no error behind
    pinned.limit = ~(size_t)0;
    CHECK(read_ok(rb, 9000001, 4) && dev.used == 64 * MiB);
    dev.limit = 70 * MiB;
    float *p = nullptr, *q = nullptr;
    CHECK(lbm::gpu_malloc(&p, 32 * MiB, &rb) == hipSuccess && dev.used == 32 * MiB);
    CHECK(lbm::gpu_malloc(&q, 64 * MiB, &rb) == hipErrorOutOfMemory && q == nullptr);
    CHECK(lbm::gpu_malloc(&q, 64 * MiB) == hipErrorOutOfMemory && q == nullptr);
    CHECK(read_ok(rb, 9000001, 4) && dev.used <= 70 * MiB);
    hipFree(p);
  }
  CHECK(last == hipSuccess);
  CHECK(dev.used == 0 && pinned.used == 0 && events == 0);
  return 0;
}
"""


def test_readback_holds_what_it_needs(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "readback"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", f"-I{tmp_path}", f"-I{CSRC}", str(tmp_path / "main.cpp"),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
