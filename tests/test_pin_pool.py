"""Downloads through pinned chunks (imexsw_pin.h) with the runtime replaced by
a host one that can refuse what it is asked for: a download succeeds whatever
of the pool cannot be had, nothing stays half built, events belong to the
stream's device, and the last user gives everything back.  CPU only."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "imex_sflow2d_v2_amd", "csrc")

RUNTIME = r"""
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400 };
enum { hipMemcpyDeviceToHost = 2, hipEventDisableTiming = 2, hipHostMallocPortable = 1 };
struct Ev { int device; };
struct St { int device; };
typedef Ev* hipEvent_t;
typedef St* hipStream_t;
// what the next calls refuse, and what is alive
inline int g_fail_malloc = 0, g_fail_event = -1, g_fail_copy = -1;
inline int g_mallocs = 0, g_live_mem = 0, g_live_events = 0;
inline std::atomic<int> g_direct{0};
inline thread_local int g_device = 0;
inline thread_local hipError_t g_last = hipSuccess;
inline hipError_t ret(hipError_t e) { if (e) g_last = e; return e; }
inline hipError_t hipGetLastError() { hipError_t e = g_last; g_last = hipSuccess; return e; }
inline hipError_t hipGetDevice(int* d) { *d = g_device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { g_device = d; return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned = 0) {
  if (g_fail_malloc) return ret(hipErrorOutOfMemory);
  g_mallocs++, g_live_mem++;
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) { g_live_mem--; std::free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  if (g_fail_event == 0) { g_fail_event = -1; return ret(hipErrorOutOfMemory); }
  if (g_fail_event > 0) g_fail_event--;
  g_live_events++;
  *e = new Ev{g_device};
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { g_live_events--; delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  return ret(e && e->device == s->device ? hipSuccess : hipErrorInvalidHandle);
}
inline hipError_t hipEventSynchronize(hipEvent_t e) { return ret(e ? hipSuccess : hipErrorInvalidHandle); }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
  if (g_fail_copy == 0) { g_fail_copy = -1; return ret(hipErrorInvalidHandle); }
  if (g_fail_copy > 0) g_fail_copy--;
  if (n > ((size_t)4 << 20)) g_direct++;
  std::memcpy(d, s, n);
  return hipSuccess;
}
"""

MAIN = r"""
#include "imexsw_pin.h"
#include <cstdio>
#include <numeric>
using namespace imexsw;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)
static std::vector<char> dev;
static bool get(int device, size_t n, hipError_t want = hipSuccess) {
  St s{device};
  std::vector<char> host(n + 1, 1);
  const hipError_t e = copy_to_host(&s, device, host.data(), dev.data(), n);
  if (e != want) { std::printf("error %d\n", (int)e); return false; }
  return e != hipSuccess || (!std::memcmp(host.data(), dev.data(), n) && host[n] == 1);
}
int main() {
  dev.resize((size_t)41 << 20);
  unsigned x = 1;
  for (char& c : dev) c = (char)((x = x * 1664525u + 1013904223u) >> 24);
  const size_t big = 2 * kPinChunk + 4099;

  // nothing can be pinned: a plain copy, no error left behind
  pin_acquire();
  g_fail_malloc = 1;
  CHECK(get(0, big) && g_direct == 1 && hipGetLastError() == hipSuccess);
  g_fail_malloc = 0;
  // the first, then the second event cannot be created: the same, nothing kept of the pair
  for (int i = 0; i < 2; i++) {
    g_fail_event = i;
    CHECK(get(0, big) && g_direct == 2 + i && hipGetLastError() == hipSuccess);
    CHECK(g_live_events == 0);
  }
  // and the next download has its chunks
  CHECK(get(0, big) && g_direct == 3 && g_live_events == 2 && g_mallocs == 1);

  // sizes around the chunks'
  for (size_t n : {kPinMin - 1, kPinMin, kPinChunk - 1, kPinChunk, kPinChunk + 1, 2 * kPinChunk,
                   3 * kPinChunk + 17, 8 * kPinChunk + 1, 10 * kPinChunk - 4097})
    CHECK(get(0, n) && g_direct == 3);

  // a stream of another device than the thread's: events of its device, the
  // thread's device as it was, the same chunks
  CHECK(get(1, big) && g_direct == 3 && g_device == 0 && g_live_events == 4);
  CHECK(get(0, big) && get(1, big) && g_mallocs == 1);
  // a device the pool has no place for
  CHECK(get(kPinDevices, big) && g_direct == 4);

  // a transfer fails on the way: reported, helpers ended, the pool usable
  for (int at : {0, 1, 2, 5}) {
    g_fail_copy = at;
    CHECK(get(0, 8 * kPinChunk, hipErrorInvalidHandle));
    CHECK(get(0, big));
  }

  // downloads that overlap
  std::vector<std::thread> ts;
  std::atomic<int> ok{0};
  for (int t = 0; t < 4; t++) {
    pin_acquire();
    ts.emplace_back([&, t] {
      for (int r = 0; r < 3; r++) ok += get(t & 1, big + 1000 * t);
      pin_release();
    });
  }
  for (auto& t : ts) t.join();
  CHECK(ok == 12 && g_mallocs == 1);

  pin_release();
  CHECK(g_live_mem == 0 && g_live_events == 0);
  pin_acquire();
  CHECK(get(0, big) && g_live_mem == 1);
  pin_release();
  CHECK(g_live_mem == 0 && g_live_events == 0);
  std::printf("ok\n");
}
"""


def test_downloads_without_the_pool(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = str(tmp_path / "pin")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-pthread", "-I", str(tmp_path), "-I", CSRC,
                           "-o", exe, str(tmp_path / "main.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
