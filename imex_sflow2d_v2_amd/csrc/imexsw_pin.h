// imexsw_pin.h -- device memory to host arrays through pinned chunks.  Host
// code on a handful of runtime calls, so that its failure paths can be run
// with the runtime replaced.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace imexsw {

// Pinned memory that large downloads pass through: two chunks for the process,
// held while contexts exist and used by one download at a time (another that
// overlaps it copies directly), and two events for each device that a download
// came from.
constexpr size_t kPinChunk = (size_t)4 << 20;
constexpr size_t kPinMin = (size_t)256 << 10;  // downloads below it are copied directly
constexpr int kPinDevices = 64;
struct PinPool {
  std::mutex mu;        // the chunks and events
  std::mutex count_mu;  // users
  int users = 0;
  char* mem = nullptr;
  hipEvent_t ev[kPinDevices][2] = {};
};
static PinPool g_pin;

inline void pin_acquire() {
  std::lock_guard<std::mutex> lk(g_pin.count_mu);
  g_pin.users++;
}
inline void pin_release() {
  std::lock_guard<std::mutex> lk(g_pin.count_mu);
  if (--g_pin.users > 0) return;
  std::lock_guard<std::mutex> lk2(g_pin.mu);
  for (auto& pair : g_pin.ev)
    for (hipEvent_t& e : pair) {
      if (e) (void)hipEventDestroy(e);
      e = nullptr;
    }
  if (g_pin.mem) (void)hipHostFree(g_pin.mem);
  g_pin.mem = nullptr;
}

// The events of `device`, an event belonging to the device current at its
// creation: both or neither.
inline bool pin_events(int device) {
  hipEvent_t* ev = g_pin.ev[device];
  if (ev[0]) return true;
  int cur = 0;
  if (hipGetDevice(&cur) != hipSuccess) return false;
  if (cur != device && hipSetDevice(device) != hipSuccess) return false;
  hipEvent_t e[2] = {nullptr, nullptr};
  bool ok = true;
  for (int i = 0; ok && i < 2; i++)
    ok = hipEventCreateWithFlags(&e[i], hipEventDisableTiming) == hipSuccess;
  if (cur != device) (void)hipSetDevice(cur);
  if (!ok) {
    if (e[0]) (void)hipEventDestroy(e[0]);
    return false;
  }
  ev[0] = e[0];
  ev[1] = e[1];
  return true;
}
// Chunks and events for a download from `device`; without them (false) it
// copies directly.  What could be had is kept, the rest is asked for again by
// the next download.
inline bool pin_ready(int device) {
  if (device < 0 || device >= kPinDevices) return false;
  if (!g_pin.mem &&
      hipHostMalloc((void**)&g_pin.mem, 2 * kPinChunk, hipHostMallocPortable) != hipSuccess)
    g_pin.mem = nullptr;
  if (g_pin.mem && pin_events(device)) return true;
  (void)hipGetLastError();  // handled here: no later call reports it
  return false;
}

// The chunks of one download: chunk i of the device memory arrives in half
// i % 2 of the pinned memory, and the caller and its helpers copy a slice each
// to the host array.
struct ChunkCopy {
  char* host;
  const char* pin;
  size_t bytes, chunks;
  int parts;
  std::atomic<size_t> ready{0};  // chunks that have arrived
  std::atomic<size_t> done[2];   // slices copied out of each half, in all
  std::atomic<bool> stop{false};
  void slice(size_t i, int part) {
    const size_t at = i * kPinChunk, len = std::min(kPinChunk, bytes - at);
    const size_t per = (len / parts + 4095) / 4096 * 4096;
    const size_t o = std::min(len, per * part);
    const size_t n = (part == parts - 1) ? len - o : std::min(per, len - o);
    if (n) std::memcpy(host + at + o, pin + (i & 1) * kPinChunk + o, n);
    done[i & 1].fetch_add(1, std::memory_order_release);
  }
  void help(int part) {
    for (size_t i = 0; i < chunks; i++) {
      while (ready.load(std::memory_order_acquire) <= i) {
        if (stop.load(std::memory_order_acquire)) return;
        std::this_thread::yield();
      }
      slice(i, part);
    }
  }
};

// Device memory to a host array, after the work of `stream`, a stream of
// `device`.  A copy into pageable memory runs at 17 GB/s, and at 10 GB/s into an
// array whose pages are touched for the first time, as an output array's are;
// through pinned chunks the transfer overlaps the copy out of them, which
// several threads make for a large array (they fault its pages side by side).
// The chunks cost the process's first large download 0.2 ms.
inline hipError_t copy_to_host(hipStream_t stream, int device, void* host, const void* dev,
                               size_t bytes) {
  std::unique_lock<std::mutex> lk(g_pin.mu, std::defer_lock);
  if (bytes < kPinMin || !lk.try_lock() || !pin_ready(device)) {
    if (lk.owns_lock()) lk.unlock();
    const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, stream);
    return e == hipSuccess ? hipStreamSynchronize(stream) : e;
  }
  hipEvent_t* ev = g_pin.ev[device];
  ChunkCopy w;
  w.host = static_cast<char*>(host);
  w.pin = g_pin.mem;
  w.bytes = bytes;
  w.chunks = (bytes + kPinChunk - 1) / kPinChunk;
  w.done[0] = w.done[1] = 0;
  // one thread for every 4 MiB, at most 8
  w.parts = (int)std::min<size_t>(8, std::max<size_t>(1, bytes / kPinChunk));
  std::vector<std::thread> helpers;
  int started = 1;
  try {
    helpers.reserve(w.parts);
    // (the slices are fixed before the first helper runs: a helper that
    // cannot be started leaves its slices to the caller)
    for (int p = 1; p < w.parts; p++, started++) helpers.emplace_back([&w, p] { w.help(p); });
  } catch (...) {
  }
  const char* d = static_cast<const char*>(dev);
  auto send = [&](size_t i) -> hipError_t {
    const size_t at = i * kPinChunk;
    hipError_t e = hipMemcpyAsync(g_pin.mem + (i & 1) * kPinChunk, d + at,
                                  std::min(kPinChunk, bytes - at), hipMemcpyDeviceToHost, stream);
    return e == hipSuccess ? hipEventRecord(ev[i & 1], stream) : e;
  };
  hipError_t err = send(0);
  if (err == hipSuccess && w.chunks > 1) err = send(1);
  for (size_t i = 0; err == hipSuccess && i < w.chunks; i++) {
    err = hipEventSynchronize(ev[i & 1]);
    if (err != hipSuccess) break;
    w.ready.store(i + 1, std::memory_order_release);
    w.slice(i, 0);
    for (int p = started; p < w.parts; p++) w.slice(i, p);
    if (i + 2 < w.chunks) {
      // the half is free once every slice of this chunk is out of it
      const size_t want = (size_t)w.parts * (i / 2 + 1);
      while (w.done[i & 1].load(std::memory_order_acquire) < want) std::this_thread::yield();
      err = send(i + 2);
    }
  }
  if (err != hipSuccess) w.stop.store(true, std::memory_order_release);
  for (std::thread& t : helpers) t.join();
  if (err != hipSuccess) (void)hipStreamSynchronize(stream);
  return err;
}

}  // namespace imexsw
