// ytm_memory.hip -- device memory kept between calls and large copies to host arrays.
//
// Calls that take host arrays (encode, fit, predict, transform) need device buffers of their
// inputs and outputs for the length of the call.  A hipMalloc and hipFree above 2 MB take 40 to
// 290 us a pair, which for a call of a few hundred microseconds is most of it, and so does a
// small one that finds the runtime's own chunk of small blocks gone; blocks are therefore kept
// here when a call is done with them, up to kKeep bytes a device, and given back by memory_trim
// (ytm_shutdown) or when an allocation fails.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <unordered_map>
#include <vector>

#include "ytm_internal.h"

namespace ytm {

namespace {

constexpr size_t kSmall = (size_t)1 << 20;  // below: powers of two
constexpr size_t kUnit = (size_t)2 << 20;   // from there on: whole units
constexpr size_t kKeep = (size_t)1 << 30;   // idle bytes kept per device

struct Block {
  int device;
  size_t bytes;
};

std::mutex g_mu;
std::unordered_map<void*, Block> g_blocks;             // every block handed out or idle
std::map<int, std::multimap<size_t, void*>> g_idle;    // device -> size -> block
std::map<int, size_t> g_idle_bytes;

// Frees the idle blocks of `device` (-1: of all); the caller holds g_mu.
void trim_locked(int device) {
  int prev = 0;
  (void)hipGetDevice(&prev);
  for (auto& d : g_idle) {
    if (device >= 0 && d.first != device) continue;
    (void)hipSetDevice(d.first);
    for (auto& b : d.second) {
      (void)hipFree(b.second);
      g_blocks.erase(b.second);
    }
    d.second.clear();
    g_idle_bytes[d.first] = 0;
  }
  (void)hipSetDevice(prev);
}

}  // namespace

hipError_t pool_alloc(void** p, size_t bytes) {
  *p = nullptr;
  size_t want = 256;
  if (bytes < kSmall)
    while (want < bytes) want *= 2;
  else
    want = (bytes + kUnit - 1) / kUnit * kUnit;
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(g_mu);
  auto& idle = g_idle[device];
  const auto it = idle.lower_bound(want);
  if (it != idle.end() && it->first <= want + want / 2) {  // at most half as much again is left unused
    *p = it->second;
    g_idle_bytes[device] -= it->first;
    idle.erase(it);
    return hipSuccess;
  }
  e = hipMalloc(p, want);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    trim_locked(device);
    e = hipMalloc(p, want);
  }
  if (e != hipSuccess) return e;
  try {
    g_blocks[*p] = Block{device, want};
  } catch (...) {  // not kept later then
  }
  return e;
}

void pool_free(void* p) {
  if (!p) return;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    const auto it = g_blocks.find(p);
    if (it != g_blocks.end()) {
      const Block b = it->second;
      try {
        if (g_idle_bytes[b.device] + b.bytes <= kKeep) {
          g_idle[b.device].emplace(b.bytes, p);
          g_idle_bytes[b.device] += b.bytes;
          return;
        }
      } catch (...) {  // freed instead
      }
      g_blocks.erase(it);
    }
  }
  (void)hipFree(p);
}

// ------------------------------------------------------------------ copies to host arrays
// A copy of many megabytes into a numpy array that was just allocated runs at 10 GB/s through
// the runtime (its single staging thread also takes the array's page faults); the link
// carries 57 GB/s into pinned memory.  So large copies go piece by piece into pinned buffers,
// and several threads move the pieces on, taking the faults side by side, while the next
// pieces are on their way.  130 MB of encoded images into a fresh array: 18.5 ms through the
// runtime, 8.5 ms so (the operating system's zeroing of the pages: filling them from the CPU
// alone takes as long); 800 MB of TA states 79 -> 21 ms, 44 MB 4.6 -> 1.4 ms.
namespace {

constexpr size_t kPiece = (size_t)1 << 20;
constexpr size_t kStaged = (size_t)4 << 20;  // from here on (below, starting the threads costs as much as it saves)
constexpr int kThreads = 8;

struct Staging {
  int device = -1;
  unsigned char* pinned = nullptr;  // [kThreads][2][kPiece]
  hipStream_t stream[kThreads] = {};
};
std::mutex g_staging_mu;  // held for a whole copy
Staging g_staging;

void release_staging() {
  Staging& s = g_staging;
  if (s.device < 0) return;
  int prev = 0;
  (void)hipGetDevice(&prev);
  (void)hipSetDevice(s.device);
  for (hipStream_t& st : s.stream) {
    if (st) (void)hipStreamDestroy(st);
    st = nullptr;
  }
  if (s.pinned) (void)hipHostFree(s.pinned);
  (void)hipSetDevice(prev);
  s = Staging{};
}

hipError_t ready_staging(int device) {
  if (g_staging.device == device) return hipSuccess;
  release_staging();
  g_staging.device = device;
  hipError_t e = hipHostMalloc((void**)&g_staging.pinned, kThreads * 2 * kPiece, hipHostMallocDefault);
  for (hipStream_t& st : g_staging.stream)
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
  if (e != hipSuccess) release_staging();
  return e;
}

}  // namespace

hipError_t copy_to_host(void* dst, const void* src, size_t bytes, hipStream_t s) {
  std::unique_lock<std::mutex> lock(g_staging_mu, std::defer_lock);
  int device = 0;
  static const int threads =  // asked once: the answer takes longer than a small copy
      (int)std::min<unsigned>(kThreads, std::max(1u, std::thread::hardware_concurrency() / 2));
  // another thread's copy has the buffers, there are few CPUs, or they cannot be had: the
  // runtime's own copy
  if (bytes < kStaged || threads < 2 || hipGetDevice(&device) != hipSuccess || !lock.try_lock() ||
      ready_staging(device) != hipSuccess) {
    (void)hipGetLastError();
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
    return e != hipSuccess ? e : hipStreamSynchronize(s);
  }
  hipError_t e = hipStreamSynchronize(s);  // src is complete
  if (e != hipSuccess) return e;
  const size_t pieces = (bytes + kPiece - 1) / kPiece;
  std::atomic<size_t> next{0};
  std::atomic<int> failed{(int)hipSuccess};
  auto work = [&](int t) {
    if (hipSetDevice(device) != hipSuccess) {
      failed = (int)hipErrorInvalidDevice;
      return;
    }
    unsigned char* buf = g_staging.pinned + (size_t)t * 2 * kPiece;
    const hipStream_t st = g_staging.stream[t];
    size_t before = pieces;  // the piece that lies in the other buffer
    auto move_on = [&](int b) {
      if (before < pieces)
        std::memcpy((unsigned char*)dst + before * kPiece, buf + b * kPiece, std::min(kPiece, bytes - before * kPiece));
    };
    for (int b = 0;; b ^= 1) {
      const size_t i = next++;
      const bool more = i < pieces && failed == (int)hipSuccess;
      if (more) {
        const hipError_t err = hipMemcpyAsync(buf + b * kPiece, (const unsigned char*)src + i * kPiece,
                                              std::min(kPiece, bytes - i * kPiece), hipMemcpyDeviceToHost, st);
        if (err != hipSuccess) failed = (int)err;
      }
      move_on(b ^ 1);
      if (!more) break;
      const hipError_t err = hipStreamSynchronize(st);
      if (err != hipSuccess) failed = (int)err;
      before = i;
    }
    if (failed != (int)hipSuccess) {  // the buffers are used again
      (void)hipStreamSynchronize(st);
      (void)hipGetLastError();
    }
  };
  std::vector<std::thread> others;
  try {
    for (int t = 1; t < threads; ++t) others.emplace_back(work, t);
  } catch (...) {  // no more threads: those there are take every piece
  }
  work(0);
  for (std::thread& t : others) t.join();
  return (hipError_t)failed.load();
}

void memory_trim() {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    trim_locked(-1);
  }
  std::lock_guard<std::mutex> lock(g_staging_mu);
  release_staging();
}

}  // namespace ytm
