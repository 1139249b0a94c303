// ytm_memory.hip -- device memory kept between calls and large copies to host arrays.
//
// Calls that take host arrays (encode, fit, predict, transform) need device buffers of their
// inputs and outputs for the length of the call.  A hipMalloc and hipFree above 2 MB take 40 to
// 290 us a pair, which for a call of a few hundred microseconds is most of it, and so does a
// small one that finds the runtime's own chunk of small blocks gone; blocks are therefore kept
// here when a call is done with them, up to kKeep bytes a device while a model lives there and
// kKeepAlone otherwise, the longest unused given back first.  (kKeepAlone: a program that has one
// model after the other waits for some ten allocations with each without it, 960 instead of 720
// us for 10 clauses of 24 literals.)  All are given back by memory_trim (ytm_shutdown) and when
// an allocation fails.  Pinned host blocks (a hipHostMalloc takes 50 to 110 us, as long as
// scoring one sample) are kept alike.
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
constexpr size_t kKeep = (size_t)1 << 30;   // idle bytes kept per device, with a model
constexpr size_t kKeepAlone = (size_t)256 << 20;  // and without one
constexpr size_t kKeepPinned = (size_t)64 << 20, kKeepPinnedAlone = (size_t)16 << 20;
constexpr int kDevices = 64;                // devices whose blocks are kept
constexpr int kHost = -1;                   // in a device's place: pinned host memory

struct Block {
  int device;
  size_t bytes;
};
struct Idle {
  void* p;
  uint64_t since;  // count of blocks given back before it
};
struct Pool {
  std::map<size_t, std::vector<Idle>> idle;  // by size, each in the order of `since`
  size_t idle_bytes = 0;
  int models = 0;  // living on the device (kHost: on any)
  size_t keep(int device) const {
    return device == kHost ? (models ? kKeepPinned : kKeepPinnedAlone) : models ? kKeep : kKeepAlone;
  }
};

// Held for the books alone: the runtime's own calls, which may take long, are made outside.
std::mutex g_mu;
std::unordered_map<void*, Block> g_blocks;  // every block handed out or idle
Pool g_pools[kDevices + 1];                 // kHost and the devices
uint64_t g_given_back = 0;

Pool& pool_of(int device) { return g_pools[device + 1]; }

// Takes the longest idle block of a device out of the books while more bytes are idle there than
// are kept (all: any); null when they are not.
void* take_oldest(int device, bool all) {
  std::lock_guard<std::mutex> lock(g_mu);
  Pool& pool = pool_of(device);
  if (pool.idle_bytes <= (all ? 0 : pool.keep(device))) return nullptr;
  auto oldest = pool.idle.end();
  for (auto it = pool.idle.begin(); it != pool.idle.end(); ++it)
    if (!it->second.empty() && (oldest == pool.idle.end() || it->second[0].since < oldest->second[0].since)) oldest = it;
  void* p = oldest->second[0].p;
  pool.idle_bytes -= oldest->first;
  oldest->second.erase(oldest->second.begin());
  if (oldest->second.empty()) pool.idle.erase(oldest);
  g_blocks.erase(p);
  return p;
}

hipError_t take(int device, void** p, size_t bytes) {
  return device == kHost ? hipHostMalloc(p, bytes, hipHostMallocDefault) : hipMalloc(p, bytes);
}
void give(int device, void* p) { (void)(device == kHost ? hipHostFree(p) : hipFree(p)); }

void trim_device(int device, bool all) {
  while (void* p = take_oldest(device, all)) give(device, p);
}

// A block of at least `bytes`, idle or new.
hipError_t alloc_block(int device, void** p, size_t bytes) {
  *p = nullptr;
  size_t want = 256;
  if (bytes < kSmall)
    while (want < bytes) want *= 2;
  else
    want = (bytes + kUnit - 1) / kUnit * kUnit;
  if (device < kDevices) {
    std::lock_guard<std::mutex> lock(g_mu);
    Pool& pool = pool_of(device);
    // at most half as much again is left unused
    for (auto it = pool.idle.lower_bound(want); it != pool.idle.end() && it->first <= want + want / 2; ++it)
      if (!it->second.empty()) {
        *p = it->second.back().p;
        it->second.pop_back();
        pool.idle_bytes -= it->first;
        return hipSuccess;
      }
  }
  hipError_t e = take(device, p, want);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    if (device < kDevices) trim_device(device, true);
    e = take(device, p, want);
  }
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(g_mu);
  try {
    g_blocks[*p] = Block{device, want};
  } catch (...) {  // not kept later then
  }
  return e;
}

void free_block(bool pinned, void* p) {
  if (!p) return;
  int device = kHost;
  bool kept = false, over = false;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    const auto it = g_blocks.find(p);
    if (it != g_blocks.end()) {
      const Block b = it->second;
      device = b.device;
      if (device < kDevices) try {
          Pool& pool = pool_of(device);
          if (b.bytes <= pool.keep(device)) {
            pool.idle[b.bytes].push_back(Idle{p, g_given_back++});
            pool.idle_bytes += b.bytes;
            kept = true;
            over = pool.idle_bytes > pool.keep(device);
          }
        } catch (...) {  // freed instead
        }
      if (!kept) g_blocks.erase(it);
    }
  }
  if (!kept)
    give(pinned ? kHost : 0, p);
  else if (over)
    trim_device(device, false);
}

}  // namespace

hipError_t pool_alloc(void** p, size_t bytes) {
  *p = nullptr;
  int device = 0;
  const hipError_t e = hipGetDevice(&device);
  return e == hipSuccess ? alloc_block(device, p, bytes) : e;
}
void pool_free(void* p) { free_block(false, p); }

hipError_t pinned_alloc(void** p, size_t bytes) { return alloc_block(kHost, p, bytes); }
void pinned_free(void* p) { free_block(true, p); }

bool memory_hold(int device) {
  if (device < 0 || device >= kDevices) return false;
  std::lock_guard<std::mutex> lock(g_mu);
  ++pool_of(device).models;
  ++pool_of(kHost).models;
  return true;
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

// A device's buffers and streams (a program that copies from several devices in turn keeps each
// one's: making them takes milliseconds), until memory_trim.
struct Staging {
  std::mutex mu;  // held for a whole copy
  unsigned char* pinned = nullptr;  // [kThreads][2][kPiece]
  hipStream_t stream[kThreads] = {};
};
Staging g_staging[kDevices];

// Both with g.mu held; ready_staging with the device current.
void release_staging(Staging& g) {
  for (hipStream_t& st : g.stream) {
    if (st) (void)hipStreamDestroy(st);
    st = nullptr;
  }
  if (g.pinned) (void)hipHostFree(g.pinned);
  g.pinned = nullptr;
}

hipError_t ready_staging(Staging& g) {
  if (g.pinned) return hipSuccess;
  hipError_t e = hipHostMalloc((void**)&g.pinned, kThreads * 2 * kPiece, hipHostMallocDefault);
  if (e != hipSuccess) g.pinned = nullptr;
  for (hipStream_t& st : g.stream)
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
  if (e != hipSuccess) release_staging(g);
  return e;
}

void trim_staging(int device) {
  std::lock_guard<std::mutex> lock(g_staging[device].mu);
  release_staging(g_staging[device]);
}

}  // namespace

hipError_t copy_to_host(void* dst, const void* src, size_t bytes, hipStream_t s) {
  std::unique_lock<std::mutex> lock;
  int device = 0;
  static const int threads =  // asked once: the answer takes longer than a small copy
      (int)std::min<unsigned>(kThreads, std::max(1u, std::thread::hardware_concurrency() / 2));
  // another thread's copy has the buffers, there are few CPUs, or they cannot be had: the
  // runtime's own copy
  auto staged = [&] {
    if (bytes < kStaged || threads < 2 || hipGetDevice(&device) != hipSuccess || device >= kDevices) return false;
    lock = std::unique_lock<std::mutex>(g_staging[device].mu, std::try_to_lock);
    return lock.owns_lock() && ready_staging(g_staging[device]) == hipSuccess;
  };
  if (!staged()) {
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
    unsigned char* buf = g_staging[device].pinned + (size_t)t * 2 * kPiece;
    const hipStream_t st = g_staging[device].stream[t];
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

void memory_release(int device) {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    --pool_of(device).models;
    --pool_of(kHost).models;
  }
  trim_device(device, false);
  trim_device(kHost, false);
}

void memory_trim() {
  for (int device = 0; device < kDevices; ++device) {
    trim_device(device, true);
    trim_staging(device);
  }
  trim_device(kHost, true);
}

}  // namespace ytm
