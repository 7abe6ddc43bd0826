// Blocks of closed handles, kept for the next call.  A call allocates ~80
// buffers (several hundred with the MG solver), and mapping and unmapping
// them took about 3 ms of a 4,096-element call and 25 ms of a 1M-element one.
// A block enters the pool only when the work that used it has finished
// (rsb_pool_release), so it may go to any thread and stream; the pool holds
// at most most_idle bytes per device, gives back blocks that kPoolIdle
// closes have not asked for, empties itself when the device runs out of
// memory, and gives everything back when the caller asks
// (rsbgpu_release_memory).
#include "runtime.hpp"

#include <sched.h>

#include <algorithm>
#include <cstdlib>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "rsbgpu.h"

namespace {

constexpr int kMaxDevices = 64;
constexpr unsigned long long kPoolIdle = 16;
constexpr size_t kPoolStreams = 8;

struct pool_block {
  void *p;
  unsigned long long tick;  // close count when it came in
};
struct dev_pool {
  std::multimap<size_t, pool_block> idle;  // by size
  size_t held = 0, live = 0, peak = 0;     // bytes idle, in use; the most of both
  unsigned long long tick = 0;
  std::vector<rsb_stream_set> streams;
  void in_use(size_t size) { live += size, peak = std::max(peak, live + held); }
};
// 4 GiB hold a call of 1M elements whole and all but the largest buffers of
// a 16.7M-element one.
constexpr size_t kPoolBytes = 4ull << 30, kNoLimit = ~(size_t)0;
struct pool_state {
  std::mutex mu;
  size_t most_idle = kPoolBytes, most = kNoLimit;  // bytes per device (rsb_pool_settings)
  std::unordered_map<const void *, std::pair<size_t, int>> live;  // size, device
  dev_pool dev[kMaxDevices];
};
pool_state &pool() {
  static pool_state *s = new pool_state();  // never destroyed: threads may outlive main
  return *s;
}

// Sizes in steps of an eighth of their power of two (at least 4 KiB), so
// that buffers of nearly equal sizes can take each other's place.
size_t pool_size(size_t bytes) {
  size_t step = 4096;
  while (step * 16 <= bytes) step *= 2;
  return (std::max<size_t>(bytes, 1) + step - 1) / step * step;
}

// hipMalloc within the limit on bytes in use and idle.  A failure leaves no
// error behind for a later launch check to find.
hipError_t device_malloc(const dev_pool &d, void **p, size_t bytes) {
  {
    std::lock_guard<std::mutex> lock(pool().mu);
    const size_t most = pool().most, used = d.live + d.held;
    if (used > most || bytes > most - used) return hipErrorOutOfMemory;
  }
  const hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
  }
  return e;
}

// Blocks idle since before `before` leave the pool (mu held); the caller
// frees them without the lock, since every free waits for the device.
std::vector<void *> pool_trim(dev_pool &d, unsigned long long before) {
  std::vector<void *> out;
  for (auto it = d.idle.begin(); it != d.idle.end();) {
    if (it->second.tick < before) {
      d.held -= it->first;
      out.push_back(it->second.p);
      it = d.idle.erase(it);
    } else {
      ++it;
    }
  }
  return out;
}
void free_all(const std::vector<void *> &v) {
  for (void *p : v) (void)hipFree(p);
}

}  // namespace

void rsb_pool_settings(void) {
  auto mib = [](const char *name, size_t unset) {
    const char *v = getenv(name);
    return v && *v ? (size_t)std::max(0ll, atoll(v)) << 20 : unset;
  };
  const size_t idle = mib("PARRSB_AMD_POOL_MB", kPoolBytes);
  const size_t most = mib("PARRSB_AMD_MEM_LIMIT_MB", kNoLimit);
  pool_state &s = pool();
  std::lock_guard<std::mutex> lock(s.mu);
  s.most_idle = idle, s.most = most;
}

hipError_t rsb_pool_malloc(void **p, size_t bytes) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipMalloc(p, bytes);
  const size_t need = pool_size(bytes);
  pool_state &s = pool();
  dev_pool &d = s.dev[dev];
  {
    std::lock_guard<std::mutex> lock(s.mu);
    auto it = d.idle.lower_bound(need);
    if (it != d.idle.end() && it->first <= 2 * need) {
      *p = it->second.p;
      s.live[*p] = {it->first, dev};
      d.held -= it->first;
      d.in_use(it->first);
      d.idle.erase(it);
      return hipSuccess;
    }
  }
  // the rounded size; with the pool emptied; the exact size
  size_t size = need;
  e = device_malloc(d, p, size);
  if (e != hipSuccess) {
    std::vector<void *> idle;
    {
      std::lock_guard<std::mutex> lock(s.mu);
      idle = pool_trim(d, ~0ull);
    }
    free_all(idle);
    e = device_malloc(d, p, size);
    if (e != hipSuccess) e = device_malloc(d, p, size = bytes);
    if (e != hipSuccess) return e;
  }
  std::lock_guard<std::mutex> lock(s.mu);
  s.live[*p] = {size, dev};
  d.in_use(size);
  return hipSuccess;
}

hipError_t rsb_pool_free(const void *p) {
  if (!p) return hipSuccess;
  pool_state &s = pool();
  {
    std::lock_guard<std::mutex> lock(s.mu);
    auto it = s.live.find(p);
    if (it != s.live.end()) {
      s.dev[it->second.second].live -= it->second.first;
      s.live.erase(it);
    }
  }
  return hipFree((void *)p);
}

void rsb_pool_release(const void *p) {
  if (!p) return;
  pool_state &s = pool();
  {
    std::lock_guard<std::mutex> lock(s.mu);
    auto it = s.live.find(p);
    if (it != s.live.end()) {
      const size_t size = it->second.first;
      dev_pool &d = s.dev[it->second.second];
      s.live.erase(it);
      d.live -= size;
      if (d.held + size <= s.most_idle) {
        d.idle.emplace(size, pool_block{(void *)p, d.tick});
        d.held += size;
        return;
      }
    }
  }
  (void)hipFree((void *)p);
}

bool rsb_drain_release(hipStream_t st, const std::vector<const void *> &blocks) {
  const bool drained = st && hipStreamSynchronize(st) == hipSuccess;
  for (const void *p : blocks) {
    if (drained) rsb_dev_release(p);
    else (void)rsb_dev_free(p);
  }
  return drained;
}

bool rsb_pool_take_streams(int device, rsb_stream_set *out) {
  if (device < 0 || device >= kMaxDevices) return false;
  pool_state &s = pool();
  std::lock_guard<std::mutex> lock(s.mu);
  auto &v = s.dev[device].streams;
  if (v.empty()) return false;
  *out = v.back();
  v.pop_back();
  return true;
}

bool rsb_pool_give_streams(int device, const rsb_stream_set &in) {
  if (device < 0 || device >= kMaxDevices) return false;
  pool_state &s = pool();
  std::lock_guard<std::mutex> lock(s.mu);
  auto &v = s.dev[device].streams;
  if (v.size() >= kPoolStreams || s.most_idle == 0) return false;
  v.push_back(in);
  return true;
}

void rsb_destroy_streams(const rsb_stream_set &s) {
  for (hipEvent_t e : s.ev)
    if (e) (void)hipEventDestroy(e);
  if (s.stream) (void)hipStreamDestroy(s.stream);
  if (s.ring) (void)hipHostFree(s.ring);
}

void rsb_pool_tick(int device) {
  if (device < 0 || device >= kMaxDevices) return;
  pool_state &s = pool();
  std::vector<void *> old;
  {
    std::lock_guard<std::mutex> lock(s.mu);
    dev_pool &d = s.dev[device];
    if (++d.tick > kPoolIdle) old = pool_trim(d, d.tick - kPoolIdle);
  }
  free_all(old);
}

extern "C" long long rsbgpu_release_memory(void) {
  pool_state &s = pool();
  size_t freed = 0;
  std::vector<void *> blocks;
  std::vector<rsb_stream_set> streams;
  {
    std::lock_guard<std::mutex> lock(s.mu);
    for (dev_pool &d : s.dev) {
      freed += d.held;
      const std::vector<void *> idle = pool_trim(d, ~0ull);
      blocks.insert(blocks.end(), idle.begin(), idle.end());
      streams.insert(streams.end(), d.streams.begin(), d.streams.end());
      d.streams.clear();
      d.peak = d.live;
    }
  }
  free_all(blocks);
  for (const rsb_stream_set &x : streams) rsb_destroy_streams(x);
  return (long long)freed;
}

extern "C" int rsbgpu_memory(int device, int64_t *out) {
  if (device < 0 || device >= kMaxDevices) return 3;
  pool_state &s = pool();
  std::lock_guard<std::mutex> lock(s.mu);
  const dev_pool &d = s.dev[device];
  out[0] = (int64_t)d.live, out[1] = (int64_t)d.held, out[2] = (int64_t)d.peak;
  return 0;
}

unsigned rsb_schedule(void) {
  unsigned f = 0;
  if (hipGetDeviceFlags(&f) != hipSuccess) {
    (void)hipGetLastError();
    f = hipDeviceScheduleAuto;
  }
  return f & hipDeviceScheduleMask;
}

// Most reports arrive within microseconds of the look, so a thread that wants
// to sleep looks for about as long first (kLooks) before it does.
hipError_t rsb_await(hipStream_t st, const int *flag, unsigned schedule) {
  constexpr unsigned kLooks = 1u << 10, kQuery = 1u << 16;
  const bool yields = schedule == hipDeviceScheduleYield;
  for (unsigned q = 1;; q++) {
    if (__atomic_load_n(flag, __ATOMIC_ACQUIRE)) return hipSuccess;
    if (schedule == hipDeviceScheduleBlockingSync && q == kLooks) {
      const hipError_t e = hipStreamSynchronize(st);
      if (e != hipSuccess) return e;
      return __atomic_load_n(flag, __ATOMIC_ACQUIRE) ? hipSuccess : hipErrorNotReady;
    }
    if (yields) sched_yield();
    else __builtin_ia32_pause();
    if (q % (yields ? kLooks : kQuery) == 0) {
      // a failed launch or a fault never sets it: ask the stream
      const hipError_t e = hipStreamQuery(st);
      if (e == hipErrorNotReady) {
        (void)hipGetLastError();
        continue;
      }
      if (e != hipSuccess) return e;
      return __atomic_load_n(flag, __ATOMIC_ACQUIRE) ? hipSuccess : hipErrorNotReady;
    }
  }
}
