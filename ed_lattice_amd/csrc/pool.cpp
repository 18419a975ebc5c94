// Device allocations and the contexts' buffer pools (see pool.hpp).
#include "pool.hpp"

#include <algorithm>
#include <set>

namespace edl {

// Every living pool.  Locked before a pool's own mutex, never after it.
struct Pools {
  std::mutex m;
  std::set<DevPool*> all;
};
static Pools& pools() {
  static Pools* p = new Pools();  // (outlives contexts that are never destroyed)
  return *p;
}

template <typename F>
static size_t on_current_device(F f) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  Pools& P = pools();
  std::lock_guard<std::mutex> g(P.m);
  size_t n = 0;
  for (DevPool* p : P.all)
    if (p->device() == dev) n += f(*p);
  return n;
}

hipError_t device_malloc_bytes(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipErrorOutOfMemory) return e;
  (void)hipGetLastError();
  // (hipFree waits for the device: a cached buffer may have launches queued)
  if (on_current_device([](DevPool& q) { return q.release(); }) == 0) return e;
  e = hipMalloc(p, bytes);
  if (e != hipSuccess) (void)hipGetLastError();
  return e;
}

size_t device_cached_bytes() {
  return on_current_device([](DevPool& q) { return q.cached(); });
}

DevPool::DevPool() {
  std::lock_guard<std::mutex> g(pools().m);
  pools().all.insert(this);
}
DevPool::~DevPool() {
  {
    std::lock_guard<std::mutex> g(pools().m);
    pools().all.erase(this);
  }
  release();
}

void* DevPool::take(size_t bytes) {
  // sizes in steps of an eighth, so that buffers of nearly equal calls match
  size_t step = 512;
  while (step * 16 <= bytes) step *= 2;
  size_t want = (std::max<size_t>(bytes, 1) + step - 1) / step * step;
  // a kept buffer may be larger than asked for, by less where that is much memory
  const size_t over = want <= ((size_t)256 << 20) ? want / 4 : want / 16;
  {
    std::lock_guard<std::mutex> g(m_);
    auto it = free_.lower_bound(want);
    if (it != free_.end() && it->first <= want + over) {
      void* p = it->second;
      cached_ -= it->first;
      live_[p] = it->first;
      free_.erase(it);
      return p;
    }
    if (device_ < 0 && hipGetDevice(&device_) != hipSuccess) {
      (void)hipGetLastError();
      device_ = -1;
    }
  }
  void* p = nullptr;
  if (device_malloc(&p, want) != hipSuccess) {
    // the bytes asked for, without the step
    (void)hipGetLastError();
    want = std::max<size_t>(bytes, 1);
    if (device_malloc(&p, want) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
  }
  std::lock_guard<std::mutex> g(m_);
  live_[p] = want;
  return p;
}

void DevPool::give(void* p) {
  if (!p) return;
  {
    std::lock_guard<std::mutex> g(m_);
    auto it = live_.find(p);
    if (it != live_.end()) {
      const size_t n = it->second;
      live_.erase(it);
      if (!bound_) {
        size_t free_b = 0, total_b = 0;
        if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) (void)hipGetLastError();
        bound_ = std::max<size_t>(total_b / 16, 1);
      }
      if (cached_ + n <= bound_) {
        free_.emplace(n, p);
        cached_ += n;
        return;
      }
    }
  }
  (void)hipFree(p);
}

size_t DevPool::release() {
  std::lock_guard<std::mutex> g(m_);
  for (auto& kv : free_) (void)hipFree(kv.second);
  const size_t n = cached_;
  free_.clear();
  cached_ = 0;
  return n;
}
size_t DevPool::cached() {
  std::lock_guard<std::mutex> g(m_);
  return cached_;
}
int DevPool::device() {
  std::lock_guard<std::mutex> g(m_);
  return device_;
}

DevPool*& current_pool() {
  static thread_local DevPool* p = nullptr;
  return p;
}
void* dev_try_alloc(size_t bytes) {
  if (DevPool* pool = current_pool()) return pool->take(bytes);
  void* p = nullptr;
  if (device_malloc(&p, bytes ? bytes : 4) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  return p;
}
hipError_t dev_upload(void** p, const void* src, size_t bytes, hipStream_t st) {
  *p = dev_try_alloc(bytes);
  if (!*p) return hipErrorOutOfMemory;
  return bytes ? hipMemcpyAsync(*p, src, bytes, hipMemcpyHostToDevice, st) : hipSuccess;
}
void dev_free(void* p) {
  if (!p) return;
  if (DevPool* pool = current_pool())
    pool->give(p);
  else
    (void)hipFree(p);
}

}  // namespace edl
