// Device memory of this library: allocations that take cached memory back
// before they fail, and the buffers a context keeps between its calls.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <exception>
#include <map>
#include <mutex>

namespace edl {

// hipMalloc.  Where the device has no memory left, the cached buffers of every
// context on it are freed and the allocation is tried once more: memory that no
// call is using never makes one fail.  A request that fails for memory leaves no
// error pending: the launches of the next call look for theirs.
hipError_t device_malloc_bytes(void** p, size_t bytes);
template <typename P>
hipError_t device_malloc(P** p, size_t bytes) {
  void* q = nullptr;
  const hipError_t e = device_malloc_bytes(&q, bytes);
  if (e == hipSuccess) *p = static_cast<P*>(q);
  return e;
}
// Bytes cached by the contexts on the current device.
size_t device_cached_bytes();

// Device buffers of finished calls, kept by their context for its next ones
// (a hipMalloc or hipFree of small buffers costs 5 to 10 us each and waits for
// the device, a gigabyte that was in use before about 25 ms).  Bounded: at most
// a sixteenth of the device's memory stays cached, the rest is freed at once; given back
// when the context is destroyed, takes a model of another number of sites, or
// an allocation of this library on the device fails (device_malloc, from any
// context and thread).  All work of a context is ordered on
// its stream, copies into its buffers too (dev_upload), so a buffer put back
// while launches that use it are queued is safe to hand to later launches; a
// call's other streams are joined before their buffers go back, and a call that
// ends with an exception waits for the device (PoolScope).
class DevPool {
 public:
  DevPool();
  ~DevPool();
  DevPool(const DevPool&) = delete;
  DevPool& operator=(const DevPool&) = delete;
  void* take(size_t bytes);       // nullptr when the device has no memory
  void give(void* p);             // p from take of any pool, or from hipMalloc
  size_t release();               // frees what is cached; its bytes
  size_t cached();
  int device();                   // of its buffers; -1 before the first

 private:
  std::mutex m_;
  std::multimap<size_t, void*> free_;
  std::map<void*, size_t> live_;
  size_t cached_ = 0, bound_ = 0;
  int device_ = -1;
};
// The pool of the context whose call this thread is in (set by PoolScope),
// null outside: dev_try_alloc and dev_free then allocate and free directly.
DevPool*& current_pool();
struct PoolScope {
  DevPool* before;
  int unwinding = std::uncaught_exceptions();
  explicit PoolScope(DevPool& p) : before(current_pool()) { current_pool() = &p; }
  ~PoolScope() {
    // the buffers of the call are back in the pool, with launches on any of its
    // streams still queued: none may be handed out before those have run
    if (std::uncaught_exceptions() > unwinding) (void)hipDeviceSynchronize();
    current_pool() = before;
  }
  PoolScope(const PoolScope&) = delete;
  PoolScope& operator=(const PoolScope&) = delete;
};
void* dev_try_alloc(size_t bytes);  // nullptr (no error left pending) when there is no memory
void dev_free(void* p);
// dev_try_alloc and a copy of host memory into it, on the stream: the copy comes
// after the launches queued there that a kept buffer may still serve.  `src` has
// to live until the stream is waited for.
hipError_t dev_upload(void** p, const void* src, size_t bytes, hipStream_t st);

}  // namespace edl
