"""The contexts' buffer pools over a small simulated device (host compiler, no GPU)."""
import glob
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ed_lattice_amd", "csrc")

# two devices of 16 MiB; an allocation past it fails and leaves an error pending
RUNTIME = r"""
#pragma once
#include <cstdlib>
#include <cstdint>
#include <map>
#include <mutex>
#include <utility>
#include <vector>
typedef int hipError_t;
typedef void* hipStream_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
struct Sim {
  std::recursive_mutex m;
  size_t total = (size_t)16 << 20, used[2] = {0, 0};
  std::map<void*, std::pair<int, size_t>> at;
  int pending = 0, syncs = 0;
  // launches and copies queued and not waited for: stream, buffer
  std::vector<std::pair<void*, void*>> queued;
  std::vector<void*> late;  // buffers written while another stream still used them
};
inline Sim& sim() { static Sim s; return s; }
inline int& sim_device() { static thread_local int d = 0; return d; }
inline hipError_t hipGetDevice(int* d) { *d = sim_device(); return hipSuccess; }
inline hipError_t hipGetLastError() { const int e = sim().pending; sim().pending = 0; return e; }
inline hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::recursive_mutex> g(sim().m);
  size_t& u = sim().used[sim_device()];
  if (u + n > sim().total) return sim().pending = hipErrorOutOfMemory;
  u += n;
  *p = std::malloc(1);
  sim().at[*p] = {sim_device(), n};
  return hipSuccess;
}
inline hipError_t hipFree(void* p) {
  std::lock_guard<std::recursive_mutex> g(sim().m);
  auto it = sim().at.find(p);
  if (it == sim().at.end()) std::abort();  // freed twice, or never allocated
  sim().used[it->second.first] -= it->second.second;
  sim().at.erase(it);
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  std::lock_guard<std::recursive_mutex> g(sim().m);
  *t = sim().total;
  *f = sim().total - sim().used[sim_device()];
  return hipSuccess;
}
inline hipError_t hipDeviceSynchronize() { ++sim().syncs; sim().queued.clear(); return hipSuccess; }
inline void sim_use(void* st, void* p) {
  for (auto& q : sim().queued)
    if (q.second == p && q.first != st) sim().late.push_back(p);
  sim().queued.push_back({st, p});
}
enum { hipMemcpyHostToDevice = 1 };
inline hipError_t hipMemcpyAsync(void* d, const void*, size_t, int, hipStream_t st) { sim_use(st, d); return hipSuccess; }
inline hipError_t hipMemcpy(void* d, const void*, size_t, int) { sim_use(nullptr, d); return hipSuccess; }
"""

HEAD = r"""
#include <cstdio>
#include <stdexcept>
#include <thread>
#include <vector>
#include "pool.hpp"
using namespace edl;
#define WANT(c) do { if (!(c)) { std::printf("failed: %s\n", #c); return 1; } } while (0)
constexpr size_t K = 1024, M = 1024 * 1024;
"""

CASES = {
    # an allocation outside the pool takes the cached buffers of its own and of another context
    "direct": r"""
  DevPool a, b;
  for (DevPool* p : {&a, &b}) { void* x = p->take(900 * K); p->give(x); }
  WANT(a.cached() >= 900 * K && device_cached_bytes() == a.cached() + b.cached());
  void* t = nullptr;
  WANT(device_malloc(&t, 15 * M) == hipSuccess && t);
  WANT(a.cached() == 0 && b.cached() == 0 && hipGetLastError() == hipSuccess);
  hipFree(t);
""",
    # ... and so does a buffer made outside a call; live buffers stay
    "live": r"""
  DevPool a;
  void* keep = a.take(4 * M);
  void* x = a.take(600 * K);
  a.give(x);
  void* t = dev_try_alloc(11 * M + 512 * K);
  WANT(t && a.cached() == 0 && sim().at.count(keep));
  WANT(dev_try_alloc(M) == nullptr && hipGetLastError() == hipSuccess);
  dev_free(t);
  a.give(keep);
""",
    # a buffer that fits without its size step
    "exact": r"""
  DevPool a;
  void* y = a.take(512 * K);
  void* x = a.take(15 * M + 1);
  WANT(x && y);
  a.give(x);
  WANT(a.cached() == 0 && sim().used[0] == 512 * K);  // above the bound: freed
  a.give(y);
""",
    # a sixteenth of the device at most
    "bound": r"""
  DevPool a;
  std::vector<void*> v;
  for (int k = 0; k < 20; ++k) v.push_back(a.take(100 * K));
  for (void* p : v) a.give(p);
  WANT(a.cached() <= M && a.cached() > 800 * K && sim().used[0] == a.cached());
  a.release();
  WANT(sim().used[0] == 0);
""",
    # the other device's cache is left alone, a failed request reports the failure
    "device": r"""
  DevPool a, b;
  sim_device() = 1;
  void* y = b.take(900 * K);
  b.give(y);
  sim_device() = 0;
  void* x = a.take(64 * K);
  a.give(x);
  void* t = nullptr;
  WANT(device_malloc(&t, 17 * M) == hipErrorOutOfMemory && !t);
  WANT(hipGetLastError() == hipSuccess);
  WANT(device_malloc(&t, 17 * M) == hipErrorOutOfMemory && hipGetLastError() == hipSuccess);
  WANT(a.cached() == 0 && b.cached() >= 900 * K);
""",
    # a buffer put back with launches queued and filled again: on the same stream
    "upload": r"""
  DevPool a;
  PoolScope s(a);
  int main_stream = 0;
  const char host[64] = {};
  void* x = dev_try_alloc(64);
  sim_use(&main_stream, x);
  dev_free(x);
  void* y = nullptr;
  WANT(dev_upload(&y, host, 64, &main_stream) == hipSuccess && y == x && sim().late.empty());
  dev_free(y);
  WANT(sim().syncs == 0);
""",
    # a call that ends with an exception and launches queued on a second stream
    "unwind": r"""
  DevPool a;
  int main_stream = 0, second = 0;
  void* used = nullptr;
  try {
    PoolScope s(a);
    struct Buf { void* p = dev_try_alloc(64); ~Buf() { dev_free(p); } } b;
    used = b.p;
    sim_use(&second, b.p);
    throw std::runtime_error("launch failed");
  } catch (const std::exception&) {
  }
  WANT(current_pool() == nullptr && sim().syncs == 1);
  {
    PoolScope s(a);
    void* x = dev_try_alloc(64);
    WANT(x == used);
    sim_use(&main_stream, x);
    dev_free(x);
  }
  WANT(sim().late.empty() && sim().syncs == 1);  // a call that ends well does not wait
""",
    # two contexts on threads of their own, both short of memory
    "threads": r"""
  DevPool a, b;
  int bad = 0;
  auto work = [&](DevPool* p, int* n) {
    PoolScope s(*p);
    for (int k = 0; k < 20000; ++k) {
      void* x = dev_try_alloc((k % 7 + 1) * 100 * K);
      void* t = nullptr;
      if (!x) ++*n;
      if (device_malloc(&t, 14 * M) == hipSuccess) hipFree(t); else (void)hipGetLastError();
      dev_free(x);
    }
  };
  int na = 0, nb = 0;
  std::thread ta(work, &a, &na), tb(work, &b, &nb);
  ta.join();
  tb.join();
  WANT(bad == 0 && sim().used[0] == a.cached() + b.cached());
""",
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_pool(case, tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    src = tmp_path / "main.cpp"
    src.write_text(HEAD + "int main() {" + CASES[case] + "  return 0;\n}\n")
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(tmp_path), "-I", CSRC, "-o", exe, str(src),
                    os.path.join(CSRC, "pool.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def test_buffers_filled_on_the_stream():
    """No kept buffer of the batched chains is filled outside the context's stream."""
    with open(os.path.join(CSRC, "batched2.hip")) as f:
        assert "hipMemcpy(" not in f.read()


def test_every_allocation_can_take_the_cache_back():
    """No device allocation of the library goes past device_malloc."""
    for path in glob.glob(os.path.join(CSRC, "*")):
        if os.path.basename(path) in ("pool.cpp", "pool.hpp"):
            continue
        with open(path) as f:
            assert "hipMalloc(" not in f.read(), path
