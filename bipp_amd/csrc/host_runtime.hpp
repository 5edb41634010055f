// Host runtime of libbipp_amd: error conversion for the C-ABI, growable device and pinned
// buffers, and the context (one HIP stream on the current device).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <numeric>
#include <string>
#include <vector>

#include "bipp_hip.h"
#include "common.hpp"

namespace bippamd {

// message of the last failing C-ABI call on this thread (one instance across the library)
inline thread_local std::string g_last_error;

// Runs f and converts exceptions into BippError codes and the thread-local message.
template <typename F>
BippError guard(F&& f) {
  try {
    f();
    g_last_error.clear();
    return BIPP_SUCCESS;
  } catch (const BippException& e) {
    // a failed runtime call leaves its code as HIP's last error: clear it, so that the next
    // launch check does not report it again
    (void)hipGetLastError();
    g_last_error = e.what();
    return e.code;
  } catch (const std::bad_alloc&) {
    (void)hipGetLastError();
    g_last_error = "host allocation failed";
    return BIPP_GENERIC_ERROR;
  } catch (const std::exception& e) {
    g_last_error = e.what();
    return BIPP_GENERIC_ERROR;
  } catch (...) {
    g_last_error = "unknown error";
    return BIPP_GENERIC_ERROR;
  }
}

inline void require(bool cond, BippError code, const char* msg) {
  if (!cond) fail(code, msg);
}
inline void require(bool cond, BippError code, const std::string& msg) {
  if (!cond) fail(code, msg);
}

// Memory blocks given back by short-lived buffers of a context (the imager of one
// image_synthesis call, the arrays of one host eigensolve), for the next ones: allocating,
// pinning and freeing them took 5.5 ms of a 15 ms call.  At most DEV_BOUND bytes of device and
// PIN_BOUND of pinned host memory are held per context; above that the blocks longest unused go
// back to the runtime (a pool that kept its first blocks instead was full of one call's sizes,
// and the next kind of call allocated everything anew: 2.2 ms became 9 to 17 ms).  Everything goes
// back when the context goes, and the blocks of every pool when an allocation of the library fails,
// in a pool's scope or not, before it is tried again.  Device blocks are handed on in stream
// order: all users of a context's pool work on its one stream.  Pinned blocks are given back
// only after the stream has been waited for.
struct BufferPool {
  static constexpr size_t DEV_BOUND = size_t(2) << 30, PIN_BOUND = size_t(256) << 20;
  enum Kind { DEV = 0, PIN = 1 };

  BufferPool() {
    std::lock_guard<std::mutex> lock(all().mu);
    all().pools.push_back(this);
  }
  BufferPool(const BufferPool&) = delete;
  ~BufferPool() {
    {
      std::lock_guard<std::mutex> lock(all().mu);
      all().pools.erase(std::find(all().pools.begin(), all().pools.end(), this));
    }
    trim();
  }
  // the held blocks of every pool back to the runtime
  static void trim_all() {
    std::lock_guard<std::mutex> lock(all().mu);
    for (BufferPool* p : all().pools) p->trim();
  }
  // a held block of at least `bytes` (and not much more), or nullptr
  void* take(Kind k, size_t bytes, size_t& cap) {
    std::lock_guard<std::mutex> lock(mu_);
    const auto it = free_[k].lower_bound(bytes);
    if (it == free_[k].end() || it->first > bytes + bytes / 2 + (64 << 10)) return nullptr;
    void* p = it->second.p;
    cap = it->first;
    held_[k] -= cap;
    free_[k].erase(it);
    return p;
  }
  void put(Kind k, void* p, size_t cap) noexcept {
    const size_t bound = k == DEV ? DEV_BOUND : PIN_BOUND;
    try {
      std::lock_guard<std::mutex> lock(mu_);
      if (cap <= bound) {
        free_[k].emplace(cap, Block{p, ++clock_});
        held_[k] += cap;
        p = nullptr;
      }
      while (held_[k] > bound) {
        auto old = free_[k].begin();
        for (auto it = old; it != free_[k].end(); ++it)
          if (it->second.since < old->second.since) old = it;
        release(k, old->second.p);
        held_[k] -= old->first;
        free_[k].erase(old);
      }
    } catch (...) {  // no memory for the entry: the block goes back to the runtime
    }
    if (p) release(k, p);
  }
  void trim() {
    std::lock_guard<std::mutex> lock(mu_);
    for (Kind k : {DEV, PIN}) {
      for (auto& e : free_[k]) release(k, e.second.p);
      free_[k].clear();
      held_[k] = 0;
    }
  }
  static void release(Kind k, void* p) {
    if (k == DEV)
      (void)hipFree(p);
    else
      (void)hipHostFree(p);
  }

 private:
  struct Block {
    void* p;
    unsigned long long since;  // of clock_
  };
  struct Registry {
    std::mutex mu;
    std::vector<BufferPool*> pools;
  };
  static Registry& all() {
    static Registry* r = new Registry;  // outlives every pool
    return *r;
  }
  std::mutex mu_;
  std::multimap<size_t, Block> free_[2];
  unsigned long long clock_ = 0;
  size_t held_[2] = {0, 0};
};

// Buffers allocated on this thread while a scope is alive take their blocks from its pool.
struct PoolScope {
  explicit PoolScope(BufferPool& p) : prev(current()) { current() = &p; }
  PoolScope(const PoolScope&) = delete;
  ~PoolScope() { current() = prev; }
  static BufferPool*& current() {
    static thread_local BufferPool* c = nullptr;
    return c;
  }

 private:
  BufferPool* prev;
};

// Growable allocation (device or pinned host memory).  A block goes back to the pool that it
// was allocated under (which outlives the buffer), else to the runtime: hipFree synchronises
// the device, so work still in flight on it has finished first.
template <BufferPool::Kind K>
struct PooledBuf {
  void* p = nullptr;
  size_t cap = 0;
  PooledBuf() = default;
  PooledBuf(const PooledBuf&) = delete;
  PooledBuf& operator=(const PooledBuf&) = delete;
  ~PooledBuf() { drop(); }
  void drop() {
    if (p && pool)
      pool->put(K, p, cap);
    else if (p)
      BufferPool::release(K, p);
    p = nullptr;
    cap = 0;
  }
  void* get(size_t bytes) {
    bytes = std::max<size_t>(bytes, 256);
    if (bytes > cap) {
      drop();
      pool = PoolScope::current();
      if (pool) p = pool->take(K, bytes, cap);
      if (!p) {
        hipError_t e = allocate(bytes);
        if (e != hipSuccess) {
          (void)hipGetLastError();
          BufferPool::trim_all();
          e = allocate(bytes);
        }
        if (e != hipSuccess) p = nullptr;
        hip_check(e, K == BufferPool::DEV ? "hipMalloc" : "hipHostMalloc");
        cap = bytes;
      }
    }
    return p;
  }
  template <typename T>
  T* as(size_t n) {
    return static_cast<T*>(get(n * sizeof(T)));
  }
  void swap(PooledBuf& o) {
    std::swap(p, o.p);
    std::swap(cap, o.cap);
    std::swap(pool, o.pool);
  }

 private:
  BufferPool* pool = nullptr;
  hipError_t allocate(size_t bytes) {
    return K == BufferPool::DEV ? hipMalloc(&p, bytes) : hipHostMalloc(&p, bytes, hipHostMallocDefault);
  }
};
using DevBuf = PooledBuf<BufferPool::DEV>;
using PinnedBuf = PooledBuf<BufferPool::PIN>;

// ---------------------------------------------------------------------------------------
// Context
// ---------------------------------------------------------------------------------------
struct ContextImpl {
  BippProcessingUnit pu = BIPP_PU_GPU;
  int device = 0;
  int n_cu = 1;
  hipStream_t stream = nullptr;
  BufferPool pool;

  explicit ContextImpl(BippProcessingUnit p) {
    require(p != BIPP_PU_CPU, BIPP_INVALID_PARAMETER_ERROR,
            "this library computes on the GPU only (processing unit CPU requested)");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0)
      fail(BIPP_GPU_SUPPORT_ERROR, "no GPU device available");
    BIPP_HIP(hipGetDevice(&device));
    hipDeviceProp_t prop;
    BIPP_HIP(hipGetDeviceProperties(&prop, device));
    n_cu = prop.multiProcessorCount;
    BIPP_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    BIPP_HIP(hipEventCreateWithFlags(&ready, hipEventDisableTiming));
    pu = BIPP_PU_GPU;
  }
  ~ContextImpl() {
    if (ready) (void)hipEventDestroy(ready);
    if (stream) (void)hipStreamDestroy(stream);
  }
  // Waits for the stream by polling an event: a blocking wait that spans a long kernel wakes
  // up about a millisecond late, which leaves the device idle between batches.
  void sync() {
    BIPP_HIP(hipEventRecord(ready, stream));
    for (;;) {
      const hipError_t q = hipEventQuery(ready);
      if (q == hipSuccess) break;
      if (q != hipErrorNotReady) BIPP_HIP(q);
    }
  }

 private:
  hipEvent_t ready = nullptr;
};

}  // namespace bippamd
