// A HIP runtime on host memory for the host-side harnesses: allocations are malloc blocks with
// guard bytes behind them, copies happen at once, and allocations can be made to fail (from the
// k-th on, or above a number of bytes in use).  Linked in place of the real runtime.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace stub {

constexpr size_t GUARD = size_t(1) << 20;
constexpr unsigned char FILL = 0xa5;

struct Space {                    // device or pinned host memory
  std::map<void*, size_t> live;
  size_t used = 0, limit = ~size_t(0);
  int fail_after = -1;            // allocations until they fail, < 0: they do not
};
inline Space dev, pin;
inline int stream_waits = 0;

inline hipError_t allocate(Space& s, void** p, size_t n) {
  *p = nullptr;
  if (s.fail_after == 0 || s.used + n > s.limit) return hipErrorOutOfMemory;
  if (s.fail_after > 0) --s.fail_after;
  unsigned char* q = static_cast<unsigned char*>(std::malloc(n + GUARD));
  std::memset(q + n, FILL, GUARD);
  s.live[q] = n;
  s.used += n;
  *p = q;
  return hipSuccess;
}
inline bool intact(const Space& s) {  // nothing written behind a block
  for (const auto& b : s.live)
    for (size_t k = 0; k < GUARD; ++k)
      if (static_cast<const unsigned char*>(b.first)[b.second + k] != FILL) return false;
  return true;
}
inline hipError_t release(Space& s, void* p) {
  const auto it = s.live.find(p);
  if (it == s.live.end()) return p ? hipErrorInvalidValue : hipSuccess;
  s.used -= it->second;
  s.live.erase(it);
  std::free(p);
  return hipSuccess;
}

// message and end of the scenario
inline void expect(bool ok, const char* what, int line) {
  if (ok) return;
  std::fprintf(stderr, "line %d: not so: %s\n", line, what);
  std::exit(1);
}
#define EXPECT(x) stub::expect(static_cast<bool>(x), #x, __LINE__)

}  // namespace stub

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return stub::allocate(stub::dev, p, n); }
hipError_t hipFree(void* p) { return stub::release(stub::dev, p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return stub::allocate(stub::pin, p, n); }
hipError_t hipHostFree(void* p) { return stub::release(stub::pin, p); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  std::memset(static_cast<void*>(p), 0, sizeof(*p));
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = nullptr, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return ++stub::stream_waits, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = nullptr, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = nullptr, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return ++stub::stream_waits, hipSuccess; }
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { return *t = 0, hipSuccess; }
}

// Kernel launches: nothing runs; the dynamic LDS of each launch is held against the limit that
// was set for its kernel before (64 KiB without one).
namespace stub {
struct Launch {
  const void* kernel;
  unsigned threads;
  size_t lds, limit;
};
inline std::map<const void*, size_t> lds_limit;
inline Launch last{};
inline int launches = 0, attribute_failures = 0;  // attribute calls to fail
inline dim3 cfg_grid, cfg_block;
inline size_t cfg_lds = 0;
}  // namespace stub

extern "C" {
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute, int v) {
  if (stub::attribute_failures > 0) return --stub::attribute_failures, hipErrorUnknown;
  return stub::lds_limit[f] = static_cast<size_t>(v), hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t) {
  stub::cfg_grid = g;
  stub::cfg_block = b;
  stub::cfg_lds = lds;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
  *g = stub::cfg_grid;
  *b = stub::cfg_block;
  *lds = stub::cfg_lds;
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3 b, void**, size_t lds, hipStream_t) {
  const auto it = stub::lds_limit.find(f);
  stub::last = {f, b.x, lds, it == stub::lds_limit.end() ? size_t(64) << 10 : it->second};
  ++stub::launches;
  return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
}
