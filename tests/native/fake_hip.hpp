// A HIP runtime on host memory, for checks of the engines' host code without
// a device: the program's own definitions take the place of the library's.
// Allocations can be made to fail, freed ranges are known, and the current
// device and every stream's are tracked.  Kernel wrappers are the check's own.
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>

namespace fake {

struct Device {
  std::map<char*, size_t> live;  // device allocations
  std::map<char*, int> home;     // and their devices
  size_t used = 0, limit = ~static_cast<size_t>(0);
  int current = 0, launches = 0;
  long room = -1;  // allocations that still succeed (-1: all)
};
inline Device& dev() {
  static Device d;
  return d;
}

// Is [p, p + bytes) inside one live allocation?
inline bool holds(const void* p, size_t bytes) {
  char* at = static_cast<char*>(const_cast<void*>(p));
  auto it = dev().live.upper_bound(at);
  if (it == dev().live.begin()) return false;
  --it;
  return at + bytes <= it->first + it->second;
}

inline void require(bool ok, const char* what) {
  if (ok) return;
  std::printf("failed: %s\n", what);
  std::fflush(stdout);
  std::_Exit(1);
}

struct Stream {
  int device;
};

// Is all memory on this device?
inline bool all_on(int device) {
  for (const auto& h : dev().home)
    if (h.second != device) return false;
  return true;
}

}  // namespace fake

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
  fake::Device& d = fake::dev();
  *p = nullptr;
  if (d.used + bytes > d.limit || d.room == 0) return hipErrorOutOfMemory;
  if (d.room > 0) --d.room;
  *p = std::calloc(1, bytes);
  d.live[static_cast<char*>(*p)] = bytes;
  d.home[static_cast<char*>(*p)] = d.current;
  d.used += bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  fake::Device& d = fake::dev();
  auto it = d.live.find(static_cast<char*>(p));
  fake::require(it != d.live.end(), "hipFree of what is not allocated");
  std::memset(p, 0xdd, std::min<size_t>(it->second, 1 << 20));
  d.used -= it->second;
  d.home.erase(it->first);
  d.live.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  *p = std::calloc(1, bytes);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  fake::dev().current = d;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = fake::dev().current;
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* free_bytes, size_t* total) {
  *total = static_cast<size_t>(288) << 30;
  *free_bytes = std::min(*total, fake::dev().limit) - fake::dev().used;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 100000;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(new fake::Stream{fake::dev().current});
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  delete reinterpret_cast<fake::Stream*>(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0;
  return hipSuccess;
}
hipError_t hipGraphCreate(hipGraph_t* g, unsigned) {
  *g = reinterpret_cast<hipGraph_t>(new int);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  *e = reinterpret_cast<hipGraphExec_t>(g);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) {
  delete reinterpret_cast<int*>(g);
  return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  std::memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipMemcpy(void* to, const void* from, size_t bytes, hipMemcpyKind) {
  std::memcpy(to, from, bytes);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* to, const void* from, size_t bytes, hipMemcpyKind, hipStream_t) {
  std::memcpy(to, from, bytes);
  return hipSuccess;
}
}

namespace fake {
// What every kernel wrapper of a check begins with: a launch on a stream of
// another device than the current one is refused by the runtime.
inline hipError_t launch(hipStream_t s) {
  ++dev().launches;
  return reinterpret_cast<Stream*>(s)->device == dev().current ? hipSuccess : hipErrorInvalidResourceHandle;
}
}  // namespace fake
