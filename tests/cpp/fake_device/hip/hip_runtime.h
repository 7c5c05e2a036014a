// A device for host-only tests of the memory code: `capacity` bytes handed out
// from the heap, no kernels, one device unless a test switches `current`.
#pragma once

#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>

#define __host__
#define __device__

struct FakeDevice {
  size_t capacity = 0, used = 0, most = 0;  // most: the largest `used` so far
  int mallocs = 0, frees = 0, current = 0;
  int waits = 0;  // hipFree waits for the device
  std::map<void*, size_t> blocks;
};
inline FakeDevice fake_device;

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorStreamCaptureUnsupported = 900 };
struct hipDeviceProp_t {
  size_t totalGlobalMem;
};
enum hipStreamCaptureMode { hipStreamCaptureModeGlobal, hipStreamCaptureModeThreadLocal,
                            hipStreamCaptureModeRelaxed };

using hipStream_t = void*;
struct uint2 {
  unsigned x, y;
};

inline unsigned __lane_id() { return 0; }
inline const char* hipGetErrorString(hipError_t) { return "fake"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) {
  *d = fake_device.current;
  return hipSuccess;
}
inline hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  p->totalGlobalMem = fake_device.capacity;
  return hipSuccess;
}
inline hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
inline hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) {
  std::memset(p, v, n < 64 ? n : 64);
  return hipSuccess;
}
inline hipError_t hipMemcpyWithStream(void*, const void*, size_t, hipMemcpyKind, hipStream_t) {
  return hipSuccess;
}
inline hipError_t hipMalloc(void** p, size_t n) {
  FakeDevice& d = fake_device;
  if (d.used + n > d.capacity) return hipErrorOutOfMemory;
  *p = std::malloc(64);
  d.blocks[*p] = n;
  d.used += n;
  d.most = d.used > d.most ? d.used : d.most;
  ++d.mallocs;
  return hipSuccess;
}
inline hipError_t hipFree(void* p) {
  FakeDevice& d = fake_device;
  auto it = d.blocks.find(p);
  if (it == d.blocks.end()) std::abort();
  d.used -= it->second;
  ++d.frees;
  ++d.waits;
  d.blocks.erase(it);
  std::free(p);
  return hipSuccess;
}
