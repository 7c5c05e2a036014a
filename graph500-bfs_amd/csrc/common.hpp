// common.hpp -- error plumbing and wave64 helpers shared by every kernel file.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstdint>
#include <cstdio>
#include <stdexcept>
#include <string>
#include <utility>

#include "../../include/g500bfs.h"

namespace g500 {

// Internal errors travel as exceptions and are turned into status codes plus
// a thread-local message at the C boundary (api.hip).
struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

[[noreturn]] void fail(int code, const char* fmt, ...);

#define G500_CHECK_HIP(expr)                                                  \
  do {                                                                        \
    hipError_t e__ = (expr);                                                  \
    if (e__ != hipSuccess)                                                    \
      ::g500::fail(G500_ERR_HIP, "%s: %s (%s:%d)", #expr,                     \
                   hipGetErrorString(e__), __FILE__, __LINE__);               \
  } while (0)

#define G500_CHECK_LAUNCH() G500_CHECK_HIP(hipGetLastError())

constexpr int kWave = 64;

__host__ __device__ inline int64_t ceil_div(int64_t a, int64_t b) {
  return (a + b - 1) / b;
}

__device__ inline int lane_id() { return (int)__lane_id(); }
// mask of lanes strictly below this one
__device__ inline uint64_t lanemask_lt() {
  const int l = lane_id();
  return l == 0 ? 0ull : (~0ull >> (64 - l));
}

// Device memory (devmem.hip): bytes on the current device, from a block kept
// from an earlier release where one fits (*used: it then holds old data).
// *got and *device go back with device_release.  Null where there is no room.
// scratch: freed again soon, so its size may be rounded up.
void* device_alloc(size_t bytes, bool scratch, bool* used, size_t* got, int* device);
// The block may still be in use by work queued so far, and who gets it next waits
// for the device, unless the releasing thread has said otherwise (IdleReleases).
void device_release(void* p, size_t bytes, int device);
// Until it ends, what the thread releases after now() is idle: every stream that
// used it has been waited for.  Declared before the buffers it is for, whose
// destructors then run inside it; left by an exception it says nothing.
struct IdleReleases {
  void now() { (void)set(true); }
  void over() { (void)set(false); }
  ~IdleReleases() { (void)set(before); }

 private:
  static bool set(bool idle);
  const bool before = set(false);
};
// Gives all kept blocks back to the device.
void device_trim();
// Gives back the kept blocks that no one took for ten seconds; a few
// nanoseconds where there are none.  For the ends of calls that wait for the
// device anyway.
void device_release_idle(
    std::chrono::steady_clock::time_point now = std::chrono::steady_clock::now());
// Releases the edge orders of graphs on the device that no validation is using
// (edgeorder.hip): they only save time, so an allocation that fails takes them.
void drop_ordered_edges(int device);

// A copy behind the work of s, done on return.  Nothing here uses the default
// stream: its every use, in any thread, ends the captures that other threads'
// engines make of their batches, and fails itself.
// (An asynchronous copy and a wait take 22 us for a few bytes, this 13.)
inline void copy_now(void* dst, const void* src, size_t bytes, hipMemcpyKind kind,
                     hipStream_t s) {
  G500_CHECK_HIP(hipMemcpyWithStream(dst, src, bytes, kind, s));
}
template <class T>
void copy_to_host(T* dst, const T* src, int64_t n, hipStream_t s) {
  copy_now(dst, src, (size_t)n * sizeof(T), hipMemcpyDeviceToHost, s);
}

// Device allocation owned by a host object.
template <typename T>
struct DevBuf {
  T* p = nullptr;
  size_t n = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { release(); }
  // a block that held other data is cleared on s, as the driver clears new ones
  void alloc(size_t count, hipStream_t s) {
    bool used;
    reserve(count, false, &used);
    if (used) G500_CHECK_HIP(hipMemsetAsync(p, 0, n * sizeof(T), s));
  }
  // for arrays that are written before they are read
  void alloc_raw(size_t count) {
    bool used;
    reserve(count, false, &used);
  }
  bool try_raw(size_t count) {
    bool used;
    return take(count, false, &used);
  }
  // scratch that is written before it is read; false where the device has no
  // room, for a caller that can do without
  bool try_scratch(size_t count) {
    bool used;
    return take(count, true, &used);
  }
  void release() {
    if (p) device_release(p, bytes_, device_);
    p = nullptr;
    n = 0;
  }
  void swap(DevBuf& o) {
    std::swap(p, o.p);
    std::swap(n, o.n);
    std::swap(bytes_, o.bytes_);
    std::swap(device_, o.device_);
  }
  T* get() const { return p; }

 private:
  size_t bytes_ = 0;
  int device_ = 0;

  bool take(size_t count, bool scratch, bool* used) {
    release();
    if (count == 0) count = 1;
    p = static_cast<T*>(device_alloc(count * sizeof(T), scratch, used, &bytes_, &device_));
    if (!p) {
      (void)hipGetLastError();
      return false;
    }
    n = count;
    return true;
  }
  void reserve(size_t count, bool scratch, bool* used) {
    if (!take(count, scratch, used))
      fail(G500_ERR_NOMEM, "hipMalloc(%zu bytes): out of memory", count * sizeof(T));
  }
};

}  // namespace g500
