// devmem.hip -- device memory that is kept for the next allocation.
//
// hipMalloc and hipFree of large blocks are quick only until the driver has to
// clear what was freed before: from then on an allocation costs ~30 ms per GB.
// A graph built, searched and freed over and over (13 GB of blocks at SCALE 24)
// took 170 to 470 ms each time that way, its kernels 40.  So blocks from 1 MiB
// on are kept when they are released and handed out again, up to an eighth of
// the device's memory; the oldest are given back first.  All of them go when an
// allocation fails (and then the validator's edge orders) or free memory is
// asked for (g500_device_memory), and those that no one took for ten seconds at
// the next call that allocates, frees, searches or validates.  A process that
// makes no more calls keeps them.
//
// A kept block is handed out only after the device has finished all work queued
// before it was released (hipFree would wait for that at once), so whichever
// thread or stream takes it next has it alone.  One wait does for all blocks
// released before it, and none is needed for blocks whose only users have just
// been waited for (IdleReleases).  With a wait at each release a build at SCALE 18
// took 3 % longer (1.56 ms against 1.51 on one card); this way as long as with none
// of them (1.57 against 1.56 on another).
#include <atomic>
#include <chrono>
#include <mutex>
#include <vector>

#include "common.hpp"

namespace g500 {

namespace {

constexpr size_t kKeepMin = size_t(1) << 20;
constexpr size_t kGranule = size_t(2) << 20;
constexpr std::chrono::seconds kIdle(10);

using Clock = std::chrono::steady_clock;

struct Block {
  void* p;
  size_t bytes;
  int device;
  uint64_t number;  // of its release, 0 where it was idle then
  Clock::time_point since;
};

// never destroyed: handles may be released by destructors that run after
// those of this file
struct Kept {
  std::mutex mu;
  std::vector<Block> blocks;  // oldest first
  uint64_t releases = 0;
  std::vector<uint64_t> waited;  // per device: releases that a wait has followed
  // when the oldest was released, the far future where there is none: read
  // without the lock by calls that only look for idle blocks
  std::atomic<Clock::rep> oldest{Clock::time_point::max().time_since_epoch().count()};

  uint64_t& waited_for(int device) {
    if ((int)waited.size() <= device) waited.resize((size_t)device + 1, 0);
    return waited[(size_t)device];
  }
  void changed() {
    const Clock::time_point t = blocks.empty() ? Clock::time_point::max() : blocks.front().since;
    oldest.store(t.time_since_epoch().count(), std::memory_order_relaxed);
  }
};
Kept& kept() {
  static Kept* k = new Kept;
  return *k;
}

size_t keep_limit(int device) {
  static std::mutex mu;
  static std::vector<size_t> limit;
  std::lock_guard<std::mutex> lock(mu);
  if ((int)limit.size() <= device) limit.resize((size_t)device + 1, 0);
  if (limit[(size_t)device] == 0) {
    size_t total = 0;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) total = prop.totalGlobalMem;
    limit[(size_t)device] = total / 8 + 1;
  }
  return limit[(size_t)device];
}

// Calls made in its scope leave the captures of other threads alone.
struct BesideCaptures {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  const bool set = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
  ~BesideCaptures() {
    if (set) (void)hipThreadExchangeStreamCaptureMode(&mode);
  }
};

thread_local bool t_idle = false;

void free_blocks(const std::vector<Block>& out) {
  if (out.empty()) return;
  BesideCaptures scope;
  for (const Block& b : out) (void)hipFree(b.p);
}

// Waits for all work queued on the device.  hipDeviceSynchronize does that too,
// but beside a capture in any thread, an engine's of its batch for one, it fails
// and ends that capture, whatever its mode; hipFree waits as well and does not.
// 10 us after the last work, then 1.  Of the current device.
bool device_wait() {
  BesideCaptures scope;
  void* p = nullptr;
  if (hipMalloc(&p, 4096) == hipSuccess && hipFree(p) == hipSuccess) return true;
  (void)hipGetLastError();
  return false;
}

}  // namespace

void* device_alloc(size_t bytes, bool scratch, bool* used, size_t* got, int* device) {
  *used = false;
  *got = bytes;
  *device = 0;
  (void)hipGetDevice(device);
  void* p = nullptr;
  const auto fresh = [&](size_t size) {
    *got = size;
    if (hipMalloc(&p, size) == hipSuccess) return true;
    (void)hipGetLastError();
    p = nullptr;
    return false;
  };
  const auto fresh_after_all = [&](size_t size) {
    device_trim();
    if (fresh(size)) return true;
    drop_ordered_edges(*device);
    device_trim();
    return fresh(size);
  };
  if (bytes < kKeepMin) {
    device_release_idle();
    if (!fresh(bytes)) (void)fresh_after_all(bytes);
    return p;
  }
  size_t want = (bytes + kGranule - 1) / kGranule * kGranule;
  if (scratch) {
    // sizes that differ a little (another seed's graph) share a block
    const size_t step = std::max(kGranule, (size_t(1) << (63 - __builtin_clzll(want))) / 16);
    want = (want + step - 1) / step * step;
  }
  const size_t most = want + (scratch ? want / 8 : want / 64);
  Kept& k = kept();
  bool idle = true;  // nothing queued before its release is left
  uint64_t releases = 0;
  {
    std::lock_guard<std::mutex> lock(k.mu);
    size_t best = k.blocks.size();
    for (size_t i = 0; i < k.blocks.size(); ++i) {
      const Block& b = k.blocks[i];
      if (b.device == *device && b.bytes >= want && b.bytes <= most &&
          (best == k.blocks.size() || b.bytes < k.blocks[best].bytes))
        best = i;
    }
    if (best < k.blocks.size()) {
      p = k.blocks[best].p;
      *got = k.blocks[best].bytes;
      *used = true;
      idle = k.blocks[best].number <= k.waited_for(*device);
      releases = k.releases;
      k.blocks.erase(k.blocks.begin() + (ptrdiff_t)best);
    }
    k.changed();
  }
  if (!idle) {
    if (device_wait()) {
      std::lock_guard<std::mutex> lock(k.mu);
      uint64_t& waited = k.waited_for(*device);
      waited = std::max(waited, releases);
    } else {  // no memory left, or a fault: hipFree waits
      (void)hipFree(p);
      p = nullptr;
      *used = false;
    }
  }
  device_release_idle();
  if (p) return p;
  if (!fresh(want) && !fresh_after_all(want)) (void)fresh(bytes);
  return p;
}

bool IdleReleases::set(bool idle) { return std::exchange(t_idle, idle); }

// Buffers are released by destructors: a lack of host memory must not leave here.
void device_release(void* p, size_t bytes, int device) {
  int current = 0;
  (void)hipGetDevice(&current);
  std::vector<Block> old;
  bool keep = bytes >= kKeepMin && current == device;
  if (keep) {
    try {
      const size_t limit = keep_limit(device);
      Kept& k = kept();
      std::lock_guard<std::mutex> lock(k.mu);
      keep = false;
      if (bytes <= limit) {
        old.reserve(k.blocks.size() + 1);
        k.blocks.push_back({p, bytes, device, t_idle ? 0 : ++k.releases, Clock::now()});
        keep = true;
        size_t total = 0;
        for (const Block& b : k.blocks) total += b.device == device ? b.bytes : 0;
        for (size_t i = 0; i < k.blocks.size() && total > limit;) {
          if (k.blocks[i].device != device) {
            ++i;
            continue;
          }
          total -= k.blocks[i].bytes;
          old.push_back(k.blocks[i]);
          k.blocks.erase(k.blocks.begin() + (ptrdiff_t)i);
        }
        k.changed();
      }
    } catch (const std::bad_alloc&) {
      keep = false;
    }
  }
  if (!keep) (void)hipFree(p);
  free_blocks(old);
  device_release_idle();
}

void device_trim() {
  std::vector<Block> old;
  {
    Kept& k = kept();
    std::lock_guard<std::mutex> lock(k.mu);
    old.swap(k.blocks);
    k.changed();
  }
  free_blocks(old);
}

void device_release_idle(Clock::time_point now) {
  Kept& k = kept();
  const auto limit = (now - kIdle).time_since_epoch().count();
  if (k.oldest.load(std::memory_order_relaxed) >= limit) return;
  std::vector<Block> old;
  {
    std::lock_guard<std::mutex> lock(k.mu);
    try {
      old.reserve(k.blocks.size());
    } catch (const std::bad_alloc&) {
      return;  // at another call
    }
    while (!k.blocks.empty() && k.blocks.front().since < now - kIdle) {
      old.push_back(k.blocks.front());
      k.blocks.erase(k.blocks.begin());
    }
    k.changed();
  }
  free_blocks(old);
}

}  // namespace g500
