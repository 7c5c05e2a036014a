// Kept device blocks against a device of 64 GiB that exists on the host only.
#include <cstdio>
#include <vector>

#include "../../graph500-bfs_amd/csrc/devmem.hip"

namespace {

constexpr size_t kMiB = size_t(1) << 20, kGiB = size_t(1) << 30, kAll = 64 * kGiB;

#define CHECK(x)                                                  \
  do {                                                            \
    if (!(x)) {                                                   \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);         \
      std::exit(1);                                               \
    }                                                             \
  } while (0)

struct Got {
  void* p;
  size_t bytes;
  int device;
};
Got take(size_t bytes, bool scratch = false) {
  bool used;
  Got g{};
  g.p = g500::device_alloc(bytes, scratch, &used, &g.bytes, &g.device);
  return g;
}
void give(const Got& g) { g500::device_release(g.p, g.bytes, g.device); }

void fresh_device() {
  g500::device_trim();
  CHECK(fake_device.used == 0 && fake_device.blocks.empty());
  fake_device = FakeDevice{};
  fake_device.capacity = kAll;
}

}  // namespace

namespace g500 {
[[noreturn]] void fail(int, const char*, ...) { std::abort(); }
}  // namespace g500

int main() {
  fresh_device();
  {  // a freed block serves the next allocation of its size
    const Got a = take(100 * kMiB);
    give(a);
    const Got b = take(100 * kMiB);
    CHECK(b.p == a.p && fake_device.mallocs == 1);
    give(b);
  }
  fresh_device();
  {  // no more than an eighth of the device is kept, the newest of it
    std::vector<Got> all;
    for (int i = 0; i < 10; ++i) all.push_back(take(2 * kGiB));
    for (const Got& g : all) give(g);
    CHECK(fake_device.used <= kAll / 8 && fake_device.used == 4 * 2 * kGiB);
    CHECK(fake_device.blocks.count(all[9].p) && !fake_device.blocks.count(all[5].p));
    const Got big = take(9 * kGiB);  // by itself past the limit
    give(big);
    CHECK(fake_device.used <= kAll / 8 && !fake_device.blocks.count(big.p));
  }
  // an allocation that fails takes the kept blocks first, a small one too
  for (size_t want : {size_t(4096), 512 * kMiB}) {
    fresh_device();
    const Got full = take(kAll - 2 * kGiB), kept = take(1 * kGiB), rest = take(1 * kGiB);
    give(kept);
    CHECK(fake_device.used == kAll);  // kept
    const Got a = take(want);
    CHECK(a.p && fake_device.used < kAll);
    const Got none = take(kAll);
    CHECK(!none.p);
    for (const Got& g : {a, full, rest}) give(g);
  }
  fresh_device();
  {  // released beside a capture that forbids the wait: not kept
    const Got a = take(100 * kMiB);
    fake_device.sync_fails = true;
    give(a);
    CHECK(fake_device.used == 0);
  }
  std::puts("devmem ok");
}
