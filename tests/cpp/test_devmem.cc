// Kept device blocks and the validator's edge orders against a device of 64 GiB
// that exists on the host only.
#include <cstdio>
#include <vector>

#include "../../graph500-bfs_amd/csrc/devmem.hip"
#include "../../graph500-bfs_amd/csrc/edgeorder.hip"

// host memory that runs out on demand
static bool no_host_memory = false;
void* operator new(size_t n) {
  void* p = no_host_memory ? nullptr : std::malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace {

constexpr size_t kMiB = size_t(1) << 20, kGiB = size_t(1) << 30, kAll = 64 * kGiB;

int making = 0;  // order_edges: how often it was called, and the error it meets
int error = 0;

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

g500_graph::~g500_graph() { g500::forget_ordered_edges(this); }

namespace g500 {
[[noreturn]] void fail(int code, const char*, ...) { throw Error(code, "fake"); }
std::shared_ptr<const OrderedEdges> order_edges(const g500_graph* g, hipStream_t) {
  ++making;
  if (error) fail(error, "");
  auto o = std::make_shared<OrderedEdges>();
  o->keys.alloc_raw((size_t)g->nedges);
  return o;
}
}  // namespace g500

int main() {
  fresh_device();
  {  // a freed block serves the next allocation of its size
    const Got a = take(100 * kMiB);
    give(a);
    const Got b = take(100 * kMiB);
    CHECK(b.p == a.p);
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
    const Got full = take(kAll - 3 * kGiB), kept = take(1 * kGiB);
    give(kept);
    const Got rest = take(2 * kGiB);
    CHECK(fake_device.used == kAll);
    const Got a = take(want);
    CHECK(a.p && fake_device.used < kAll);
    const Got none = take(kAll);
    CHECK(!none.p);
    for (const Got& g : {a, full, rest}) give(g);
  }
  // then the edge orders that no validation uses
  for (size_t want : {size_t(4096), 512 * kMiB}) {
    fresh_device();
    making = 0;
    g500_graph g, other;
    g.nedges = other.nedges = kGiB / 8;
    other.device = 1;
    for (g500_graph* x : {&g, &other}) {
      CHECK(!g500::order_for_pass(x, nullptr) && !g500::held_order(x));  // a graph's first pass
      CHECK(g500::order_for_pass(x, nullptr) && g500::held_order(x));
    }
    CHECK(making == 2 && fake_device.used == 2 * kGiB);
    const Got full = take(kAll - fake_device.used);
    auto in_use = g500::held_order(&g);
    CHECK(!take(want).p && g500::held_order(&g) == in_use);
    in_use.reset();
    const Got a = take(want);
    CHECK(a.p && !g500::held_order(&g) && g500::held_order(&other));
    CHECK(!g500::order_for_pass(&g, nullptr) && making == 2);  // not made again
    give(a);
    give(full);
  }
  // no room for an order: passes go without, and later ones do not try again
  fresh_device();
  {
    g500_graph g;
    g.nedges = (int64_t)kAll / 8;
    const Got full = take(1 * kGiB);
    making = 0;
    for (int i = 0; i < 3; ++i) CHECK(!g500::order_for_pass(&g, nullptr));
    CHECK(making == 1);
    give(full);
    g500_graph broken;  // other errors are not swallowed
    error = G500_ERR_HIP;
    CHECK(!g500::order_for_pass(&broken, nullptr));
    bool thrown = false;
    try {
      (void)g500::order_for_pass(&broken, nullptr);
    } catch (const g500::Error& e) {
      thrown = e.code == G500_ERR_HIP;
    }
    CHECK(thrown);
    error = 0;
  }
  {  // a graph that goes takes its order along and is not asked for it later
    fresh_device();
    {
      g500_graph g;
      g.nedges = kGiB / 8;
      (void)g500::order_for_pass(&g, nullptr);
      CHECK(g500::order_for_pass(&g, nullptr));
    }
    const Got all = take(kAll);
    CHECK(all.p);
    give(all);
  }
  fresh_device();
  {  // blocks go back once they are ten seconds old, however the library is called
    const auto later = std::chrono::steady_clock::now() + std::chrono::seconds(11);
    const Got a = take(100 * kMiB), b = take(200 * kMiB);
    give(a);
    give(b);
    g500::device_release_idle();
    CHECK(fake_device.used == 300 * kMiB);
    g500::device_release_idle(later);
    CHECK(fake_device.used == 0);
    const Got c = take(300 * kMiB);
    give(c);
    g500::device_release_idle();  // younger
    CHECK(fake_device.used == 300 * kMiB);
  }
  fresh_device();
  {  // a kept block is handed out only after the device was waited for, once for all
     // that were released before, else it goes back
    const Got a = take(100 * kMiB), b = take(200 * kMiB), c = take(300 * kMiB);
    give(a);
    give(b);
    const int waits = fake_device.waits;
    CHECK(take(100 * kMiB).p == a.p && fake_device.waits == waits + 1);
    CHECK(take(200 * kMiB).p == b.p && fake_device.waits == waits + 1);
    give(c);
    give(a);
    CHECK(take(300 * kMiB).p == c.p && fake_device.waits == waits + 2);
    CHECK(take(100 * kMiB).p == a.p && fake_device.waits == waits + 2);
    give(a);
    CHECK(take(100 * kMiB).p == a.p && fake_device.waits == waits + 3);
    {  // idle ones need none, until the releasing thread takes it back
      g500::IdleReleases released;
      give(a);
      CHECK(take(100 * kMiB).p == a.p && fake_device.waits == waits + 4);
      released.now();
      give(a);
      CHECK(take(100 * kMiB).p == a.p && fake_device.waits == waits + 4);
      {
        g500::IdleReleases inner;
        give(a);
        CHECK(take(100 * kMiB).p == a.p && fake_device.waits == waits + 5);
        inner.now();
      }
      give(a);
      CHECK(take(100 * kMiB).p == a.p && fake_device.waits == waits + 5);
      released.over();
      give(a);
      CHECK(take(100 * kMiB).p == a.p && fake_device.waits == waits + 6);
      released.now();
    }
    give(a);
    CHECK(take(100 * kMiB).p == a.p && fake_device.waits == waits + 7);
    give(a);
    const Got full = take(kAll - fake_device.used);
    CHECK(fake_device.used == kAll);
    const Got d = take(100 * kMiB);  // no room for the wait's own bytes: hipFree waits
    CHECK(d.p && fake_device.waits > waits + 7 && fake_device.used == kAll);
    for (const Got& g : {b, c, d, full}) give(g);
  }
  fresh_device();
  {  // every device has its own
    const Got a = take(100 * kMiB);
    fake_device.current = 1;
    const Got b = take(100 * kMiB);
    give(b);
    fake_device.current = 0;
    give(a);
    const int waits = fake_device.waits;
    CHECK(take(100 * kMiB).p == a.p && fake_device.waits == waits + 1);
    fake_device.current = 1;
    CHECK(take(100 * kMiB).p == b.p && fake_device.waits == waits + 2);
    fake_device.current = 0;
    give(a);  // b is device 1's: released from device 0 it goes back at once
    give(b);
    CHECK(fake_device.used == 100 * kMiB);
  }
  fresh_device();
  {  // without host memory a released block goes back, and nothing is thrown
    std::vector<Got> all;
    for (int i = 0; i < 100; ++i) all.push_back(take(2 * kMiB));
    no_host_memory = true;
    for (const Got& g : all) give(g);
    g500::device_release_idle(std::chrono::steady_clock::now() + std::chrono::seconds(11));
    no_host_memory = false;
    CHECK(fake_device.used < 200 * kMiB);
    g500::device_trim();
    CHECK(fake_device.used == 0);
  }
  std::puts("devmem ok");
}
