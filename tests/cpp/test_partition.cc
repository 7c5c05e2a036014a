// The split of the row buckets into groups for two partition passes.
#include <cstdio>
#include <cstdlib>

#include "../../graph500-bfs_amd/csrc/internal.hpp"


#define CHECK(x)                                                          \
  do {                                                                    \
    if (!(x)) {                                                           \
      std::printf("%s:%d: %s (%lld)\n", __FILE__, __LINE__, #x, (long long)b); \
      std::exit(1);                                                       \
    }                                                                     \
  } while (0)

int main() {
  constexpr int64_t kMost = 2048;
  auto check = [](int64_t b) {
    const int64_t step = g500::group_buckets(b, kMost);
    if (b <= kMost) {
      CHECK(step == 1);
    } else if (b > kMost * kMost) {
      CHECK(step == 0);
    } else {  // two passes make every number up to the square of one's
      const int64_t groups = g500::ceil_div(b, step);
      CHECK(step > 1 && step <= kMost && groups <= kMost);
      CHECK((step & (step - 1)) == 0 && step < 2 * groups + 2 && groups <= 4 * step);
    }
  };
  for (int64_t b = 1; b <= kMost * kMost + 10; b += b < 10000 ? 1 : 97) check(b);
  for (int64_t b : {kMost * kMost / 2, kMost * kMost / 2 + 1, kMost * kMost - 1, kMost * kMost,
                    kMost * kMost + 1})
    check(b);
  std::puts("partition ok");
}
