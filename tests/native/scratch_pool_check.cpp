// Host check of the scratch pool (dyng_amd/csrc/scratch_pool.hpp) with malloc: which block a call gets, how
// many stay, what happens when memory runs out, and several threads at once. Prints "ok" or what differs
// and exits nonzero.
#include "../../dyng_amd/csrc/scratch_pool.hpp"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <thread>

using dyng_hip::scratch_block;
using dyng_hip::scratch_pool;

namespace {

std::atomic<long> live{0}, made{0};
std::atomic<size_t> most{~size_t{0}};  ///< no memory past this size

void* get(size_t bytes) {
  if (bytes > most.load()) return nullptr;
  ++live;
  ++made;
  return std::malloc(bytes);
}
void put(void* p) {
  --live;
  std::free(p);
}

#define EXPECT(what)                                \
  do {                                              \
    if (!(what)) {                                  \
      std::printf("line %d: %s\n", __LINE__, #what); \
      return 1;                                     \
    }                                               \
  } while (0)

}  // namespace

int main() {
  {
    scratch_pool pool(get, put);
    pool.join();
    scratch_block a = pool.take(1000);
    EXPECT(a.p != nullptr && a.bytes >= 1000 && live == 1);
    pool.give(a);
    EXPECT(live == 1);
    scratch_block b = pool.take(900);  // the kept one
    EXPECT(b.p == a.p && made == 1);
    pool.give(b);
    b = pool.take(1 << 20);  // too small: another in its place
    EXPECT(b.bytes >= (1 << 20) && b.bytes <= (1 << 20) + (1 << 17) && live == 1 && made == 2);
    scratch_block c = pool.take(5000), d = pool.take(100000), e = pool.take(200000);  // calls at the same time
    EXPECT(live == 4);
    pool.give(c);
    pool.give(b);
    pool.give(d);
    pool.give(e);
    EXPECT(live == scratch_pool::kKept);
    c = pool.take(1);  // the smaller of the two largest
    EXPECT(c.bytes >= 200000 && c.bytes < (1 << 20));
    pool.give(c);
    // memory runs out: what is kept is given up, and exactly what was asked for is tried
    most = 3000000;
    scratch_block f = pool.take(3000000);
    EXPECT(f.p != nullptr && f.bytes == 3000000 && live == 1);
    scratch_block g = pool.take(4000000);
    EXPECT(g.p == nullptr && g.bytes == 0 && live == 1);
    most = ~size_t{0};
    pool.give(f);
    pool.join();
    pool.leave();
    EXPECT(live == 1);  // a user is left
    pool.leave();
    EXPECT(live == 0);  // none is: nothing is kept
    pool.give(pool.take(10));
    EXPECT(live == 0);
  }
  {
    // two sizes far apart in turn keep a block each
    scratch_pool pool(get, put);
    pool.join();
    scratch_block a = pool.take(1 << 20), b = pool.take(1 << 10);
    pool.give(a);
    pool.give(b);
    const long before = made;
    for (int i = 0; i < 20; ++i) pool.give(pool.take(i % 2 ? 1 << 20 : 1 << 10));
    EXPECT(made == before);
    pool.leave();
    EXPECT(live == 0);
  }
  {
    scratch_pool pool(get, put);
    std::atomic<bool> wrong{false};
    std::vector<std::thread> threads;
    for (int t = 0; t < 6; ++t) {
      threads.emplace_back([&, t] {
        pool.join();
        std::mt19937 rng(t);
        for (int i = 0; i < 3000; ++i) {
          const size_t bytes = 1 + rng() % 50000;
          scratch_block b = pool.take(bytes);
          if (b.p == nullptr || b.bytes < bytes) wrong = true;
          std::memset(b.p, t + 1, bytes);
          for (size_t k = 0; k < bytes; k += 97) {
            if (static_cast<unsigned char*>(b.p)[k] != t + 1) wrong = true;  // nobody else has it
          }
          pool.give(b);
        }
        pool.leave();
      });
    }
    for (auto& t : threads) t.join();
    EXPECT(!wrong && live == 0);
  }
  std::printf("ok\n");
  return 0;
}
