// Host check of MOSP's path doubling (dyng_amd/csrc/path_costs.hpp), a thread of the host per workgroup:
// the sums of random trees on 1 to 8 workgroups, and what is reported when a workgroup gives up a wait at
// the moment the round is released. Prints "ok <checks>" or what differs and exits nonzero.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstring>
#include <random>
#include <thread>
#include <vector>

#include "../../dyng_amd/csrc/path_costs.hpp"

using namespace dyng_hip;

namespace {

/// The workgroup that gives up, at which round (0: none): in that round it is the first to arrive, polls
/// once, and its clock runs past every limit when all the others, which the round's release lets go, have
/// left the kernel.
std::atomic<int> quitter{-1};
std::atomic<unsigned int> quit_round{0};
std::atomic<bool> polled{false};
std::atomic<int> left{0};
thread_local unsigned int clock_reads = 0, barriers = 0;

bool is_quitter() { return static_cast<int>(blockIdx.x) == quitter.load(); }

}  // namespace

/// A wait reads the clock as it begins and after its first poll.
unsigned long long __builtin_amdgcn_s_memrealtime() {
  ++clock_reads;
  if (!is_quitter() || clock_reads != 2 || (barriers + 1) / 2 != quit_round.load()) return 0;
  polled = true;
  while (left.load() + 1 < static_cast<int>(gridDim.x)) std::this_thread::yield();
  return 1000000000ULL;
}
void __builtin_amdgcn_s_sleep(int) { std::this_thread::yield(); }

/// A round of the grid barrier has a workgroup barrier before the arrival and one behind the wait.
void __syncthreads() {
  if ((++barriers & 1) != 0) clock_reads = 0;
  if (quitter.load() < 0 || barriers != 2 * quit_round.load() - 1) return;
  while (!is_quitter() && !polled.load()) std::this_thread::yield();
}

namespace {

struct problem {
  int n, columns;
  std::vector<int> parent;
  std::vector<int64_t> edge, want;
};

problem random_tree(std::mt19937_64& rng, int n, int columns, int reach) {
  problem t{n, columns, std::vector<int>(n, -1), std::vector<int64_t>(size_t(n) * columns), {}};
  for (int v = 0; v < n; ++v) {
    t.parent[v] = v == 0 || rng() % 50 == 0 ? -1 : static_cast<int>(v - 1 - rng() % std::min<uint64_t>(v, reach));
    for (int c = 0; c < columns; ++c) t.edge[size_t(v) * columns + c] = rng() % 1000;
  }
  t.want = t.edge;
  for (int v = 0; v < n; ++v) {
    for (int c = 0; c < columns; ++c) {
      if (t.parent[v] >= 0) t.want[size_t(v) * columns + c] += t.want[size_t(t.parent[v]) * columns + c];
    }
  }
  return t;
}

/// One launch on `blocks` workgroups: whether the kernel says that it ended, and the sums.
bool launch(const problem& t, unsigned int blocks, unsigned long long limit, std::vector<int64_t>& costs) {
  costs = t.edge;
  std::vector<int64_t> other(costs.size(), -7);
  std::vector<int32_t> jump_a(t.parent.begin(), t.parent.end()), jump_b(t.n, -9);
  static grid_sync_state bar;
  std::memset(&bar, 0, sizeof(bar));
  int state[2] = {INT32_MAX, 0};
  path_report report{INT32_MAX, 0};
  unsigned int rounds = 1;
  while ((int64_t{1} << rounds) < t.n) ++rounds;
  path_params p{{costs.data(), other.data()}, {jump_a.data(), jump_b.data()}, t.n, t.columns, &bar, limit, rounds + 1,
                &state[0], &state[1], &report};
  left = 0;
  polled = false;
  std::vector<std::thread> groups;
  for (unsigned int b = 0; b < blocks; ++b) {
    groups.emplace_back([&, b] {
      blockIdx.x = b;
      gridDim.x = blocks;
      barriers = 0;
      k_path_costs(p);
      ++left;
    });
  }
  for (auto& g : groups) g.join();
  return report.ended != 0;
}

}  // namespace

int main() {
  std::mt19937_64 rng(7);
  int checks = 0;
  std::vector<int64_t> costs;
  for (int n : {1, 2, 5, 64, 1000}) {
    for (int reach : {1, 3, 1000}) {
      const problem t = random_tree(rng, n, 1 + n % 3, reach);
      for (unsigned int blocks : {1u, 2u, 3u, 8u}) {
        if (!launch(t, blocks, 1000000000000ULL, costs) || costs != t.want) {
          std::printf("n %d reach %d on %u workgroups: wrong\n", n, reach, blocks);
          return 1;
        }
        ++checks;
      }
    }
  }
  // a workgroup that gives up in the last round while the others are released: chains of 2 to 300 vertices
  // end after even and after odd numbers of rounds; after odd ones its part is not brought home
  for (int n : {2, 3, 5, 9, 17, 33, 65, 129, 257, 300}) {
    problem t = random_tree(rng, n, 1, 1);
    for (int v = 1; v < n; ++v) t.parent[v] = v - 1;
    t.want = t.edge;
    for (int v = 1; v < n; ++v) t.want[v] += t.want[v - 1];
    unsigned int rounds = 1;  // until no vertex has an ancestor
    while ((1 << rounds) <= n - 1) ++rounds;
    for (unsigned int blocks : {2u, 5u}) {
      quitter = static_cast<int>(blocks) - 1;
      quit_round = rounds;
      const bool ended = launch(t, blocks, 1000, costs);
      quitter = -1;
      if (ended) {
        std::printf("chain of %d on %u workgroups, one gave up: reported as ended, sums %s\n", n, blocks,
                    costs == t.want ? "right" : "wrong");
        return 1;
      }
      ++checks;
      // and the costs are there all the same, from a launch that waits for nobody
      std::vector<unsigned int> tried;
      const bool done = run_path_costs(blocks, [&](unsigned int on) {
        tried.push_back(on);
        quitter = on > 1 ? static_cast<int>(on) - 1 : -1;
        return launch(t, on, on > 1 ? 1000 : 0, costs);
      });
      if (!done || tried != std::vector<unsigned int>{blocks, 1u} || costs != t.want) {
        std::printf("chain of %d on %u workgroups, one gave up: no costs\n", n, blocks);
        return 1;
      }
      ++checks;
    }
  }
  std::printf("ok %d\n", checks);
  return 0;
}
