// Which of several repairs share a launch. Host code only.
#pragma once

#include <algorithm>
#include <cstdint>

namespace dyng_hip {

/// Edges a repair may scan past the average of those beside it and still share their launch. Side by side,
/// `count` runs have a share of the processors each and take the time of the slowest; one after another,
/// each has the whole device, and each pays again for its chain of barriers and round trips (70 to 100 us).
/// A heavy run beside light ones (RMAT-22, milliseconds of a whole update side by side and one after
/// another): beside one, 0.98 and 1.01 at 2.8 M edges, 1.50 and 1.51 at 3.7 M, 5.8 and 5.5 at 18 M; beside
/// three, 1.06 and 1.12 at 2.8 M, 2.06 and 1.88 at 7.2 M (1.64 with the heavy run alone and the light ones
/// sharing a launch), 15.7 and 14.6 at 47 M (14.1).
constexpr int64_t kAloneEdges = int64_t{4} << 20;

/// `edges`: what each run's result scanned in its last repair (0: none yet). The runs in the order of
/// their launches go to `order`; the first ones, whose number is returned, take a launch of their own and
/// the others share one.
inline int runs_alone(const int64_t* edges, int count, int* order) {
  int64_t rest = 0;  // edges of the runs from the one looked at on
  for (int i = 0; i < count; ++i) {
    order[i] = i;
    rest += edges[i];
  }
  std::stable_sort(order, order + count, [&](int a, int b) { return edges[a] > edges[b]; });
  int alone = 0;
  for (; count - alone > 1; ++alone) {
    const int64_t most = edges[order[alone]], others = count - alone - 1;
    rest -= most;
    if (others * (most - kAloneEdges) <= rest) break;
  }
  return count - alone == 1 ? count : alone;
}

}  // namespace dyng_hip
