// Host check of which repairs share a launch (dyng_amd/csrc/team_rule.hpp). Prints "ok" or the first case
// that differs and exits nonzero.
#include "../../dyng_amd/csrc/team_rule.hpp"

#include <cstdio>
#include <vector>

namespace {

constexpr int64_t M = 1 << 20;

bool expect(const std::vector<int64_t>& edges, int want_alone, const std::vector<int>& want_order) {
  std::vector<int> order(edges.size(), -1);
  const int alone = dyng_hip::runs_alone(edges.data(), static_cast<int>(edges.size()), order.data());
  if (alone == want_alone && order == want_order) return true;
  std::printf("edges");
  for (auto e : edges) std::printf(" %lld", static_cast<long long>(e));
  std::printf(": %d alone (want %d), order", alone, want_alone);
  for (auto o : order) std::printf(" %d", o);
  std::printf("\n");
  return false;
}

}  // namespace

int main() {
  const bool ok = expect({}, 0, {}) && expect({0}, 1, {0}) && expect({50 * M}, 1, {0}) &&
                  expect({0, 0, 0, 0}, 0, {0, 1, 2, 3}) &&                    // nothing known: side by side
                  expect({50 * M, 50 * M, 50 * M, 50 * M}, 0, {0, 1, 2, 3}) &&  // heavy alike
                  expect({0, 0, 8 * M, 0}, 1, {2, 0, 1, 3}) &&                // one heavy, the others share
                  expect({0, 8 * M}, 2, {1, 0}) &&                            // two: one after another
                  expect({0, 40 * M, 20 * M, 1000}, 2, {1, 2, 3, 0}) &&       // two heavy ones, each alone
                  expect({9 * M, 6 * M, 7 * M, 8 * M}, 0, {0, 3, 2, 1}) &&    // unequal, but not by much
                  expect({4 * M, 0, 0, 0}, 0, {0, 1, 2, 3}) &&                // at the limit
                  expect({4 * M + 1, 0, 0, 0}, 1, {0, 1, 2, 3}) &&
                  expect({5 * M, 1 * M, 1 * M}, 0, {0, 1, 2}) && expect({5 * M + 1, 1 * M, 1 * M}, 1, {0, 1, 2});
  if (!ok) return 1;
  std::printf("ok\n");
  return 0;
}
