// MOSP's path costs by path doubling (cpp/src/algorithms/mosp/sequential.cpp:172-236): the persistent
// kernel and how its launches are tried. A host build with stand-ins for the device's builtins runs the
// kernel with a thread per workgroup and checks what it reports when a wait gives up.
#pragma once

#include "common.hpp"

namespace dyng_hip {

/// What the path doubling tells the host (pinned memory).
struct path_report {
  int missing;  ///< the lowest vertex whose tree edge is not in the graph (INT32_MAX: none)
  int ended;    ///< 1: every workgroup ended
};

struct path_params {
  int64_t* acc[2];   ///< sums of the even and odd rounds; acc[0] is the caller's
  int32_t* jump[2];
  int32_t n;
  int columns;
  grid_sync_state* bar;
  unsigned long long limit;  ///< ticks a grid barrier waits at most
  unsigned int rounds;       ///< at most: log2(n) rounded up, and one
  const int* missing;
  int* finished;             ///< workgroups that ended, zero at the start
  path_report* report;
};

constexpr int kPathBlock = 1024;
constexpr int kPathSlots = 4;  ///< vertices of a thread in flight

/// Path doubling: in each round every vertex adds its ancestor's sum and jumps to the ancestor's
/// ancestor, until none has one. A vertex's jump is -1 in the round after its sum became final (that
/// round copies the sum to the other buffer) and -2 from then on (both buffers hold it: a round only
/// passes the -2 on). One launch of resident workgroups with a grid barrier per round, at which each
/// tells how many of its vertices go on: a launch per round had to queue log2(n) + 1 of them, 21 for
/// 2^20 vertices whose trees are 5 rounds deep, and each empty one took 7 us with its gap. The rounds
/// read what other workgroups wrote, so those accesses are at device scope.
__global__ void __launch_bounds__(kPathBlock) k_path_costs(path_params p) {
  const int threads = static_cast<int>(gridDim.x * blockDim.x);
  const int tid = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  const grid_place at{blockIdx.x, gridDim.x};
  int cur = 0;
  for (unsigned int round = 1; round <= p.rounds; ++round) {
    const int64_t* acc_in = p.acc[cur];
    const int32_t* jump_in = p.jump[cur];
    int64_t* acc_out = p.acc[cur ^ 1];
    int32_t* jump_out = p.jump[cur ^ 1];
    bool more = false;  // some vertex of this thread still has an ancestor
    for (int64_t v0 = tid; v0 < p.n; v0 += int64_t{kPathSlots} * threads) {
      int32_t j[kPathSlots], up[kPathSlots];
#pragma unroll
      for (int q = 0; q < kPathSlots; ++q) {
        const int64_t v = v0 + int64_t{q} * threads;
        j[q] = v < p.n ? ld(&jump_in[v]) : -2;
      }
#pragma unroll
      for (int q = 0; q < kPathSlots; ++q) up[q] = j[q] >= 0 ? ld(&jump_in[j[q]]) : -2;
      for (int c = 0; c < p.columns; ++c) {
        int64_t a[kPathSlots], b[kPathSlots];
#pragma unroll
        for (int q = 0; q < kPathSlots; ++q) {
          const int64_t v = v0 + int64_t{q} * threads;
          a[q] = j[q] != -2 ? ld(&acc_in[v * p.columns + c]) : 0;
          b[q] = j[q] >= 0 ? ld(&acc_in[static_cast<int64_t>(j[q]) * p.columns + c]) : 0;
        }
#pragma unroll
        for (int q = 0; q < kPathSlots; ++q) {
          const int64_t v = v0 + int64_t{q} * threads;
          if (j[q] != -2) st(&acc_out[v * p.columns + c], a[q] + b[q]);
        }
      }
#pragma unroll
      for (int q = 0; q < kPathSlots; ++q) {
        const int64_t v = v0 + int64_t{q} * threads;
        const int32_t next = j[q] < 0 ? -2 : up[q] < 0 ? -1 : up[q];
        if (v < p.n) st(&jump_out[v], next);
        more = more || next >= 0;
      }
    }
    cur ^= 1;
    const unsigned int mine = static_cast<unsigned int>(__syncthreads_count(more ? 1 : 0));
    const grid_found found = grid_barrier<false>(p.bar, at, round, p.limit, [&] { grid_arrive(p.bar, at, round, mine); });
    if (!found.ok) return;  // uniform: `finished` stays short and the host finds `ended` clear
    if (found.published == 0) break;
  }
  if (cur == 1) {
    // an odd number of rounds: the sums are in the other buffer, each vertex's written by this thread
    for (int64_t v = tid; v < p.n; v += threads) {
      for (int c = 0; c < p.columns; ++c) p.acc[0][v * p.columns + c] = ld(&p.acc[1][v * p.columns + c]);
    }
  }
  // The last workgroup to get here tells the host: one that gave up a wait may have done so as the last
  // round was released to the others, and its part of an odd last round is not home then.
  if (threadIdx.x == 0 && atomicAdd(p.finished, 1) == static_cast<int>(gridDim.x) - 1) {
    p.report->missing = *p.missing;
    p.report->ended = 1;
  }
}

/// The doubling on `blocks` workgroups; if a wait gave up, again on one. Other work can hold enough of the
/// device for the whole of the limit that the workgroups are not all resident; one workgroup waits for
/// nobody, so the costs come late then and never not at all. `attempt(blocks)` starts from the tree
/// edges' costs and says whether every workgroup ended.
template <class Attempt>
bool run_path_costs(unsigned int blocks, Attempt attempt) {
  return attempt(blocks) || (blocks > 1 && attempt(1u));
}

}  // namespace dyng_hip
