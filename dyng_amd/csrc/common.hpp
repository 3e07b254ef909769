// Shared device and host helpers of the HIP sssp path (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "row_search.hpp"

namespace dyng_hip {

using u64 = unsigned long long;
constexpr u64 packed_inf = ~0ULL;
/// DISTANCE_INF of the reference (INT64_MAX / 4): distances at or above half of it are
/// unreachable (cpp/include/dyng/core/types.hpp:91).
constexpr int64_t sssp_infinity = INT64_MAX / 4;
/// The largest finite distance an output may hold (kernels.cuh:40).
constexpr u64 output_max_distance = static_cast<u64>(sssp_infinity / 2 - 1);

#define DYNG_DEV __device__ __forceinline__

/// Packed (distance << bits | parent) words; bits == 0 means distance-only words
/// (kernels.cuh:52-78). The all-ones parent field is "no parent"; the all-ones word is INF.
struct packing {
  int bits;
  u64 no_parent;
  DYNG_DEV u64 pack(u64 distance, int32_t parent) const {
    if (bits == 0) return distance;
    return (distance << bits) | (parent < 0 ? no_parent : static_cast<u64>(static_cast<uint32_t>(parent)));
  }
  DYNG_DEV u64 distance(u64 word) const { return word >> bits; }
  DYNG_DEV int32_t parent(u64 word) const {
    const u64 p = word & no_parent;
    return p == no_parent ? -1 : static_cast<int32_t>(p);
  }
};

// ---- agent-scope loads and stores of data other workgroups write during the same kernel ----

template <typename T>
DYNG_DEV T ld(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
DYNG_DEV void st(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

DYNG_DEV int lane() { return static_cast<int>(__lane_id()); }

/// A value that is the same on every lane (a grid-wide count read after a barrier), moved to a
/// scalar register.
DYNG_DEV int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
DYNG_DEV unsigned long long uniform(unsigned long long v) {
  const unsigned int lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned int>(v));
  const unsigned int hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned int>(v >> 32));
  return (static_cast<unsigned long long>(hi) << 32) | lo;
}

DYNG_DEV u64 lanes_below() {
  const int l = lane();
  return l == 0 ? 0ULL : (~0ULL >> (64 - l));
}

/// The value of v in lane `from` (uniform over the wave), through a scalar register: a few cycles,
/// where a shuffle is an LDS operation of about a hundred.
DYNG_DEV int from_lane(int v, int from) { return __builtin_amdgcn_readlane(v, from); }

/// Inclusive prefix sum over the wave by six DPP additions (row shifts within 16 lanes, then the row
/// broadcasts): about 0.05 us, where six shuffles through LDS take 0.35 us.
DYNG_DEV int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

/// Fold `f` over the wave by the same six moves: the last lane has the result (a lane without a
/// source folds its own value in again, so f(x, x) must be x).
template <class F>
DYNG_DEV int wave_fold(int v, F f) {
  v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x111, 0xf, 0xf, false));
  v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x112, 0xf, 0xf, false));
  v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x114, 0xf, 0xf, false));
  v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x118, 0xf, 0xf, false));
  v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xa, 0xf, false));
  v = f(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xc, 0xf, false));
  return v;
}

/// The same sums within each row of 16 lanes.
DYNG_DEV int row_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  return v;
}

/// Reserve one slot of a shared list per lane with `pred`: one atomicAdd per wave (the active
/// lanes with pred vote, the lowest of them reserves for all). Every active lane must call it.
DYNG_DEV int wave_append(int* counter, bool pred) {
  const u64 mask = __ballot(pred);
  if (!pred) return -1;
  const int leader = __builtin_amdgcn_readfirstlane(__ffsll(static_cast<long long>(mask)) - 1);
  const int rank = __popcll(mask & lanes_below());
  int base = 0;
  if (lane() == leader) base = atomicAdd(counter, __popcll(mask));
  base = from_lane(base, leader);
  return base + rank;
}

DYNG_DEV u64 wave_min(u64 v) {
  for (int off = 32; off > 0; off >>= 1) {
    const u64 o = __shfl_xor(v, off);
    v = o < v ? o : v;
  }
  return v;
}

DYNG_DEV u64 wave_sum(u64 v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

/// Reduce v over the workgroup with op; every thread gets the result. Every thread of the
/// workgroup calls it. `part` is an LDS array of at least blockDim.x / 64 entries (reused across
/// calls: the leading barrier keeps a call from overwriting what the previous one still reads).
/// Counters that every workgroup bumps are single addresses, and device-scope atomics on one
/// address serialize (1-2 ns each), so kernels reduce per workgroup before their atomics.
template <class T, class Op>
DYNG_DEV T block_reduce(T v, T* part, Op op) {
  for (int off = 32; off > 0; off >>= 1) v = op(v, static_cast<T>(__shfl_xor(v, off)));
  const int waves = static_cast<int>((blockDim.x + 63) / 64);
  __syncthreads();
  if (lane() == 0) part[threadIdx.x / 64] = v;
  __syncthreads();
  T t = part[0];
  for (int w = 1; w < waves; ++w) t = op(t, part[w]);
  return t;
}

struct op_sum {
  template <class T>
  DYNG_DEV T operator()(T a, T b) const { return a + b; }
};
struct op_max {
  template <class T>
  DYNG_DEV T operator()(T a, T b) const { return b > a ? b : a; }
};


/// Grid-wide barrier of a persistent kernel whose workgroups are all resident (the grid is sized to at
/// most what the occupancy calculator says fits at once), in two halves.
///
/// Arrivals go up a two-level tree: workgroup b adds to the word of group b % G (G = min(16,
/// workgroups)); the last member of a group to arrive adds the group's totals to the root's word,
/// and the last group stores the release to every group's line, which that group's members poll.
/// Device-scope atomics on one address serialize, so 16-way groups cut the arrival chain from one
/// atomic per workgroup to about 16 + 16, and no line is polled by more than a sixteenth of the
/// grid: polls slow everybody's memory operations (with 256 idle workgroups polling one line, a
/// working one's dependent loads took 0.56 us each instead of 0.27). Each line is 128 bytes.
///
/// A workgroup may do work of its own between its arrival and its wait. An arrival also carries how
/// many entries the workgroup published and whether any of them is marked; the release brings the
/// totals, so the length of a list comes with the wait instead of one more dependent load.
///
/// Rounds strictly follow each other: a workgroup arrives at round r + 1 only after its own wait for
/// round r. Round r counts in words r % 4, which start at zero; a workgroup arrives at round r + 2
/// only when everybody has arrived at r + 1 and so left r, so a group's first workgroup clears the
/// group's word of round r (and workgroup 0 the root's) as it arrives at r + 2. It waits for the
/// answer to that arrival and for its earlier stores with it, so the word is clear before it arrives
/// at r + 3 and anybody at r + 4. The state is cleared once per launch.
///
/// Measured on MI355X, 256 workgroups of 1024 threads with one of them late: 4.5 us for eight
/// dependent loads of the late one and from its arrival to the last departure (6.2 us with 64-bit
/// divisions by the member counts in the arrival and one polled line; 6.3 us when everybody polls
/// all the groups' words).
///
/// Two flavours of the whole barrier. `Fenced` adds an agent-scope release fence before the arrival
/// and an acquire fence after the wait (on MI355X they write back and invalidate the XCD's L2), so
/// plain loads and stores on either side are ordered. Without it the barrier only waits for each
/// wave's own memory operations to complete (s_waitcnt) before the arrival: the phases it separates
/// must access every location that another workgroup writes during the kernel with agent-scope
/// operations only (ld / st / atomics), which are coherent across the XCDs' L2s by themselves.
/// That saves the two cache walks, the bulk of a fenced barrier's cost.
///
/// Every wait is bounded: a workgroup that waits longer than `limit` ticks of the 100 MHz
/// real-time counter raises `abort`, and every workgroup that sees `abort` while waiting leaves
/// too (both are checked on the first poll and every 32nd after). The wait then returns
/// false and the caller leaves the kernel, so a grid whose workgroups could not all be resident
/// ends with an error instead of spinning forever.
struct alignas(128) barrier_line {
  /// of round r % 4: arrivals in bits 0-15, arrivals with a marked entry in bits 16-31, published
  /// entries in bits 32-63
  unsigned long long v[4];
  unsigned long long pad0[4];
  /// the last released round in bits 0-30, whether an entry was marked in bit 31, published entries
  /// in bits 32-63
  unsigned long long release;
  unsigned long long pad1[7];
};
static_assert(sizeof(barrier_line) == 128, "one line of the barrier is one cache line");

constexpr unsigned int kBarrierGroups = 16;

struct grid_sync_state {
  barrier_line abort;  ///< v[0] nonzero: a wait timed out
  barrier_line root;
  barrier_line group[kBarrierGroups];
  barrier_line spare;  ///< keeps the state's size, and with it the no-allocation scratch's limit on graphs
};

/// What a wait found: the entries published in the round, and whether any was marked. ok: 0 when the
/// wait gave up.
struct grid_found {
  int ok, published, marked;
};

/// A workgroup's number among the `blocks` that meet at a barrier (a launch may hold several teams, each
/// with a barrier of its own).
struct grid_place {
  unsigned int block, blocks;
};

/// Arrive at round `round` (1, 2, ...), with `published` entries to tell of, some of them marked or
/// not. One thread of the workgroup calls it, after every wave's loads and stores have completed and
/// a workgroup barrier.
DYNG_DEV void grid_arrive(grid_sync_state* s, const grid_place& at, unsigned int round, unsigned int published,
                          bool marked = false) {
  const unsigned int blocks = at.blocks;
  const unsigned int G = blocks < kBarrierGroups ? blocks : kBarrierGroups;
  const unsigned int grp = at.block % G;
  const unsigned int members = blocks / G + (blocks % G > grp ? 1u : 0u);
  barrier_line& line = s->group[grp];
  if (at.block < G && round > 2) {
    const unsigned int old = (round - 2) & 3u;
    __hip_atomic_store(&line.v[old], 0ULL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (at.block == 0) __hip_atomic_store(&s->root.v[old], 0ULL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  const unsigned long long mine =
      1ULL | (marked ? 1ULL << 16 : 0ULL) | (static_cast<unsigned long long>(published) << 32);
  unsigned long long all =
      mine + __hip_atomic_fetch_add(&line.v[round & 3u], mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if ((all & 0xffff) != members) return;
  all = (all & ~0xffffULL) | 1ULL;  // one group arrived
  all += __hip_atomic_fetch_add(&s->root.v[round & 3u], all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if ((all & 0xffff) != G) return;
  const unsigned long long word =
      (all & 0xffffffff00000000ULL) | ((all & 0xffff0000ULL) != 0 ? 1ULL << 31 : 0ULL) | (round & 0x7fffffffu);
  for (unsigned int g = 0; g < G; ++g) {
    __hip_atomic_store(&s->group[g].release, word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

/// Wait for round `round`, at which this workgroup has arrived. Called by the thread that arrived.
DYNG_DEV grid_found grid_poll(grid_sync_state* s, const grid_place& at, unsigned int round, unsigned long long limit) {
  const unsigned int blocks = at.blocks;
  const unsigned int G = blocks < kBarrierGroups ? blocks : kBarrierGroups;
  const unsigned long long* const word = &s->group[at.block % G].release;
  const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
  unsigned int polls = 0;
  for (;;) {
    const unsigned long long v = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((static_cast<unsigned int>(v) & 0x7fffffffu) == (round & 0x7fffffffu)) {
      return grid_found{1, static_cast<int>(v >> 32), static_cast<int>((v >> 31) & 1)};
    }
    if ((polls++ & 31u) == 0) {
      if (__hip_atomic_load(&s->abort.v[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) break;
      if (__builtin_amdgcn_s_memrealtime() - t0 > limit) {
        __hip_atomic_store(&s->abort.v[0], 1ULL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
    }
    __builtin_amdgcn_s_sleep(1);
  }
  return grid_found{0, 0, 0};
}

/// The whole barrier: every thread of the workgroup calls it; `arrive()` (one thread, after the
/// workgroup barrier) is grid_arrive with what this workgroup publishes.
template <bool Fenced, class Arrive>
DYNG_DEV grid_found grid_barrier(grid_sync_state* s, const grid_place& at, unsigned int round, unsigned long long limit,
                                 Arrive arrive) {
  __shared__ grid_found found;
  // every wave's loads and stores have completed (at the scope they were issued with) before the
  // arrival
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    if (Fenced) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    arrive();
    found = grid_poll(s, at, round, limit);
    if (Fenced) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
  return grid_found{uniform(found.ok), uniform(found.published), uniform(found.marked)};
}

}  // namespace dyng_hip
