// The device graph of the HIP sssp path: out- and in-rows in slack storage, built on the device
// and updated in place by each batch.
//
// Layout (HBM): per vertex an int2 {offset, length}, a capacity, the length of the row's base run
// and the count of dead entries in it; one slot arena per direction holding the neighbour ids,
// then one int32 weight column per objective (column k at w + k * slot_cap). A row is two sorted
// runs: the base [offset, offset + base) and the tail [offset + base, offset + length), each
// sorted by neighbour id with parallel edges in the order they were added; among equal
// neighbours the base entry is the older one. A deletion marks an entry dead (the sign bit of its
// neighbour id) instead of moving the row. So the first alive (u,v) of row u in MOSP's append
// order is the first alive entry of v's run in the base, else in the tail. A batch rewrites only
// a row's tail while the tail stays short and the base has few dead entries (tail_limit,
// dead_limit); otherwise the whole row is merged into one new base run. A row's capacity is
// len + ceil(len * headroom) + 2; a row that outgrows it moves to the free tail of the arena;
// compaction rebuilds the arena when the tail runs short.
//
// A batch (MOSP applyChangeBatch under upsert_last_wins, cpp/src/graph/apply_host.cpp:57-401) is
// applied without leaving the device:
//   1. k_batch_scan: ids, self-loops and weight ranges, before anything changes.
//   2. k_group_front, Step 0 (apply_host.cpp:80-147): self-loops, vertex growth, undirected
//      expansion; each effective operation goes to the group of its row, for the out-rows and for
//      the in-rows. Rows are hashed into groups, so all of a row's operations are in one.
//   3. k_group_pairs, a workgroup per group: the operations sorted by row, neighbour and application
//      order (deletions first), then one thread per pair (u,v) replays its operations on the runs of
//      v in row u (searches in both runs): deletions mark the first alive match dead, insertions
//      overwrite the first alive match (upsert) or add a pending entry; then the weight-increase
//      flags of :348-394 (final first (u,v) against the original first (u,v)). The in-rows replay
//      the same operations; with parallel edges their groups come in a second launch, which matches
//      the copy that each operation took by its old weights. Last, the group's touched rows are
//      planned: a tail merged by a thread, a wave or a workgroup, or the whole row into a new base,
//      and the staging and relocation slots that takes.
//   4. k_tails and k_rows merge the alive entries with the pending ones (positions from prefix sums
//      and searches), in place, or at the arena's tail when the row outgrew its capacity. For a small
//      batch they are queued behind the plan and look for themselves whether the arenas take it; else
//      the host reads the plan, and grows or compacts an arena first.
// Batches that a group cannot take (more operations on a row than a workgroup sorts), past the
// groups' number, or checked by an error mode before anything changes go through one device-wide
// stable sort of both directions' keys (u << b | v) instead of steps 2 and 3, then a launch each for
// the pairing, the scans and the plan (rows_sorted).
#include "internal.hpp"

#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <rocprim/rocprim.hpp>

#include <algorithm>
#include <cmath>
#include <map>
#include <memory>
#include <mutex>
#include <type_traits>
#include <vector>

namespace dyng_hip {

namespace {

constexpr int kBlock = 256;
constexpr int32_t kDead = static_cast<int32_t>(0x80000000u);
constexpr u64 kNoKey = ~0ULL;

unsigned int blocks_for(int64_t work, int block = kBlock) {
  int64_t b = (work + block - 1) / block;
  if (b < 1) b = 1;
  if (b > 65535LL * 16) b = 65535LL * 16;
  return static_cast<unsigned int>(b);
}

int bits_for(int64_t n_after) {
  int b = 1;
  while ((int64_t{1} << b) <= n_after) ++b;  // n_after < 2^b, so ids < 2^b - 1 < the all-ones key
  return b;
}

DYNG_DEV int64_t lower_key(const u64* keys, int64_t lo, int64_t hi, u64 key) {
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (keys[mid] < key) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// ---------------------------------------------------------------------------------------------
// rocPRIM wrappers
// ---------------------------------------------------------------------------------------------

void sort_pairs(dbuf<unsigned char>& tmp, const u64* kin, u64* kout, const uint32_t* vin,
                uint32_t* vout, size_t n, int end_bit, hipStream_t s) {
  if (n == 0) return;
  size_t bytes = 0;
  DYNG_HIP_TRY(rocprim::radix_sort_pairs(nullptr, bytes, kin, kout, vin, vout, n, 0, end_bit, s));
  tmp.reserve(bytes);
  DYNG_HIP_TRY(rocprim::radix_sort_pairs(static_cast<void*>(tmp.p), bytes, kin, kout, vin, vout, n, 0,
                                         end_bit, s));
}

template <typename T>
void exclusive_scan(dbuf<unsigned char>& tmp, const T* in, T* out, size_t n, hipStream_t s) {
  if (n == 0) return;
  size_t bytes = 0;
  DYNG_HIP_TRY(rocprim::exclusive_scan(nullptr, bytes, in, out, T{0}, n, rocprim::plus<T>(), s));
  tmp.reserve(bytes);
  DYNG_HIP_TRY(rocprim::exclusive_scan(static_cast<void*>(tmp.p), bytes, in, out, T{0}, n,
                                       rocprim::plus<T>(), s));
}

/// The exclusive prefix sums of four int32 arrays of n entries (the pending and killed flags of
/// both directions' operations), in two launches: the sums of tiles of kScan4Tile entries, then
/// each tile scanned from the sum of the tiles before it (each workgroup adds those up itself).
/// No chain of look-backs between workgroups: on a few hundred thousand entries a decoupled
/// look-back scan is a serial chain of device-scope round trips (rocPRIM's took 16 us here, its
/// state initialisation included).
constexpr int kScan4Block = 1024;
constexpr int kScan4Items = 1;  ///< entries per thread: tiles of 1024 (four per thread measured 5 us slower)
constexpr int kScan4Tile = kScan4Block * kScan4Items;

struct scan4_args {
  const int32_t* in[4];
  int32_t* out[4];
  int64_t n;
  int4* tile_sums;
};

/// Sum over the workgroup of one int4 per thread; thread 0 gets it.
DYNG_DEV int4 block_sum4(int4 v, int4* part) {
  for (int off = 32; off > 0; off >>= 1) {
    v.x += __shfl_xor(v.x, off);
    v.y += __shfl_xor(v.y, off);
    v.z += __shfl_xor(v.z, off);
    v.w += __shfl_xor(v.w, off);
  }
  if (lane() == 0) part[threadIdx.x / 64] = v;
  __syncthreads();
  int4 t = make_int4(0, 0, 0, 0);
  if (threadIdx.x == 0) {
    for (int w = 0; w < static_cast<int>(blockDim.x / 64); ++w) {
      t.x += part[w].x;
      t.y += part[w].y;
      t.z += part[w].z;
      t.w += part[w].w;
    }
  }
  return t;
}

__global__ void __launch_bounds__(kScan4Block) k_scan4_tiles(scan4_args a) {
  __shared__ int4 part[kScan4Block / 64];
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kScan4Tile;
  int4 v = make_int4(0, 0, 0, 0);
  for (int j = 0; j < kScan4Items; ++j) {
    const int64_t i = t0 + static_cast<int64_t>(j) * kScan4Block + threadIdx.x;
    if (i < a.n) {
      v.x += a.in[0][i];
      v.y += a.in[1][i];
      v.z += a.in[2][i];
      v.w += a.in[3][i];
    }
  }
  const int4 t = block_sum4(v, part);
  if (threadIdx.x == 0) a.tile_sums[blockIdx.x] = t;
}

__global__ void __launch_bounds__(kScan4Block) k_scan4_apply(scan4_args a) {
  __shared__ int4 part[kScan4Block / 64];
  __shared__ int4 wave_sum[kScan4Block / 64];
  __shared__ int4 base;
  // the sum of the tiles before this one
  int4 v = make_int4(0, 0, 0, 0);
  for (int b = threadIdx.x; b < static_cast<int>(blockIdx.x); b += blockDim.x) {
    const int4 x = a.tile_sums[b];
    v.x += x.x;
    v.y += x.y;
    v.z += x.z;
    v.w += x.w;
  }
  const int4 before = block_sum4(v, part);
  if (threadIdx.x == 0) base = before;
  // this thread's kScan4Items consecutive entries, their sums, then the workgroup's exclusive scan
  const int64_t first = static_cast<int64_t>(blockIdx.x) * kScan4Tile + static_cast<int64_t>(threadIdx.x) * kScan4Items;
  int32_t x[4][kScan4Items];
  int4 own = make_int4(0, 0, 0, 0);
#pragma unroll
  for (int j = 0; j < kScan4Items; ++j) {
    const int64_t i = first + j;
    const bool in = i < a.n;
    x[0][j] = in ? a.in[0][i] : 0;
    x[1][j] = in ? a.in[1][i] : 0;
    x[2][j] = in ? a.in[2][i] : 0;
    x[3][j] = in ? a.in[3][i] : 0;
    own.x += x[0][j];
    own.y += x[1][j];
    own.z += x[2][j];
    own.w += x[3][j];
  }
  int4 inc = own;  // inclusive scan over the wave
  for (int off = 1; off < 64; off <<= 1) {
    const int4 y = make_int4(__shfl_up(inc.x, off), __shfl_up(inc.y, off), __shfl_up(inc.z, off), __shfl_up(inc.w, off));
    if (lane() >= off) {
      inc.x += y.x;
      inc.y += y.y;
      inc.z += y.z;
      inc.w += y.w;
    }
  }
  const int wv = static_cast<int>(threadIdx.x / 64);
  if (lane() == 63) wave_sum[wv] = inc;
  __syncthreads();  // wave sums and base are in LDS
  int4 run = base;
  for (int w = 0; w < wv; ++w) {
    run.x += wave_sum[w].x;
    run.y += wave_sum[w].y;
    run.z += wave_sum[w].z;
    run.w += wave_sum[w].w;
  }
  run.x += inc.x - own.x;
  run.y += inc.y - own.y;
  run.z += inc.z - own.z;
  run.w += inc.w - own.w;
#pragma unroll
  for (int j = 0; j < kScan4Items; ++j) {
    const int64_t i = first + j;
    if (i < a.n) {
      a.out[0][i] = run.x;
      a.out[1][i] = run.y;
      a.out[2][i] = run.z;
      a.out[3][i] = run.w;
    }
    run.x += x[0][j];
    run.y += x[1][j];
    run.z += x[2][j];
    run.w += x[3][j];
  }
}

void exclusive_scan4(dbuf<unsigned char>& tmp, const int32_t* a, const int32_t* b, const int32_t* c, const int32_t* d,
                     int32_t* oa, int32_t* ob, int32_t* oc, int32_t* od, size_t n, hipStream_t s) {
  if (n == 0) return;
  const int64_t tiles = (static_cast<int64_t>(n) + kScan4Tile - 1) / kScan4Tile;
  tmp.reserve(static_cast<size_t>(tiles) * sizeof(int4));
  scan4_args args{{a, b, c, d}, {oa, ob, oc, od}, static_cast<int64_t>(n), reinterpret_cast<int4*>(tmp.p)};
  hipLaunchKernelGGL(k_scan4_tiles, dim3(static_cast<unsigned>(tiles)), dim3(kScan4Block), 0, s, args);
  hipLaunchKernelGGL(k_scan4_apply, dim3(static_cast<unsigned>(tiles)), dim3(kScan4Block), 0, s, args);
  DYNG_HIP_TRY(hipGetLastError());
}

template <typename T>
__global__ void k_fill(T* p, int64_t n, T v) {
  for (int64_t i = blockIdx.x * int64_t{blockDim.x} + threadIdx.x; i < n; i += int64_t{gridDim.x} * blockDim.x) p[i] = v;
}

template <typename T>
void fill(T* p, int64_t n, T v, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill<T>, dim3(blocks_for(n)), dim3(kBlock), 0, s, p, n, v);
  DYNG_HIP_TRY(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------
// Construction
// ---------------------------------------------------------------------------------------------

/// One key per (expanded) input edge: (u << b | v), or kNoKey for a dropped self-loop or the
/// missing reverse arc of a directed edge. val = slot (edge index * stride + reversed).
__global__ void k_edge_keys(const int32_t* src, const int32_t* dst, int64_t count, int stride,
                            int directed, int drop_self_loops, int vbits, u64* keys, uint32_t* vals) {
  const int64_t total = count * stride;
  for (int64_t e = blockIdx.x * int64_t{blockDim.x} + threadIdx.x; e < total; e += int64_t{gridDim.x} * blockDim.x) {
    const int64_t j = e / stride;
    const int r = static_cast<int>(e % stride);
    const int32_t u0 = src[j], v0 = dst[j];
    bool valid = true;
    if (r == 1 && (directed || u0 == v0)) valid = false;
    if (u0 == v0 && drop_self_loops) valid = false;
    const int32_t u = r ? v0 : u0, v = r ? u0 : v0;
    keys[e] = valid ? ((static_cast<u64>(u) << vbits) | static_cast<u64>(v)) : kNoKey;
    vals[e] = static_cast<uint32_t>(e);
  }
}

/// keep[i]: sorted edge i survives (a simple graph keeps the last of a run of equal pairs).
__global__ void k_keep(const u64* keys, int64_t N, int allow_parallel, int32_t* keep) {
  for (int64_t i = blockIdx.x * int64_t{blockDim.x} + threadIdx.x; i <= N; i += int64_t{gridDim.x} * blockDim.x) {
    if (i == N) { keep[i] = 0; continue; }
    const u64 k = keys[i];
    keep[i] = (k != kNoKey && (allow_parallel || i + 1 == N || keys[i + 1] != k)) ? 1 : 0;
  }
}

/// Degree and capacity of every row from the sorted keys and the keep prefix.
__global__ void k_row_degrees(const u64* keys, int64_t N, const int32_t* keep_prefix, int64_t n,
                              int vbits, double headroom, int2* meta, int32_t* cap, int64_t* cap64) {
  for (int64_t u = blockIdx.x * int64_t{blockDim.x} + threadIdx.x; u < n; u += int64_t{gridDim.x} * blockDim.x) {
    const int64_t a = lower_key(keys, 0, N, static_cast<u64>(u) << vbits);
    const int64_t b = lower_key(keys, a, N, static_cast<u64>(u + 1) << vbits);
    const int deg = keep_prefix[b] - keep_prefix[a];
    const int c = deg + static_cast<int>(ceil(deg * headroom)) + 2;
    meta[u] = make_int2(0, deg);
    cap[u] = c;
    cap64[u] = c;
  }
}

__global__ void k_set_offsets(const int64_t* off64, int64_t n, int2* meta) {
  for (int64_t u = blockIdx.x * int64_t{blockDim.x} + threadIdx.x; u < n; u += int64_t{gridDim.x} * blockDim.x) {
    meta[u].x = static_cast<int32_t>(off64[u]);
  }
}

/// Scatter the kept sorted edges into their rows. Weights come from the input list
/// (w_in[edge * K + k], edge = slot / stride) or, when `from_slots`, from an arena column
/// (w_in[k * in_slot_cap + slot]).
__global__ void k_fill_rows(const u64* keys, const uint32_t* vals, int64_t N, const int32_t* keep,
                            const int32_t* keep_prefix, int vbits, int stride, const int2* meta,
                            int32_t* nbr, int32_t* w, int64_t slot_cap, int K, const int32_t* w_in,
                            int from_slots, int64_t in_slot_cap) {
  const u64 mask = (1ULL << vbits) - 1;
  for (int64_t i = blockIdx.x * int64_t{blockDim.x} + threadIdx.x; i < N; i += int64_t{gridDim.x} * blockDim.x) {
    if (!keep[i]) continue;
    const u64 key = keys[i];
    const int64_t u = static_cast<int64_t>(key >> vbits);
    const int32_t v = static_cast<int32_t>(key & mask);
    const int64_t a = lower_key(keys, 0, i + 1, static_cast<u64>(u) << vbits);
    const int64_t slot = meta[u].x + (keep_prefix[i] - keep_prefix[a]);
    nbr[slot] = v;
    const uint32_t val = vals[i];
    for (int k = 0; k < K; ++k) {
      w[k * slot_cap + slot] = from_slots ? w_in[k * in_slot_cap + val] : w_in[(static_cast<int64_t>(val) / stride) * K + k];
    }
  }
}

/// Keys of the in-rows from the out-rows: (v << b | u), val = out slot.
__global__ void k_reverse_keys(const int2* meta, const int32_t* nbr, int64_t n, int vbits, u64* keys,
                               uint32_t* vals, const int64_t* row_pos) {
  // one wave per row
  const int64_t wave = (blockIdx.x * int64_t{blockDim.x} + threadIdx.x) / 64;
  const int64_t waves = (int64_t{gridDim.x} * blockDim.x) / 64;
  for (int64_t u = wave; u < n; u += waves) {
    const int2 mt = meta[u];
    const int64_t base = row_pos[u];
    for (int j = lane(); j < mt.y; j += 64) {
      const int32_t v = nbr[mt.x + j];
      keys[base + j] = (static_cast<u64>(v) << vbits) | static_cast<u64>(u);
      vals[base + j] = static_cast<uint32_t>(mt.x + j);
    }
  }
}

__global__ void k_len64(const int2* meta, int64_t n, int64_t* out) {
  for (int64_t u = blockIdx.x * int64_t{blockDim.x} + threadIdx.x; u < n; u += int64_t{gridDim.x} * blockDim.x) out[u] = meta[u].y;
}

/// Column summary of every objective: pass 0 max and sum, pass 1 the count of maximal weights.
/// Each wave takes 64 consecutive rows at a time: a short row is scanned by its own lane, a long
/// one by the whole wave (a wave per row would leave most lanes idle on sparse rows and chain one
/// row's latency after another).
constexpr int kShortRow = 16;

__global__ void k_column_summary(const int2* meta, const int32_t* nbr, const int32_t* w, int64_t n, int64_t slot_cap,
                                 int K, int pass, apply_control* ctl) {
  const int64_t wave = (blockIdx.x * int64_t{blockDim.x} + threadIdx.x) / 64;
  const int64_t waves = (int64_t{gridDim.x} * blockDim.x) / 64;
  for (int k = 0; k < K; ++k) {
    long long mx = 0, sum = 0, cnt = 0, bad = 0;
    const long long target = ctl->col_max[k];
    const int32_t* col = w + k * slot_cap;
    auto visit = [&](int64_t slot) {
      if (nbr[slot] < 0) return;  // dead
      const long long x = col[slot];
      if (pass == 0) {
        mx = x > mx ? x : mx;
        sum += x;
        bad += x < 1 ? 1 : 0;
      } else {
        cnt += x == target ? 1 : 0;
      }
    };
    for (int64_t r0 = wave * 64; r0 < n; r0 += waves * 64) {
      const int64_t u = r0 + lane();
      const int2 mt = u < n ? meta[u] : make_int2(0, 0);
      const bool is_long = mt.y > kShortRow;
      if (!is_long) {
        for (int j = 0; j < mt.y; ++j) visit(mt.x + int64_t{j});
      }
      u64 longs = __ballot(is_long);
      while (longs) {
        const int l = __ffsll(static_cast<unsigned long long>(longs)) - 1;
        longs &= longs - 1;
        const int off = __shfl(mt.x, l), len = __shfl(mt.y, l);
        for (int j = lane(); j < len; j += 64) visit(off + int64_t{j});
      }
    }
    if (pass == 0) {
      mx = static_cast<long long>(wave_min(~static_cast<u64>(mx)));
      mx = static_cast<long long>(~static_cast<u64>(mx));
      sum = static_cast<long long>(wave_sum(static_cast<u64>(sum)));
      bad = static_cast<long long>(wave_sum(static_cast<u64>(bad)));
      if (lane() == 0) {
        atomicMax(reinterpret_cast<unsigned long long*>(&ctl->col_max[k]), static_cast<unsigned long long>(mx));
        atomicAdd(reinterpret_cast<unsigned long long*>(&ctl->col_dsum[k]), static_cast<unsigned long long>(sum));
        if (bad) atomicAdd(reinterpret_cast<unsigned long long*>(&ctl->col_bad[k]), static_cast<unsigned long long>(bad));
      }
    } else {
      cnt = static_cast<long long>(wave_sum(static_cast<u64>(cnt)));
      if (lane() == 0) atomicAdd(reinterpret_cast<unsigned long long*>(&ctl->col_dcount[k]), static_cast<unsigned long long>(cnt));
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Apply
// ---------------------------------------------------------------------------------------------

/// Batch scan (before anything changes): id range, self-loops, weight range per objective. The
/// insertions and deletions are read in one loop (their loads in flight together); each workgroup
/// folds its values by lane-to-lane moves and one barrier and writes them to pinned host memory, where
/// the host folds the workgroups': no control block sent up, no copy back. A batch of 10: 11 us of
/// shuffles and atomics between two copies of 4 us each before.
constexpr int kScanBlock = 1024;
constexpr int64_t kGatherBytes = int64_t{1} << 20;  ///< host batches up to this many bytes go as one copy from pinned memory
constexpr int kScanColumns = 4;  ///< weight columns per pass of the batch scan
__global__ void __launch_bounds__(kScanBlock) k_batch_scan(const int32_t* ins_src, const int32_t* ins_dst,
                                                            const int32_t* ins_w, int64_t num_ins,
                                                            const int32_t* del_src, const int32_t* del_dst,
                                                            int64_t num_del, int K, scan_part* parts) {
  constexpr int kVals = 4 + 2 * kScanColumns;
  __shared__ int part[kScanBlock / 64][kVals];
  const int64_t stride = int64_t{gridDim.x} * blockDim.x;
  const int64_t first = blockIdx.x * int64_t{blockDim.x} + threadIdx.x;
  scan_part& to = parts[blockIdx.x];
  for (int k0 = 0; k0 == 0 || k0 < K; k0 += kScanColumns) {
    int mn = INT32_MAX, mx = -1, sl_i = 0, sl_d = 0;
    int top[kScanColumns], low[kScanColumns];
#pragma unroll
    for (int c = 0; c < kScanColumns; ++c) {
      top[c] = 0;
      low[c] = 1;
    }
    const int64_t total = k0 == 0 && num_del > num_ins ? num_del : num_ins;
    for (int64_t i = first; i < total; i += stride) {
      const bool ins = i < num_ins, del = k0 == 0 && i < num_del;
      int32_t u = 0, v = 0, du = 0, dv = 0, x[kScanColumns];
      if (ins && k0 == 0) {
        u = ins_src[i];
        v = ins_dst[i];
      }
      if (del) {
        du = del_src[i];
        dv = del_dst[i];
      }
#pragma unroll
      for (int c = 0; c < kScanColumns; ++c) x[c] = ins && k0 + c < K ? ins_w[i * K + k0 + c] : 1;
      if (ins && k0 == 0) {
        mn = min(mn, min(u, v));
        mx = max(mx, max(u, v));
        sl_i += u == v ? 1 : 0;
      }
      if (del) {
        mn = min(mn, min(du, dv));
        sl_d += du == dv ? 1 : 0;
      }
#pragma unroll
      for (int c = 0; c < kScanColumns; ++c) {
        if (ins && k0 + c < K) top[c] = max(top[c], x[c]);
        low[c] = min(low[c], x[c]);
      }
    }
    // the last lane has the wave's, then a thread per value the workgroup's
    auto least = [](int a, int b) { return min(a, b); };
    auto most = [](int a, int b) { return max(a, b); };
    mn = wave_fold(mn, least);
    mx = wave_fold(mx, most);
    sl_i = wave_scan(sl_i);
    sl_d = wave_scan(sl_d);
#pragma unroll
    for (int c = 0; c < kScanColumns; ++c) {
      top[c] = wave_fold(top[c], most);
      low[c] = wave_fold(low[c], least);
    }
    if (k0 > 0) __syncthreads();  // the last pass's values are read
    if (lane() == 63) {
      int* mine = part[threadIdx.x / 64];
      mine[0] = mn;
      mine[1] = mx;
      mine[2] = sl_i;
      mine[3] = sl_d;
#pragma unroll
      for (int c = 0; c < kScanColumns; ++c) {
        mine[4 + c] = top[c];
        mine[4 + kScanColumns + c] = low[c];
      }
    }
    __syncthreads();
    const int q = static_cast<int>(threadIdx.x);
    if (q < kVals) {
      const bool column = q >= 4;
      const int c = k0 + ((q - 4) & (kScanColumns - 1));
      const bool is_max = q == 1 || (column && q < 4 + kScanColumns), is_sum = q == 2 || q == 3;
      int t = part[0][q];
      for (int w = 1; w < kScanBlock / 64; ++w) {
        const int x = part[w][q];
        t = is_sum ? t + x : is_max ? max(t, x) : min(t, x);
      }
      if (!column && k0 == 0) to.id[q] = t;
      if (column && c < K) (is_max ? to.wmax : to.wmin)[c] = t;
    }
  }
}

struct op_layout {
  int64_t num_first, num_second;  ///< batch operations of the first / second kind
  int first_is_del;               ///< deletions_first
  int stride;                     ///< 1 directed, 2 undirected (reverse arc slot)
  DYNG_DEV bool is_del(int64_t e) const {
    return (e < num_first * stride) ? first_is_del != 0 : first_is_del == 0;
  }
  DYNG_DEV int64_t local(int64_t e) const { return e < num_first * stride ? e : e - num_first * stride; }
  DYNG_DEV int64_t del_base() const { return first_is_del ? 0 : num_first * stride; }
  DYNG_DEV int64_t ins_base() const { return first_is_del ? num_first * stride : 0; }
};

/// Ranks of offending operations in the error modes, in the order the reference's host apply
/// meets them (apply_host.cpp:80-252): first the deletions naming a vertex past the vertex count
/// (batch order), then row by row (ascending u), within a row the first phase's operations (the
/// deletions when deletions_first) before the second phase's, each in batch order. The lowest
/// rank is the error reported. Layout: bit 63 row phase, bits 62-32 the row, bit 31 the second
/// phase, bits 30-0 the operation's batch index.
constexpr unsigned long long kNoError = ~0ULL;
DYNG_DEV unsigned long long error_rank_prescan(int64_t j) { return static_cast<unsigned long long>(j); }
DYNG_DEV unsigned long long error_rank_row(int32_t u, int second_phase, int64_t j) {
  return (1ULL << 63) | (static_cast<unsigned long long>(u) << 32) | (static_cast<unsigned long long>(second_phase) << 31) |
         static_cast<unsigned long long>(j);
}

__global__ void k_make_ops(op_layout L, const int32_t* ins_src, const int32_t* ins_dst,
                           const int32_t* del_src, const int32_t* del_dst, int directed,
                           int drop_self_loops, int64_t n_after, int vbits, u64* keys, uint32_t* vals,
                           int32_t* e_del_src, int32_t* e_del_dst, int32_t* e_ins_src,
                           int32_t* e_ins_dst, uint8_t* e_inc, int32_t* e_fw, int K, int missing_delete_error,
                           apply_control* ctl) {
  const int64_t total = (L.num_first + L.num_second) * L.stride;
  unsigned long long dropped = 0, ignored = 0;
  for (int64_t e = blockIdx.x * int64_t{blockDim.x} + threadIdx.x; e < total; e += int64_t{gridDim.x} * blockDim.x) {
    const bool del = L.is_del(e);
    const int64_t loc = L.local(e);
    const int64_t j = loc / L.stride;
    const int r = static_cast<int>(loc % L.stride);
    const int32_t u0 = del ? del_src[j] : ins_src[j];
    const int32_t v0 = del ? del_dst[j] : ins_dst[j];
    bool valid = true;
    if (r == 1 && (directed || u0 == v0)) valid = false;
    if (valid && u0 == v0 && drop_self_loops) {
      valid = false;
      dropped += 1;
    }
    const int32_t u = r ? v0 : u0, v = r ? u0 : v0;
    if (valid && del && (u >= n_after || v >= n_after)) {
      valid = false;
      ignored += 1;
      // no such vertex, so no such edge: in the error mode, the batch's first such deletion
      // (apply_host.cpp:116-138 finds these before any row)
      if (missing_delete_error) atomicMin(&ctl->first_error, error_rank_prescan(j));
    }
    // Both directions' keys go through one sort: the out-row key (u, v) at e and the in-row key
    // (v, u) at total + e, tagged with bit 2 * vbits so that every out-key sorts before every
    // in-key (what an operation does to the in-row is decided later by the out-row pass). A
    // dropped operation takes the all-ones key of its half (no vertex id is all ones); k_untag
    // restores kNoKey and removes the tag after the sort.
    const u64 low = (u64{1} << (2 * vbits)) - 1;
    const u64 tag = u64{1} << (2 * vbits);
    keys[e] = valid ? ((static_cast<u64>(u) << vbits) | static_cast<u64>(v)) : low;
    vals[e] = static_cast<uint32_t>(e);
    keys[total + e] = tag | (valid ? ((static_cast<u64>(v) << vbits) | static_cast<u64>(u)) : low);
    vals[total + e] = static_cast<uint32_t>(e);
    if (del) {
      e_del_src[loc] = valid ? u : -1;
      e_del_dst[loc] = valid ? v : -1;
    } else {
      e_ins_src[loc] = valid ? u : -1;
      e_ins_dst[loc] = valid ? v : -1;
      for (int k = 0; k < K; ++k) e_inc[loc * K + k] = 0;
      if (e_fw != nullptr) {
        for (int k = 0; k < K; ++k) e_fw[loc * K + k] = -1;
      }
    }
  }
  dropped = wave_sum(dropped);
  ignored = wave_sum(ignored);
  if (lane() == 0) {
    if (dropped) atomicAdd(&ctl->dropped_self_loops, dropped);
    if (ignored) atomicAdd(&ctl->ignored_deletions, ignored);
  }
}

/// After the joint sort: the keys without their direction tag, kNoKey for dropped operations.
__global__ void k_untag(u64* keys, int64_t count, int vbits) {
  const u64 low = (u64{1} << (2 * vbits)) - 1;
  for (int64_t i = blockIdx.x * int64_t{blockDim.x} + threadIdx.x; i < count; i += int64_t{gridDim.x} * blockDim.x) {
    const u64 k = keys[i] & low;
    keys[i] = k == low ? kNoKey : k;
  }
}

/// Rows up to this many entries are merged by one wave, longer ones by a workgroup.
constexpr int kMergeSmall = 512;

struct out_pair_params {
  op_layout L;
  const u64* keys;
  const uint32_t* vals;
  int64_t N;
  int64_t stride;  ///< of the weight columns of pend_w and of the iop arrays
  int vbits;
  int K;
  int64_t n_before;  ///< rows that existed before the batch (classification)
  int upsert;        ///< on_existing_insert: 1 upsert, 0 ignore
  const int32_t* ins_w;  ///< batch insertion weights (j * K + k)
  int2* meta;
  const int32_t* base;
  int32_t* dead;
  int32_t* nbr;
  int32_t* w;
  int64_t slot_cap;
  int32_t* pend_alive;
  int32_t* kill;    ///< 1: the operation killed a tail entry
  int32_t* pend_w;  ///< k * N + position
  uint8_t* e_inc;
  /// simple graphs: per insertion (batch slot, K weights) the pair's weights after the batch, -1
  /// if the pair is gone (null with parallel edges, where several entries may hold the pair)
  int32_t* e_fw;
  // what each operation (by batch slot e) does to the in-rows: kInNone, or the type and weights
  int32_t* iop_type;
  int32_t* iop_wold;
  int32_t* iop_wnew;
  int32_t* mark;
  int mark_gen;
  int4* touched;  ///< rows whose entries change: row, and its operations (-1: in row_a and row_b)
  int32_t* flag;  ///< grouped: per operation, whether its pair changes the row's entries
  int32_t* row_a;  ///< per vertex: first operation of its row in the sorted keys
  int32_t* row_b;  ///< per vertex: one past its last operation
  apply_control* ctl;
};

enum { kInDelete = 0, kInModify = 1, kInInsert = 2, kInNone = 3 };

/// The entries of neighbour v in a row's two sorted runs: [lb, ub) in the base, [tl, tu) in the
/// tail (row-relative indices).
struct run_pair {
  int bl, lb, ub, tl, tu;
};

/// One probe per round: a batch's operations search different rows, so each probe is a line of its own,
/// and the lines are what bounds a large batch's pairing (1,000,000 operations on RMAT-23: 510 us with
/// one probe per round, 552 with three, 600 with seven; 100,000 on RMAT-22: 112, 119 and 134).
DYNG_DEV run_pair find_runs(const int32_t* row, int base_len, int len, int32_t v) {
  run_pair r;
  r.bl = base_len;
  r.lb = row_lower_bound<1>(row, 0, base_len, v);
  r.ub = row_upper_bound_from(row, r.lb, base_len, v);
  r.tl = row_lower_bound<1>(row, base_len, len, v);
  r.tu = row_upper_bound_from(row, r.tl, len, v);
  return r;
}

/// The error modes, checked before anything changes (read only): one thread per (u, v) segment of
/// the sorted out-row keys replays the segment's operations in batch order on counts of the alive
/// (u, v) entries (old ones in the row, pending ones of the batch). A deletion that finds none is a
/// missing edge, an insertion that finds one an existing edge (apply_host.cpp:117-120, 206-226);
/// the lowest rank of an offending operation lands in ctl->first_error.
__global__ void __launch_bounds__(kBlock) k_check_pairs(op_layout L, const u64* keys, const uint32_t* vals,
                                                         int64_t N, int vbits, int64_t n_before, const int2* meta,
                                                         const int32_t* base, const int32_t* nbr,
                                                         int missing_delete_error, int existing_insert_error,
                                                         apply_control* ctl) {
  const int64_t i = blockIdx.x * int64_t{blockDim.x} + threadIdx.x;
  if (i >= N) return;
  const u64 key = keys[i];
  if (key == kNoKey || (i > 0 && keys[i - 1] == key)) return;
  const u64 mask = (1ULL << vbits) - 1;
  const int32_t u = static_cast<int32_t>(key >> vbits);
  const int32_t v = static_cast<int32_t>(key & mask);
  int alive = 0;
  if (u < n_before) {
    const int2 mt = meta[u];
    const int32_t* row = nbr + mt.x;
    const run_pair rr = find_runs(row, base[u], mt.y, v);
    for (int x = rr.lb; x < rr.ub; ++x) alive += row[x] >= 0 ? 1 : 0;
    for (int x = rr.tl; x < rr.tu; ++x) alive += row[x] >= 0 ? 1 : 0;
  }
  unsigned long long first = kNoError;
  for (int64_t q = i; q < N && keys[q] == key; ++q) {
    const int64_t e = vals[q];
    const int second = e >= L.num_first * L.stride ? 1 : 0;
    const int64_t j = L.local(e) / L.stride;
    if (L.is_del(e)) {
      if (alive > 0) {
        --alive;
      } else if (missing_delete_error) {
        first = min(first, error_rank_row(u, second, j));
      }
    } else if (alive > 0) {
      if (existing_insert_error) first = min(first, error_rank_row(u, second, j));
    } else {
      ++alive;  // appended
    }
  }
  if (first != kNoError) atomicMin(&ctl->first_error, first);
}

/// Record where row r's operations start and end in the sorted keys (row = key >> vbits).
DYNG_DEV void mark_row_range(const u64* keys, int64_t i, int64_t N, int vbits, int32_t* row_a, int32_t* row_b) {
  const u64 key = keys[i];
  const u64 r = key >> vbits;
  if (i == 0 || (keys[i - 1] >> vbits) != r) row_a[r] = static_cast<int32_t>(i);
  if (i + 1 == N || (keys[i + 1] >> vbits) != r) row_b[r] = static_cast<int32_t>(i + 1);
}

/// A pair whose operations change its row's entries: flagged for the plan of the row's group
/// (`kGrouped`: one workgroup holds all the row's operations), or the row listed.
template <bool kGrouped, class Params>
DYNG_DEV void touch_row(const Params& p, bool structural, int64_t i, int32_t r, int* touched_count) {
  if (kGrouped) {
    if (structural) p.flag[i] = 1;
    return;
  }
  const bool first_touch = structural && atomicExch(&p.mark[r], p.mark_gen) != p.mark_gen;
  const int t = wave_append(touched_count, first_touch);
  if (first_touch) p.touched[t] = make_int4(r, -1, -1, 0);
}

/// The out-row pass of thread i (every thread of the workgroup calls it: it ends with the
/// workgroup's counter reduction).
template <int kThreads, bool kGrouped>
DYNG_DEV void out_pairs(const out_pair_params& p, int64_t i) {
  unsigned long long c_ins = 0, c_upd = 0, c_del = 0, c_ign_del = 0, c_ign_ins = 0;
  // weight sum and count-at-maximum deltas of columns 0..3 (named, not an array: a private
  // array indexed by a runtime column would live in scratch memory)
  long long ds0 = 0, ds1 = 0, ds2 = 0, ds3 = 0, dc0 = 0, dc1 = 0, dc2 = 0, dc3 = 0;
  const u64 mask = (1ULL << p.vbits) - 1;
  const int K = p.K;
  if (i == p.N) {
    p.pend_alive[i] = 0;
    p.kill[i] = 0;
  }
  if (i < p.N) {
    const u64 key = p.keys[i];
    if (!kGrouped && key != kNoKey) mark_row_range(p.keys, i, p.N, p.vbits, p.row_a, p.row_b);
    if (key == kNoKey) {
      p.pend_alive[i] = 0;
      p.kill[i] = 0;
    } else if (i == 0 || p.keys[i - 1] != key) {
      int64_t j = i + 1;
      while (j < p.N && p.keys[j] == key) ++j;
      const int32_t u = static_cast<int32_t>(key >> p.vbits);
      const int32_t v = static_cast<int32_t>(key & mask);
      const int2 mt = p.meta[u];
      const int32_t* row = p.nbr + mt.x;
      const run_pair rr = find_runs(row, u < p.n_before ? p.base[u] : 0, mt.y, v);
      // the first alive (u,v) of the row in order: the base run's, then the tail's
      auto first_alive = [&]() -> int {
        for (int x = rr.lb; x < rr.ub; ++x) {
          if (row[x] >= 0) return x;
        }
        for (int x = rr.tl; x < rr.tu; ++x) {
          if (row[x] >= 0) return x;
        }
        return -1;
      };
      const int init_hit = u < p.n_before ? first_alive() : -1;
      const bool had = init_hit >= 0;
      // the first operation that overwrote the original first (u,v)'s weights: its recorded old
      // weights are the original ones (else the slot still holds them)
      int64_t first_mod = -1;
      bool structural = false;
      auto account = [&](int k, long long wold, long long wnew, bool removed, bool added) {
        const long long target = p.ctl->col_max[k];
        const long long ds = (added ? wnew : 0) - (removed ? wold : 0);
        const long long dc = ((added && wnew == target) ? 1 : 0) - ((removed && wold == target) ? 1 : 0);
        if (k == 0) {
          ds0 += ds;
          dc0 += dc;
        } else if (k == 1) {
          ds1 += ds;
          dc1 += dc;
        } else if (k == 2) {
          ds2 += ds;
          dc2 += dc;
        } else if (k == 3) {
          ds3 += ds;
          dc3 += dc;
        } else {
          if (ds) atomicAdd(reinterpret_cast<unsigned long long*>(&p.ctl->col_dsum[k]), static_cast<unsigned long long>(ds));
          if (dc) atomicAdd(reinterpret_cast<unsigned long long*>(&p.ctl->col_dcount[k]), static_cast<unsigned long long>(dc));
        }
      };
      for (int64_t q = i; q < j; ++q) {
        const int64_t e = p.vals[q];
        const bool del = p.L.is_del(e);
        p.pend_alive[q] = 0;
        p.kill[q] = 0;
        p.iop_type[e] = kInNone;
        // first alive match: old entries of the runs, then pending entries of this pair
        const int old_hit = first_alive();
        int64_t pend_hit = -1;
        if (old_hit < 0) {
          for (int64_t x = i; x < q; ++x) {
            if (p.pend_alive[x]) { pend_hit = x; break; }
          }
        }
        if (del) {
          if (old_hit >= 0) {
            p.nbr[mt.x + old_hit] = v | kDead;
            if (old_hit < rr.bl) {
              atomicAdd(&p.dead[u], 1);
            } else {
              p.kill[q] = 1;  // a tail entry
            }
            for (int k = 0; k < K; ++k) {
              const int32_t wo = p.w[k * p.slot_cap + mt.x + old_hit];
              p.iop_wold[k * p.stride + e] = wo;
              account(k, wo, 0, true, false);
            }
            p.iop_type[e] = kInDelete;
            structural = true;
            ++c_del;
          } else if (pend_hit >= 0) {
            p.pend_alive[pend_hit] = 0;
            for (int k = 0; k < K; ++k) {
              const int32_t wo = p.pend_w[k * p.stride + pend_hit];
              p.iop_wold[k * p.stride + e] = wo;
              account(k, wo, 0, true, false);
            }
            p.iop_type[e] = kInDelete;
            ++c_del;
          } else {
            ++c_ign_del;
          }
        } else {
          const int64_t bj = p.L.local(e) / p.L.stride;
          if (old_hit >= 0 || pend_hit >= 0) {
            if (!p.upsert) {
              ++c_ign_ins;
            } else {
              if (old_hit >= 0 && old_hit == init_hit && first_mod < 0) first_mod = e;
              for (int k = 0; k < K; ++k) {
                const int32_t wn = p.ins_w[bj * K + k];
                int32_t* slot = old_hit >= 0 ? &p.w[k * p.slot_cap + mt.x + old_hit] : &p.pend_w[k * p.stride + pend_hit];
                const int32_t wo = *slot;
                *slot = wn;
                p.iop_wold[k * p.stride + e] = wo;
                p.iop_wnew[k * p.stride + e] = wn;
                account(k, wo, wn, true, true);
              }
              p.iop_type[e] = kInModify;
              ++c_upd;
            }
          } else {
            p.pend_alive[q] = 1;
            for (int k = 0; k < K; ++k) {
              const int32_t wn = p.ins_w[bj * K + k];
              p.pend_w[k * p.stride + q] = wn;
              p.iop_wnew[k * p.stride + e] = wn;
              account(k, 0, wn, false, true);
            }
            p.iop_type[e] = kInInsert;
            structural = true;
            ++c_ins;
          }
        }
      }
      // weight-increase classification: final first (u,v) against the original first (u,v)
      if (had) {
        const int32_t* wf = nullptr;
        int64_t wf_stride = 0;
        const int final_hit = first_alive();
        if (final_hit >= 0) {
          wf = p.w + mt.x + final_hit;
          wf_stride = p.slot_cap;
        }
        if (wf == nullptr) {
          for (int64_t x = i; x < j; ++x) {
            if (p.pend_alive[x]) { wf = p.pend_w + x; wf_stride = p.stride; break; }
          }
        }
        if (wf != nullptr) {
          for (int64_t q = i; q < j; ++q) {
            const int64_t e = p.vals[q];
            if (p.L.is_del(e)) continue;
            const int64_t loc = p.L.local(e);
            for (int k = 0; k < K; ++k) {
              const int32_t orig = first_mod >= 0 ? p.iop_wold[k * p.stride + first_mod] : p.w[k * p.slot_cap + mt.x + init_hit];
              p.e_inc[loc * K + k] = wf[k * wf_stride] > orig ? 1 : 0;
            }
          }
        }
      }
      // simple graphs: the pair's final weights for each of its insertions (what the engine offers
      // the insertion's head, without searching the row again)
      if (p.e_fw != nullptr) {
        const int32_t* wf = nullptr;
        int64_t wf_stride = 0;
        const int final_hit = first_alive();
        if (final_hit >= 0) {
          wf = p.w + mt.x + final_hit;
          wf_stride = p.slot_cap;
        } else {
          for (int64_t x = i; x < j; ++x) {
            if (p.pend_alive[x]) { wf = p.pend_w + x; wf_stride = p.stride; break; }
          }
        }
        for (int64_t q = i; q < j; ++q) {
          const int64_t e = p.vals[q];
          if (p.L.is_del(e)) continue;
          const int64_t loc = p.L.local(e);
          for (int k = 0; k < K; ++k) p.e_fw[loc * K + k] = wf != nullptr ? wf[k * wf_stride] : -1;
        }
      }
      touch_row<kGrouped>(p, structural, i, u, &p.ctl->touched_out);
    }
  }
  // the workgroup's counters in one pass: wave sums by lane-to-lane moves (a count fits 32 bits; a
  // weight sum goes in three parts, modulo 2^64), one barrier, then a thread per counter adds the
  // waves' sums
  constexpr int kSums = 13;
  __shared__ u64 part[kThreads / 64][kSums];
  const int w = static_cast<int>(threadIdx.x) / 64;
  auto count_sum = [&](int q, long long x) {
    const int t = wave_scan(static_cast<int>(x));
    if (lane() == 63) part[w][q] = static_cast<u64>(static_cast<long long>(t));
  };
  auto weight_sum = [&](int q, long long x) {
    const int lo = wave_scan(static_cast<int>(x & 0xffff)), mid = wave_scan(static_cast<int>((x >> 16) & 0xffff)),
              hi = wave_scan(static_cast<int>(x >> 32));
    if (lane() == 63) {
      part[w][q] = static_cast<u64>(lo) + (static_cast<u64>(mid) << 16) + (static_cast<u64>(static_cast<uint32_t>(hi)) << 32);
    }
  };
  count_sum(0, static_cast<long long>(c_ins));
  count_sum(1, static_cast<long long>(c_upd));
  count_sum(2, static_cast<long long>(c_del));
  count_sum(3, static_cast<long long>(c_ign_del));
  count_sum(4, static_cast<long long>(c_ign_ins));
  weight_sum(5, ds0);
  count_sum(9, dc0);
  if (K > 1) {
    weight_sum(6, ds1);
    weight_sum(7, ds2);
    weight_sum(8, ds3);
    count_sum(10, dc1);
    count_sum(11, dc2);
    count_sum(12, dc3);
  }
  __syncthreads();
  const int q = static_cast<int>(threadIdx.x);
  if (q < kSums && (q < 5 || ((q - 5) & 3) < K)) {
    u64 t = 0;
    for (int wv = 0; wv < kThreads / 64; ++wv) t += part[wv][q];
    u64* to = &p.ctl->inserted_edges + q;  // inserted, updated, deleted, ignored deletions
    if (q == 4) to = &p.ctl->ignored_insertions;
    if (q >= 5) to = reinterpret_cast<u64*>(&p.ctl->col_dsum[q - 5]);
    if (q >= 9) to = reinterpret_cast<u64*>(&p.ctl->col_dcount[q - 9]);
    if (t != 0) atomicAdd(to, t);
  }
}

__global__ void __launch_bounds__(kBlock) k_out_pairs(out_pair_params p) {
  out_pairs<kBlock, false>(p, blockIdx.x * int64_t{blockDim.x} + threadIdx.x);
}

struct in_pair_params {
  op_layout L;
  const int32_t* ins_w;  ///< batch insertion weights (j * K + k), for the simple graphs' own replay
  int upsert;            ///< on_existing_insert: 1 upsert, 0 ignore
  const u64* keys;  ///< sorted in-operation keys (v << b | u)
  const uint32_t* vals;  ///< out-operation position of each
  int64_t N;
  int64_t stride;  ///< of the weight columns of pend_w and of the iop arrays
  int vbits;
  int K;
  const int32_t* iop_type;
  const int32_t* iop_wold;
  const int32_t* iop_wnew;
  int2* meta;
  const int32_t* base;
  int32_t* dead;
  int32_t* nbr;
  int32_t* w;
  int64_t slot_cap;
  int32_t* pend_alive;
  int32_t* kill;
  int32_t* pend_w;
  int32_t* mark;
  int mark_gen;
  int4* touched;  ///< rows whose entries change: row, and its operations (-1: in row_a and row_b)
  int32_t* flag;  ///< grouped: per operation, whether its pair changes the row's entries
  int32_t* row_a;
  int32_t* row_b;
  apply_control* ctl;
};

/// The in-row pass of a graph with parallel edges, thread i: each operation's effect as the out-row
/// pass recorded it.
template <bool kGrouped>
DYNG_DEV void in_pairs(const in_pair_params& p, int64_t i) {
  if (i == p.N) {
    p.pend_alive[i] = 0;
    p.kill[i] = 0;
  }
  if (i >= p.N) return;
  const u64 key = p.keys[i];
  if (key == kNoKey) {
    p.pend_alive[i] = 0;
    p.kill[i] = 0;
    return;
  }
  if (!kGrouped) mark_row_range(p.keys, i, p.N, p.vbits, p.row_a, p.row_b);
  if (i > 0 && p.keys[i - 1] == key) return;
  int64_t j = i + 1;
  while (j < p.N && p.keys[j] == key) ++j;
  const u64 mask = (1ULL << p.vbits) - 1;
  const int32_t v = static_cast<int32_t>(key >> p.vbits);
  const int32_t u = static_cast<int32_t>(key & mask);
  const int2 mt = p.meta[v];
  const int32_t* row = p.nbr + mt.x;
  const run_pair rr = find_runs(row, p.base[v], mt.y, u);
  const int K = p.K;
  bool structural = false;
  for (int64_t q = i; q < j; ++q) {
    p.pend_alive[q] = 0;
    p.kill[q] = 0;
    const uint32_t o = p.vals[q];  // the operation's batch slot
    const int type = p.iop_type[o];
    if (type == kInNone) continue;  // ignored by the out-row pass
    if (type == kInInsert) {
      p.pend_alive[q] = 1;
      for (int k = 0; k < K; ++k) p.pend_w[k * p.stride + q] = p.iop_wnew[k * p.stride + o];
      structural = true;
      continue;
    }
    // first alive entry of u with the old weights: the base run's, the tail's, then pending ones
    int old_hit = -1;
    for (int x = rr.lb; x < rr.tu && old_hit < 0; ++x) {
      if (x == rr.ub) x = rr.tl;
      if (x >= rr.tu) break;
      if (row[x] < 0) continue;
      bool same = true;
      for (int k = 0; k < K && same; ++k) same = p.w[k * p.slot_cap + mt.x + x] == p.iop_wold[k * p.stride + o];
      if (same) old_hit = x;
    }
    int64_t pend_hit = -1;
    if (old_hit < 0) {
      for (int64_t x = i; x < q && pend_hit < 0; ++x) {
        if (!p.pend_alive[x]) continue;
        bool same = true;
        for (int k = 0; k < K && same; ++k) same = p.pend_w[k * p.stride + x] == p.iop_wold[k * p.stride + o];
        if (same) pend_hit = x;
      }
    }
    if (old_hit < 0 && pend_hit < 0) {
      atomicOr(&p.ctl->error_bits, static_cast<int>(DYNG_HIP_DEVICE_ERROR_INTERNAL));
      continue;
    }
    if (type == kInDelete) {
      if (old_hit >= 0) {
        p.nbr[mt.x + old_hit] = u | kDead;
        if (old_hit < rr.bl) {
          atomicAdd(&p.dead[v], 1);
        } else {
          p.kill[q] = 1;  // a tail entry
        }
        structural = true;
      } else {
        p.pend_alive[pend_hit] = 0;
      }
    } else {
      for (int k = 0; k < K; ++k) {
        const int32_t wn = p.iop_wnew[k * p.stride + o];
        if (old_hit >= 0) p.w[k * p.slot_cap + mt.x + old_hit] = wn; else p.pend_w[k * p.stride + pend_hit] = wn;
      }
    }
  }
  touch_row<kGrouped>(p, structural, i, v, &p.ctl->touched_in);
}

__global__ void __launch_bounds__(kBlock) k_in_pairs(in_pair_params p) {
  in_pairs<false>(p, blockIdx.x * int64_t{blockDim.x} + threadIdx.x);
}

/// The in-row pass of a simple graph, thread i. A simple graph holds at most one alive (u, v), and
/// its in-row entry (v, u) carries the same weights, so replaying the segment's operations in
/// batch order on the in-row as the out-row pass replays them on the out-row (the first alive old
/// entry, else the first alive pending one; deletions remove it, insertions upsert or append)
/// reaches the same decisions and weights without that pass's results: both passes run in one
/// launch (k_pairs_simple). With parallel edges the copy an operation takes is matched by weight
/// to the out-row's (k_in_pairs, after k_out_pairs).
template <bool kGrouped>
DYNG_DEV void in_pairs_simple(const in_pair_params& p, int64_t i) {
  if (i == p.N) {
    p.pend_alive[i] = 0;
    p.kill[i] = 0;
  }
  if (i >= p.N) return;
  const u64 key = p.keys[i];
  if (key == kNoKey) {
    p.pend_alive[i] = 0;
    p.kill[i] = 0;
    return;
  }
  if (!kGrouped) mark_row_range(p.keys, i, p.N, p.vbits, p.row_a, p.row_b);
  if (i > 0 && p.keys[i - 1] == key) return;
  int64_t j = i + 1;
  while (j < p.N && p.keys[j] == key) ++j;
  const u64 mask = (1ULL << p.vbits) - 1;
  const int32_t v = static_cast<int32_t>(key >> p.vbits);
  const int32_t u = static_cast<int32_t>(key & mask);
  const int2 mt = p.meta[v];
  const int32_t* row = p.nbr + mt.x;
  const run_pair rr = find_runs(row, p.base[v], mt.y, u);
  const int K = p.K;
  auto first_alive = [&]() -> int {
    for (int x = rr.lb; x < rr.ub; ++x) {
      if (row[x] >= 0) return x;
    }
    for (int x = rr.tl; x < rr.tu; ++x) {
      if (row[x] >= 0) return x;
    }
    return -1;
  };
  bool structural = false;
  for (int64_t q = i; q < j; ++q) {
    p.pend_alive[q] = 0;
    p.kill[q] = 0;
    const int64_t e = p.vals[q];
    const int old_hit = first_alive();
    int64_t pend_hit = -1;
    if (old_hit < 0) {
      for (int64_t x = i; x < q; ++x) {
        if (p.pend_alive[x]) {
          pend_hit = x;
          break;
        }
      }
    }
    if (p.L.is_del(e)) {
      if (old_hit >= 0) {
        p.nbr[mt.x + old_hit] = u | kDead;
        if (old_hit < rr.bl) {
          atomicAdd(&p.dead[v], 1);
        } else {
          p.kill[q] = 1;  // a tail entry
        }
        structural = true;
      } else if (pend_hit >= 0) {
        p.pend_alive[pend_hit] = 0;
      }
    } else {
      const int64_t bj = p.L.local(e) / p.L.stride;
      if (old_hit >= 0 || pend_hit >= 0) {
        if (p.upsert) {
          for (int k = 0; k < K; ++k) {
            const int32_t wn = p.ins_w[bj * K + k];
            if (old_hit >= 0) p.w[k * p.slot_cap + mt.x + old_hit] = wn; else p.pend_w[k * p.stride + pend_hit] = wn;
          }
        }
      } else {
        p.pend_alive[q] = 1;
        for (int k = 0; k < K; ++k) p.pend_w[k * p.stride + q] = p.ins_w[bj * K + k];
        structural = true;
      }
    }
  }
  touch_row<kGrouped>(p, structural, i, v, &p.ctl->touched_in);
}

/// Both pairing passes of a simple graph in one launch: workgroups [0, split) the out-rows,
/// the rest the in-rows (their own replay, independent of the out-row pass).
__global__ void __launch_bounds__(kBlock) k_pairs_simple(out_pair_params po, in_pair_params pi, int split) {
  const int b = static_cast<int>(blockIdx.x);
  if (b < split) {
    out_pairs<kBlock, false>(po, b * int64_t{blockDim.x} + threadIdx.x);
  } else {
    in_pairs_simple<false>(pi, (b - split) * int64_t{blockDim.x} + threadIdx.x);
  }
}

struct merge_params {
  int2* meta;
  int32_t* cap;
  int32_t* base;
  int32_t* dead;
  int32_t* nbr;
  int32_t* w;
  int64_t slot_cap;
  int K;
  const u64* keys;
  int64_t N;
  int vbits;
  const int32_t* pend_alive;
  const int32_t* pend_prefix;
  const int32_t* kill_prefix;  ///< prefix of the tail entries each operation killed
  const int32_t* pend_w;
  const int4* touched;
  const int* touched_count;
  int32_t* row_a;  ///< the row's operations: keys[row_a[u], row_b[u])
  int32_t* row_b;
  int4* lane_rows;  ///< rows of the threads' list, two words each: see plan_rows
  int32_t* lists;        ///< the merge plan: kModes lists of rows, N + 1 entries each
  int* list_count;       ///< rows per list
  int32_t* stage_nbr;
  int32_t* stage_w;
  int64_t stage_cap;
  long long* stage_used;
  long long* tail;
  long long* garbage;
  unsigned long long* relocated;
  long long* need_reloc;
  long long* need_stage;
  int* error_bits;
  double headroom;
};

/// The merges of both stores in one launch: a workgroup's role and store by its place in the grid. The
/// stores share nothing that the merges write, the error bits aside, which they set atomically.
struct merge_roles {
  merge_params side[2];
  int groups[4];        ///< workgroups per role and store: first role's out-rows, in-rows, second role's out-rows, in-rows
  apply_control* gate;  ///< null, or where the first launch's workgroups find whether the merges fit (merges_fit)
};

struct merge_sides {
  merge_params side[2];
  int split;
};

/// Runs `body(p, block, blocks)` with this workgroup's store and its index and count among that
/// store's workgroups (one copy of the body: the store's parameters are selected, not branched on).
template <typename Body>
DYNG_DEV void for_side(const merge_sides& m, Body&& body) {
  const int b = static_cast<int>(blockIdx.x);
  const bool in = b >= m.split;
  const merge_params p = in ? m.side[1] : m.side[0];
  body(p, in ? b - m.split : b, in ? static_cast<int>(gridDim.x) - m.split : m.split);
}

constexpr int kTailsBlock = 256;   ///< threads of a workgroup that merges short tails (a thread's needs 162 registers)
constexpr int kMergeBlock = 1024;  ///< threads of a merge workgroup
constexpr int kMergeWaves = kMergeBlock / 64;
constexpr int kMergeSeg = 2048;    ///< operations of one row a workgroup stages in LDS
constexpr int kRegChunks = kMergeSmall / 64;  ///< a short tail held in registers, 64 entries per chunk
constexpr int kRegWeights = 2;                ///< weight columns a tail merge moves per pass
constexpr int kTailMin = 64;                  ///< a tail may always grow to this many entries
constexpr int kTailMax = 4096;                ///< and never past this (a workgroup's registers)
constexpr int kTailPerThread = kTailMax / kMergeBlock;
static_assert(kMergeSmall % 64 == 0, "short tails are whole chunks of 64");
static_assert(kTailMax % kMergeBlock == 0, "a long tail is whole slabs of a workgroup");

constexpr int kLaneTail = 32;  ///< a tail one thread merges in registers: at most this many entries
constexpr int kLaneOps = 8;    ///< and at most this many operations

/// How a touched row is merged: its tail rewritten by one thread (a short tail and a few
/// operations, the common case), by one wave or by a workgroup, or the whole row rewritten as one
/// base run.
enum merge_mode { kTailWave = 0, kTailBlock = 1, kFull = 2, kTailLane = 3, kModes = 4 };

DYNG_DEV int tail_limit(int base_len) { return min(kTailMax, max(kTailMin, base_len >> 3)); }
DYNG_DEV int dead_limit(int base_len) { return max(16, base_len >> 2); }
DYNG_DEV int grown_cap(int len, double headroom) { return len + static_cast<int>(ceil(len * headroom)) + 2; }

/// First index in [0, len) of an LDS array whose value is >= v (strict: > v when `upper`).
DYNG_DEV int lds_bound(const int32_t* a, int len, int32_t v, bool upper) {
  int lo = 0, hi = len;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (a[mid] < v || (upper && a[mid] == v)) lo = mid + 1; else hi = mid;
  }
  return lo;
}

/// The shape of a touched row's merge.
struct row_plan {
  int mode;
  int base_len, tail_len, new_tail;
  int alive_base, alive_tail, pending;
  int new_len;  ///< full merge: the rewritten row's length
};

/// What a row's plan is made from: its place, base run, capacity and dead base entries, and its
/// operations [a, b) with the pending entries and the killed tail entries among them.
struct row_facts {
  int2 mt;
  int32_t base, cap, dead;
  int32_t a, b, pending, killed;
};

DYNG_DEV row_plan plan_row(const row_facts& f) {
  row_plan r;
  r.base_len = f.base;
  r.tail_len = f.mt.y - r.base_len;
  r.pending = f.pending;
  r.alive_tail = r.tail_len - f.killed;
  r.alive_base = r.base_len - f.dead;
  r.new_tail = r.alive_tail + r.pending;
  r.new_len = r.alive_base + r.new_tail;
  const int nops = f.b - f.a;
  const bool tail_ok = r.new_tail <= tail_limit(r.base_len) && r.base_len + r.new_tail <= f.cap &&
                       f.dead <= dead_limit(r.base_len);
  if (tail_ok && r.tail_len <= kLaneTail && nops <= kLaneOps) {
    r.mode = kTailLane;
  } else if (tail_ok && r.tail_len <= kMergeSmall && nops <= 64) {
    r.mode = kTailWave;
  } else if (tail_ok && nops <= kMergeSeg) {
    r.mode = kTailBlock;
  } else {
    r.mode = kFull;
  }
  return r;
}

/// A row's facts as the pairing and the scans left them in memory.
DYNG_DEV row_facts read_facts(const merge_params& p, int32_t u, int32_t a, int32_t b) {
  row_facts f;
  f.mt = p.meta[u];
  f.base = p.base[u];
  f.cap = p.cap[u];
  f.dead = p.dead[u];
  f.a = a;
  f.b = b;
  f.pending = p.pend_prefix[b] - p.pend_prefix[a];
  f.killed = p.kill_prefix[b] - p.kill_prefix[a];
  return f;
}

/// Before the merges: each touched row's mode (appended to its list) and, for full merges, the
/// staging slots (its alive entries) and the tail slots (a row that outgrew its capacity), so the
/// host can compact or grow first and no row is refused. One row per thread; the lists are
/// appended per workgroup (one atomic per mode and workgroup: the list counters are single
/// addresses every workgroup hits).
constexpr int kPlanBlock = 1024;

/// Plan one row per thread (u < 0: none) and append it to its mode's list: a row for one thread with
/// all its merge needs (row, place, base length, tail length; first operation, operations), so that the
/// merge reads them in a row instead of five arrays by vertex (short-tail merges of 1,000,000 operations
/// on RMAT-23: 245 -> 210 us), the others by their number, their operations in row_a and row_b. Every thread of the
/// workgroup calls it. `touched`: where the row joins the touched rows (null: it is one already).
template <int kThreads>
DYNG_DEV void plan_rows(const merge_params& p, int32_t u, const row_facts& f, int* touched_count, int4* touched) {
  __shared__ int wave_offset[kThreads / 64][kModes + 1];
  __shared__ int base[kModes + 1];
  __shared__ long long part[kThreads / 64];
  const int lists = kModes + (touched != nullptr ? 1 : 0);
  const int w = threadIdx.x / 64;
  long long reloc = 0, stage = 0;
  int mode = -1;
  if (u >= 0) {
    const row_plan r = plan_row(f);
    mode = r.mode;
    if (r.mode == kFull) {
      stage = r.alive_base + r.alive_tail;
      if (r.new_len > f.cap) reloc = grown_cap(r.new_len, p.headroom);
    }
  }
  int rank = 0, row_rank = 0;  // among the wave's rows of the same mode, and among all its rows
#pragma unroll
  for (int m = 0; m <= kModes; ++m) {
    const u64 b = __ballot(m == kModes ? mode >= 0 : mode == m);
    if (m == kModes) {
      row_rank = __popcll(b & lanes_below());
    } else if (mode == m) {
      rank = __popcll(b & lanes_below());
    }
    if (lane() == 0) wave_offset[w][m] = __popcll(b);
  }
  __syncthreads();
  if (static_cast<int>(threadIdx.x) < lists) {
    const int m = threadIdx.x;
    int run = 0;
    for (int i = 0; i < kThreads / 64; ++i) {
      const int c = wave_offset[i][m];
      wave_offset[i][m] = run;
      run += c;
    }
    base[m] = run > 0 ? atomicAdd(m == kModes ? touched_count : &p.list_count[m], run) : 0;
  }
  __syncthreads();
  if (mode >= 0) {
    const int64_t place = base[mode] + wave_offset[w][mode] + rank;
    if (mode == kTailLane) {
      p.lane_rows[2 * place] = make_int4(u, f.mt.x, f.base, f.mt.y - f.base);
      p.lane_rows[2 * place + 1] = make_int4(f.a, f.b - f.a, 0, 0);
    } else {
      p.lists[mode * (p.N + 1) + place] = u;
      p.row_a[u] = f.a;
      p.row_b[u] = f.b;
    }
    if (touched != nullptr) touched[base[kModes] + wave_offset[w][kModes] + row_rank] = make_int4(u, f.a, f.b, 0);
  }
  if (__syncthreads_or(mode == kFull ? 1 : 0) == 0) return;  // the sums are zero
  reloc = block_reduce(reloc, part, op_sum{});
  stage = block_reduce(stage, part, op_sum{});
  if (threadIdx.x == 0) {
    if (reloc) atomicAdd(reinterpret_cast<unsigned long long*>(p.need_reloc), static_cast<unsigned long long>(reloc));
    if (stage) atomicAdd(reinterpret_cast<unsigned long long*>(p.need_stage), static_cast<unsigned long long>(stage));
  }
}

DYNG_DEV void merge_plan(const merge_params& p, int block) {
  const int count = *p.touched_count;
  const int t = block * kPlanBlock + threadIdx.x;
  row_facts f{};
  int32_t u = -1;
  if (t < count) {
    const int4 x = p.touched[t];
    u = x.x;
    f = read_facts(p, u, x.y >= 0 ? x.y : p.row_a[u], x.y >= 0 ? x.z : p.row_b[u]);
  }
  plan_rows<kPlanBlock>(p, u, f, nullptr, nullptr);
}

__global__ void __launch_bounds__(kPlanBlock) k_merge_plan(merge_sides m) {
  for_side(m, [](const merge_params& p, int block, int) { merge_plan(p, block); });
}

/// Slots a relocating merge leaves free at the arena's tail (the host's plan keeps the same).
constexpr long long kArenaMargin = 1024;

/// After a plan that the host does not read back: whether the merges fit as planned (the arenas'
/// free tails take the relocations, the staging arena both stores' full merges) and nothing came
/// first that stops them.
DYNG_DEV bool merges_fit(const apply_control* c, long long slot_cap_out, long long slot_cap_in, long long stage_cap) {
  return c->miss == 0 && c->error_bits == 0 && c->need_reloc_out + kArenaMargin <= slot_cap_out - c->tail_out &&
         c->need_reloc_in + kArenaMargin <= slot_cap_in - c->tail_in &&
         c->need_stage_out + c->need_stage_in <= stage_cap;
}

// ---------------------------------------------------------------------------------------------
// The grouped apply: operations scattered into groups of whole rows, then everything up to the merge
// plan of a group's rows in one workgroup
// ---------------------------------------------------------------------------------------------

/// A batch's operations need not be sorted as a whole: the pairing needs each (u, v) together in
/// batch order, the merges each row's operations together by neighbour. So the rows are hashed into
/// groups of 32 to 512 operations per direction (an odd multiplier modulo 2^vbits is a
/// bijection, its top bits the group), one launch scatters the operations into their groups, and in
/// the next one workgroup per group sorts its operations in LDS, pairs them with their rows, scans
/// their flags and plans its rows' merges. That replaces a device-wide sort (75 us of block sort and
/// eight merge passes for a batch of 100,000 on RMAT-22, 269 us of radix passes for 1,000,000 on
/// RMAT-23), the untagging, the pairing, two scan launches and the plan: two launches for ten to
/// seventeen, nothing between them through memory but the operations.
constexpr int kGroupBlock = 256;
/// Least operations of a group and direction on average before there are twice as many groups, by how
/// many there are: few while processors are idle (2^7 groups per direction give every one of the 256 a
/// workgroup), more up to the workgroups it holds at once (2^9), and beyond that what the front's
/// reservations and the per-group work favour. So the groups of 4,096 to 32,767 operations hold 32 to 256
/// each, of 65,536 to 262,143 operations 128 to 512, of more 256 to 512 (1,024 at 2^22 operations). 2,000 arcs of an undirected 64 K graph: 25 us with 32 each, 43 with
/// 128; 100,000 operations on RMAT-22: 103 us with 128, 110 with 256; 1,000,000 on RMAT-23: 515 us with
/// 256, 550 to 590 with 128.
constexpr int kGroupBitsFew = 7, kGroupOpsFew = 32;
constexpr int kGroupBitsSome = 9, kGroupOpsSome = 128;
constexpr int kGroupOps = 256;
constexpr int64_t kGroupMost = int64_t{1} << 22;  ///< operations of a batch (1024 per group)
constexpr int kGroupCap = 4096;   ///< most a group takes; one row with more operations sends the batch to the sort
constexpr int kGroupLds = 1024;   ///< a group with fewer operations keeps them in LDS (8 KB of segments, 24 KB of the rest)
constexpr int kGroupPause = 15;   ///< batches sorted device-wide after one that a group could not take
constexpr int kGroupBits = 12;    ///< at most 2^12 groups per direction
constexpr uint32_t kGroupHash = 0x9E3779B1u;

/// Why the grouped apply did nothing (apply_control::miss).
enum { kMissFull = 1 };

/// What the control block starts an apply with, and the group counters to clear. A launch with these
/// in its arguments in place of a copy from host memory: one launch clears both.
struct begin_params {
  long long tail_out, tail_in;
  long long col_max[max_weights];
  int* counts;
  int num_counts;
};
__global__ void __launch_bounds__(1024) k_begin(apply_control* c, begin_params b) {
  static_assert(sizeof(apply_control) % sizeof(int) == 0);
  for (int i = threadIdx.x; i < static_cast<int>(sizeof(apply_control) / sizeof(int)); i += blockDim.x) {
    reinterpret_cast<int*>(c)[i] = 0;
  }
  for (int i = threadIdx.x; i < b.num_counts; i += blockDim.x) b.counts[i] = 0;
  __syncthreads();  // the words are cleared
  if (threadIdx.x < max_weights) c->col_max[threadIdx.x] = b.col_max[threadIdx.x];
  if (threadIdx.x == 0) {
    c->tail_out = b.tail_out;
    c->tail_in = b.tail_in;
    c->first_error = kNoError;
  }
}

struct front_params {
  op_layout L;
  const int32_t *ins_src, *ins_dst, *del_src, *del_dst;
  int directed, drop_self_loops;
  int64_t n_after;
  int vbits, ebits, lb, K;
  int groups;
  int room;      ///< operations a group has room for
  u64* entries;  ///< `room` per group: out-row groups, then in-row groups
  int* counts;
  int32_t *e_del_src, *e_del_dst, *e_ins_src, *e_ins_dst;
  uint8_t* e_inc;
  int32_t* e_fw;
  apply_control* ctl;
};

/// One arc of the batch: operation e of the layout. False when it is dropped (a self-loop, the
/// second arc of a directed graph, a deletion naming a vertex that does not exist).
struct front_op {
  bool del, dropped, ignored;
  int64_t loc;
  int32_t u, v;
};
DYNG_DEV bool front_decode(const front_params& f, int64_t e, front_op& o) {
  o.del = f.L.is_del(e);
  o.loc = f.L.local(e);
  const int64_t j = o.loc / f.L.stride;
  const int r = static_cast<int>(o.loc % f.L.stride);
  const int32_t u0 = o.del ? f.del_src[j] : f.ins_src[j];
  const int32_t v0 = o.del ? f.del_dst[j] : f.ins_dst[j];
  o.u = r ? v0 : u0;
  o.v = r ? u0 : v0;
  bool valid = !(r == 1 && (f.directed || u0 == v0));
  o.dropped = valid && u0 == v0 && f.drop_self_loops;
  valid = valid && !o.dropped;
  o.ignored = valid && o.del && (o.u >= f.n_after || o.v >= f.n_after);
  return valid && !o.ignored;
}

/// The effective operation lists, and each operation's out- and in-key in its group. A workgroup
/// counts its operations per group in LDS and reserves their places with one atomic per group it
/// touches (the counters of all groups share a few cache lines). kOps operations per thread.
template <int kOps>
__global__ void __launch_bounds__(1024) k_group_front(front_params f) {
  __shared__ int hist[2 << kGroupBits];
  const int all = 2 * f.groups;
  for (int b = threadIdx.x; b < all; b += blockDim.x) hist[b] = 0;
  __syncthreads();
  const int64_t total = (f.L.num_first + f.L.num_second) * f.L.stride;
  const int64_t e0 = (int64_t{blockIdx.x} * kOps) * blockDim.x + threadIdx.x;
  const uint32_t mask = static_cast<uint32_t>((u64{1} << f.vbits) - 1);
  const int low = f.vbits - f.lb;  // bits of a hashed row below its group's
  int rank[2][kOps];
  unsigned long long dropped = 0, ignored = 0;
#pragma unroll
  for (int j = 0; j < kOps; ++j) {
    const int64_t e = e0 + int64_t{j} * blockDim.x;
    front_op o{};
    const bool valid = e < total && front_decode(f, e, o);
    dropped += __popcll(__ballot(e < total && o.dropped));
    ignored += __popcll(__ballot(e < total && o.ignored));
    if (e < total) {
      if (o.del) {
        f.e_del_src[o.loc] = valid ? o.u : -1;
        f.e_del_dst[o.loc] = valid ? o.v : -1;
      } else {
        f.e_ins_src[o.loc] = valid ? o.u : -1;
        f.e_ins_dst[o.loc] = valid ? o.v : -1;
        for (int k = 0; k < f.K; ++k) f.e_inc[o.loc * f.K + k] = 0;
        if (f.e_fw != nullptr) {
          for (int k = 0; k < f.K; ++k) f.e_fw[o.loc * f.K + k] = -1;
        }
      }
    }
    rank[0][j] = rank[1][j] = -1;
    if (valid) {
      const uint32_t hu = (static_cast<uint32_t>(o.u) * kGroupHash) & mask;
      const uint32_t hv = (static_cast<uint32_t>(o.v) * kGroupHash) & mask;
      rank[0][j] = atomicAdd(&hist[hu >> low], 1);
      rank[1][j] = atomicAdd(&hist[f.groups + static_cast<int>(hv >> low)], 1);
    }
  }
  if (lane() == 0) {
    if (dropped) atomicAdd(&f.ctl->dropped_self_loops, dropped);
    if (ignored) atomicAdd(&f.ctl->ignored_deletions, ignored);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < all; b += blockDim.x) {
    if (hist[b] > 0) {
      const int mine = hist[b];
      hist[b] = atomicAdd(&f.counts[b], mine);
      if (hist[b] + mine > f.room) atomicOr(&f.ctl->miss, kMissFull);
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kOps; ++j) {
    if (rank[0][j] < 0) continue;
    const int64_t e = e0 + int64_t{j} * blockDim.x;
    front_op o;
    (void)front_decode(f, e, o);
    const uint32_t hu = (static_cast<uint32_t>(o.u) * kGroupHash) & mask;
    const uint32_t hv = (static_cast<uint32_t>(o.v) * kGroupHash) & mask;
    const u64 below = (u64{1} << low) - 1;
    const int gu = static_cast<int>(hu >> low), gv = f.groups + static_cast<int>(hv >> low);
    const int at_u = hist[gu] + rank[0][j], at_v = hist[gv] + rank[1][j];
    if (at_u < f.room) {
      f.entries[int64_t{gu} * f.room + at_u] =
          ((((hu & below) << f.vbits) | static_cast<u64>(o.v)) << f.ebits) | static_cast<u64>(e);
    }
    if (at_v < f.room) {
      f.entries[int64_t{gv} * f.room + at_v] =
          ((((hv & below) << f.vbits) | static_cast<u64>(o.u)) << f.ebits) | static_cast<u64>(e);
    }
  }
}

/// Entries below x in 64 sorted words of LDS.
DYNG_DEV int segment_rank(const u64* S, u64 x) {
  int at = 0;
#pragma unroll
  for (int step = 32; step > 0; step >>= 1) at += S[at + step - 1] < x ? step : 0;
  return at + (S[at] < x ? 1 : 0);
}

/// Sort the `count` words of src (distinct, below 2^63): place(rank, word) for each. Every wave
/// ranks 64 words at a time among themselves (each lane counts the smaller ones, broadcast from
/// register to register) and leaves them sorted in S; then a word's rank is the sum of its ranks in
/// all the sorted segments, searched independently of each other. 256 words: about 1 us, where a bitonic
/// sort's 36 dependent LDS steps take 9. Every thread of the workgroup calls it.
template <class Place>
DYNG_DEV void group_sort(const u64* src, int count, u64* S, Place place) {
  const int segments = (count + 63) / 64;
  const int wave = uniform(static_cast<int>(threadIdx.x) / 64);
  for (int s = wave; s < segments; s += kGroupBlock / 64) {
    const int i = s * 64 + lane();
    const u64 x = i < count ? src[i] : ~u64{0} - 63 + lane();
    const int lo = static_cast<int>(x), hi = static_cast<int>(x >> 32);
    int rank = 0;
#pragma unroll 8
    for (int j = 0; j < 64; ++j) {
      const u64 y = (static_cast<u64>(static_cast<uint32_t>(__builtin_amdgcn_readlane(hi, j))) << 32) |
                    static_cast<uint32_t>(__builtin_amdgcn_readlane(lo, j));
      rank += y < x ? 1 : 0;
    }
    S[s * 64 + rank] = x;
  }
  __syncthreads();
  for (int s = wave; s < segments; s += kGroupBlock / 64) {
    const u64 x = S[s * 64 + lane()];
    int rank = lane();
    if (segments > 1) {
      rank = 0;
#pragma unroll 4
      for (int t = 0; t < segments; ++t) rank += segment_rank(S + t * 64, x);
    }
    if (s * 64 + lane() < count) place(rank, x);  // the fillers sort behind the last segment's words
  }
}

struct group_params {
  const u64* entries;
  const int* counts;
  int groups, vbits, ebits, lb, room;
  uint32_t inverse;  ///< of kGroupHash modulo 2^32
  u64* keys;         ///< sorted operations: out-rows [0, P), in-rows [P, 2P)
  uint32_t* vals;
  int64_t P;         ///< operations plus one place per group
  out_pair_params out;
  in_pair_params in;
  merge_params merge_out, merge_in;
  int32_t *pend_prefix_out, *kill_prefix_out, *pend_prefix_in, *kill_prefix_in;
  apply_control* ctl;
};

enum { kGroupsBoth = 0, kGroupsOut = 1, kGroupsIn = 2 };

/// One group per workgroup: its operations sorted by (row, neighbour, batch order), paired with
/// their rows, their flags scanned (a row's operations are in one group, and only differences within
/// a row are used), and its rows' merges planned. kGroupsBoth: a simple graph's out-rows and in-rows
/// side by side; else one direction (with parallel edges the in-row pass reads what the out-row pass
/// recorded). What bounds it is the chain of dependent reads, so the sorted operations, their flags and
/// the scans stay in LDS (a group of more than kGroupLds keeps them in memory), a row's plan takes
/// what it needs of them from there, and its operations are found there and not by vertex in memory.
template <int kWhich>
__global__ void __launch_bounds__(kGroupBlock, 4) k_group_pairs(group_params g) {
  __shared__ u64 S[kGroupCap];
  __shared__ int part[kGroupBlock / 64];
  __shared__ int3 sums[kGroupBlock / 64];
  const int tid = static_cast<int>(threadIdx.x);
  const bool in = kWhich == kGroupsIn || (kWhich == kGroupsBoth && static_cast<int>(blockIdx.x) >= g.groups);
  const int q = static_cast<int>(blockIdx.x) - (kWhich == kGroupsBoth && in ? g.groups : 0);
  const int* counts = g.counts + (in ? g.groups : 0);
  const int missed = g.ctl->miss, here = counts[q];
  int before = 0;
  for (int b = tid; b < q; b += kGroupBlock) before += counts[b];
  const int count = uniform(here);
  if (missed != 0 || count == 0) return;  // uniform
  before = wave_scan(before);
  if (lane() == 63) part[tid / 64] = before;
  const bool lds = count < kGroupLds;
  const u64* src = g.entries + int64_t{(in ? g.groups : 0) + q} * g.room;
  const int low = g.vbits - g.lb;
  const u64 vmask = (u64{1} << g.vbits) - 1, emask = (u64{1} << g.ebits) - 1;
  int64_t at = q;
  u64* keys = S + kGroupLds;
  uint32_t* vals = reinterpret_cast<uint32_t*>(S + 2 * kGroupLds);
  if (!lds) {
    __syncthreads();
    for (int w = 0; w < kGroupBlock / 64; ++w) at += uniform(part[w]);
    keys = g.keys + (in ? g.P : 0) + at;
    vals = g.vals + (in ? g.P : 0) + at;
  }
  group_sort(src, count, S, [&](int i, u64 x) {
    const uint32_t h = static_cast<uint32_t>((static_cast<u64>(q) << low) | (x >> (g.vbits + g.ebits)));
    const u64 row = (h * g.inverse) & static_cast<uint32_t>(vmask);
    keys[i] = (row << g.vbits) | ((x >> g.ebits) & vmask);
    vals[i] = static_cast<uint32_t>(x & emask);
  });
  if (lds) {
    for (int w = 0; w < kGroupBlock / 64; ++w) at += uniform(part[w]);  // behind group_sort's barrier
  }
  // per operation: pending, killed tail entry, changed row; scanned in place, and the killed ones
  // where the sort's words were
  int32_t* const out_alive = (in ? g.in.pend_alive : g.out.pend_alive) + at;
  int32_t* const out_pend = (in ? g.pend_prefix_in : g.pend_prefix_out) + at;
  int32_t* const out_kill = (in ? g.kill_prefix_in : g.kill_prefix_out) + at;
  int32_t* const ints = reinterpret_cast<int32_t*>(S + 2 * kGroupLds + kGroupLds / 2);
  int32_t* const alive = lds ? ints : out_alive;
  int32_t* const killed = lds ? ints + kGroupLds : (in ? g.in.kill : g.out.kill) + at;  // then changed rows before
  int32_t* const flag = lds ? ints + 2 * kGroupLds : out_pend;                           // then pending before
  int32_t* const killed_before = lds ? reinterpret_cast<int32_t*>(S) : out_kill;
  for (int i = tid; i < count; i += kGroupBlock) flag[i] = 0;
  __syncthreads();  // the sorted operations and the cleared flags are there for the whole workgroup
  if (!in) {
    out_pair_params p = g.out;
    p.keys = keys;
    p.vals = vals;
    p.N = count;
    p.pend_alive = alive;
    p.kill = killed;
    p.flag = flag;
    p.pend_w += at;
    for (int t = 0; t < count; t += kGroupBlock) {
      out_pairs<kGroupBlock, true>(p, t + tid);
      __syncthreads();  // its sums are read
    }
  } else {
    in_pair_params p = g.in;
    p.keys = keys;
    p.vals = vals;
    p.N = count;
    p.pend_alive = alive;
    p.kill = killed;
    p.flag = flag;
    p.pend_w += at;
    for (int t = 0; t < count; t += kGroupBlock) {
      if (kWhich == kGroupsIn) {
        in_pairs<true>(p, t + tid);
      } else {
        in_pairs_simple<true>(p, t + tid);
      }
    }
  }
  __syncthreads();  // the flags are written
  int3 carry = make_int3(0, 0, 0);
  for (int t = 0; t < count; t += kGroupBlock) {
    const int i = t + tid;
    const int xp = i < count ? alive[i] : 0, xk = i < count ? killed[i] : 0, xf = i < count ? flag[i] : 0;
    const int sp = wave_scan(xp), sk = wave_scan(xk), sf = wave_scan(xf);
    __syncthreads();
    if (lane() == 63) sums[tid / 64] = make_int3(sp, sk, sf);
    __syncthreads();
    int3 b = carry;
    for (int w = 0; w < kGroupBlock / 64; ++w) {
      const int3 x = sums[w];
      if (w < tid / 64) {
        b.x += x.x;
        b.y += x.y;
        b.z += x.z;
      }
      carry.x += x.x;
      carry.y += x.y;
      carry.z += x.z;
    }
    if (i < count) {
      flag[i] = b.x + sp - xp;
      killed_before[i] = b.y + sk - xk;
      killed[i] = b.z + sf - xf;
      if (lds) {
        g.keys[(in ? g.P : 0) + at + i] = keys[i];
        out_alive[i] = xp;
        out_pend[i] = b.x + sp - xp;
        out_kill[i] = b.y + sk - xk;
      }
    }
  }
  if (tid == 0) {
    flag[count] = out_pend[count] = carry.x;
    killed_before[count] = out_kill[count] = carry.y;
    killed[count] = carry.z;
  }
  __syncthreads();
  const merge_params& m = in ? g.merge_in : g.merge_out;
  for (int t = 0; t < count; t += kGroupBlock) {
    const int i = t + tid;
    int32_t u = -1;
    row_facts f{};
    if (i < count) {
      const u64 r = keys[i] >> g.vbits;
      if (i == 0 || keys[i - 1] >> g.vbits != r) {
        int b = i + 1;  // the row's operations end at b
        if (b < count && keys[b] >> g.vbits == r) {
          int end = count;
          ++b;
          while (b < end) {
            const int mid = (b + end) >> 1;
            if (keys[mid] >> g.vbits == r) b = mid + 1; else end = mid;
          }
        }
        if (killed[b] != killed[i]) {
          u = static_cast<int32_t>(r);
          f.mt = m.meta[u];
          f.base = m.base[u];
          f.cap = m.cap[u];
          f.dead = ld(&m.dead[u]);  // counted by device-scope additions of this launch
          f.a = static_cast<int32_t>(at + i);
          f.b = static_cast<int32_t>(at + b);
          f.pending = flag[b] - flag[i];
          f.killed = killed_before[b] - killed_before[i];
        }
      }
    }
    plan_rows<kGroupBlock>(m, u, f, in ? &g.ctl->touched_in : &g.ctl->touched_out, in ? g.in.touched : g.out.touched);
    __syncthreads();  // plan_rows' arrays are free again
  }
}

/// One thread per row whose tail holds at most kLaneTail entries and that has at most kLaneOps
/// operations: the tail and the operations are read into registers with independent loads, every
/// entry's place is counted with static indices (an alive entry: the alive entries before it plus
/// the pending entries with a smaller neighbour; a pending entry: the alive entries up to its
/// neighbour plus the pending entries before it), then each is stored at its place. The weights
/// move KW columns per pass, each pass reading its columns before writing them (KW = 1 for a
/// single weight column: 162 VGPRs instead of 186, three waves per SIMD instead of two). Old
/// entries come first among equal neighbours, as in the wave merge below.
template <int KW, int T, int O>
DYNG_DEV int merge_lane(const merge_params& p, int64_t at, int tl, int64_t a, int nops) {
  const u64 mask = (1ULL << p.vbits) - 1;
  const int K = p.K;
  int32_t x[T];
#pragma unroll
  for (int j = 0; j < T; ++j) x[j] = j < tl ? p.nbr[at + j] : -1;
  int32_t ov[O];
  bool pend[O];
#pragma unroll
  for (int j = 0; j < O; ++j) {
    pend[j] = j < nops && p.pend_alive[a + j] != 0;
    ov[j] = pend[j] ? static_cast<int32_t>(p.keys[a + j] & mask) : 0;
  }
  int alive = 0, pending = 0;
  for (int k0 = 0; k0 == 0 || k0 < K; k0 += KW) {
    int32_t wr[KW][T];
    int32_t ow[KW][O];
#pragma unroll
    for (int j = 0; j < T; ++j) {
#pragma unroll
      for (int k = 0; k < KW; ++k) {
        wr[k][j] = (j < tl && k0 + k < K) ? p.w[(k0 + k) * p.slot_cap + at + j] : 0;
      }
    }
#pragma unroll
    for (int j = 0; j < O; ++j) {
#pragma unroll
      for (int k = 0; k < KW; ++k) ow[k][j] = (pend[j] && k0 + k < K) ? p.pend_w[(k0 + k) * p.N + a + j] : 0;
    }
    // alive entries, at their places (the tail is sorted, dead entries carry the sign bit)
    alive = 0;
#pragma unroll
    for (int i = 0; i < T; ++i) {
      if (x[i] >= 0) {
        int pos = alive;
#pragma unroll
        for (int j = 0; j < O; ++j) pos += (pend[j] && ov[j] < x[i]) ? 1 : 0;
        if (k0 == 0) p.nbr[at + pos] = x[i];
#pragma unroll
        for (int k = 0; k < KW; ++k) {
          if (k0 + k < K) p.w[(k0 + k) * p.slot_cap + at + pos] = wr[k][i];
        }
        ++alive;
      }
    }
    // pending entries (the operations are sorted by neighbour, then batch order)
    pending = 0;
#pragma unroll
    for (int j = 0; j < O; ++j) {
      if (pend[j]) {
        int pos = pending;
#pragma unroll
        for (int i = 0; i < T; ++i) pos += (x[i] >= 0 && x[i] <= ov[j]) ? 1 : 0;
        if (k0 == 0) p.nbr[at + pos] = ov[j];
#pragma unroll
        for (int k = 0; k < KW; ++k) {
          if (k0 + k < K) p.w[(k0 + k) * p.slot_cap + at + pos] = ow[k][j];
        }
        ++pending;
      }
    }
  }
  return alive + pending;
}

/// The wave's longest tail and most operations choose how many entries and operations are counted out:
/// the full 32 x 8 is 1,500 instructions, which a small batch's few waves wait for (10 operations:
/// 11 us, 3.4 with 8 x 2; a large batch waits for memory either way).
template <int KW>
DYNG_DEV void tail_lane(const merge_params& p, int block, int blocks) {
  const int count = p.list_count[kTailLane];
  for (int t = block * blockDim.x + threadIdx.x; t < count; t += blocks * blockDim.x) {
    const int4 row = p.lane_rows[2 * int64_t{t}], ops = p.lane_rows[2 * int64_t{t} + 1];
    const int64_t a = ops.x;
    const int nops = ops.y;
    const int bl = row.z;
    const int tl = row.w;
    const int64_t at = row.y + int64_t{bl};  // the tail's first slot
    int len;
    if (!__any(tl > kLaneTail / 4 || nops > kLaneOps / 4)) {
      len = merge_lane<KW, kLaneTail / 4, kLaneOps / 4>(p, at, tl, a, nops);
    } else if (!__any(tl > kLaneTail / 2 || nops > kLaneOps / 2)) {
      len = merge_lane<KW, kLaneTail / 2, kLaneOps / 2>(p, at, tl, a, nops);
    } else {
      len = merge_lane<KW, kLaneTail, kLaneOps>(p, at, tl, a, nops);
    }
    p.meta[row.x] = make_int2(row.y, bl + len);
  }
}

/// One wave per row whose tail is short (at most kMergeSmall entries, 64 operations): the tail
/// is read into registers and the merged tail (its alive entries and the pending ones, by
/// neighbour id, old entries first among equal ones) written back in place. An alive entry's
/// place is the alive entries before it plus the pending entries with a smaller neighbour (the
/// operations one per lane); a pending entry's place is the alive entries up to its neighbour
/// (ballots over the registers) plus the pending entries before it.
DYNG_DEV void tail_wave(const merge_params& p, int block, int blocks) {
  const int count = p.list_count[kTailWave];
  const int32_t* list = p.lists + kTailWave * (p.N + 1);
  const u64 mask = (1ULL << p.vbits) - 1;
  const int wave = static_cast<int>((block * int64_t{blockDim.x} + threadIdx.x) / 64);
  const int waves = static_cast<int>((int64_t{blocks} * blockDim.x) / 64);
  const int K = p.K;
  for (int t = wave; t < count; t += waves) {
    const int32_t u = list[t];
    const int2 mt = p.meta[u];
    const int64_t a = p.row_a[u], b = p.row_b[u];
    const int nops = static_cast<int>(b - a);
    const int bl = p.base[u];
    const int tl = mt.y - bl;
    const int64_t at = mt.x + int64_t{bl};  // the tail's first slot
    int32_t x[kRegChunks];
#pragma unroll
    for (int c = 0; c < kRegChunks; ++c) {
      const int jx = c * 64 + lane();
      x[c] = jx < tl ? p.nbr[at + jx] : -1;
    }
    const bool has = lane() < nops;
    const int32_t ov = has ? static_cast<int32_t>(p.keys[a + lane()] & mask) : INT32_MAX;
    const bool opend = has && p.pend_alive[a + lane()] != 0;
    int before[kRegChunks];
#pragma unroll
    for (int c = 0; c < kRegChunks; ++c) before[c] = 0;
    const u64 pend_mask = __ballot(opend);
    for (int j = 0; j < nops; ++j) {
      if (!((pend_mask >> j) & 1)) continue;  // uniform
      const int32_t vj = __shfl(ov, j);
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c) before[c] += (x[c] >= 0 && vj < x[c]) ? 1 : 0;
    }
    // pending entries: their places, computed before any store
    int64_t ppos = -1;
    for (int j = 0; j < nops; ++j) {
      if (!((pend_mask >> j) & 1)) continue;  // uniform
      const int32_t vj = __shfl(ov, j);
      int y = 0;
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c) y += __popcll(__ballot(x[c] >= 0 && x[c] <= vj));
      if (lane() == j) ppos = at + y + __popcll(pend_mask & ((1ULL << j) - 1));
    }
    // the stores, kRegWeights weight columns per pass: every lane of the wave reads its entries'
    // old weights of the pass's columns before any lane writes them
    int carry = 0;
    for (int k0 = 0; k0 == 0 || k0 < K; k0 += kRegWeights) {
      int32_t wr[kRegWeights][kRegChunks];
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c) {
        const int jx = c * 64 + lane();
#pragma unroll
        for (int k = 0; k < kRegWeights; ++k) {
          wr[k][c] = (jx < tl && k0 + k < K) ? p.w[(k0 + k) * p.slot_cap + at + jx] : 0;
        }
      }
      carry = 0;
#pragma unroll
      for (int c = 0; c < kRegChunks; ++c) {
        const bool alive = x[c] >= 0;
        const u64 ballot = __ballot(alive);
        if (alive) {
          const int64_t pos = at + carry + __popcll(ballot & lanes_below()) + before[c];
          if (k0 == 0) p.nbr[pos] = x[c];
#pragma unroll
          for (int k = 0; k < kRegWeights; ++k) {
            if (k0 + k < K) p.w[(k0 + k) * p.slot_cap + pos] = wr[k][c];
          }
        }
        carry += __popcll(ballot);
      }
      if (opend) {
        if (k0 == 0) p.nbr[ppos] = ov;
#pragma unroll
        for (int k = 0; k < kRegWeights; ++k) {
          if (k0 + k < K) p.w[(k0 + k) * p.slot_cap + ppos] = p.pend_w[(k0 + k) * p.N + a + lane()];
        }
      }
    }
    if (lane() == 0) p.meta[u] = make_int2(mt.x, bl + carry + __popcll(pend_mask));
  }
}

/// The tails short enough for a wave or a thread each, of both stores. Without a plan read back by the
/// host every workgroup looks for itself whether the merges fit; if not, nothing is merged and the
/// first workgroup says so (`hold`) to the launch and any engine run queued behind. One launch where
/// three (the check, the lanes', the waves') took 10 us for a batch of 10.
template <int KW>
__global__ void __launch_bounds__(kTailsBlock) k_tails(merge_roles m) {
  if (m.gate != nullptr && !merges_fit(m.gate, m.side[0].slot_cap, m.side[1].slot_cap, m.side[0].stage_cap)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) m.gate->hold = 1;
    return;
  }
  int b = static_cast<int>(blockIdx.x), role = 0;
  while (role < 3 && b >= m.groups[role]) b -= m.groups[role++];
  const merge_params& p = m.side[role & 1];
  if (role < 2) tail_wave(p, b, m.groups[role]); else tail_lane<KW>(p, b, m.groups[role]);
}

/// One workgroup per row whose tail needs more than a wave (up to kTailMax entries, kMergeSeg
/// operations): the tail in registers (kTailPerThread per thread), the operations and the
/// alive tail in LDS, the merged tail written back in place. The LDS arrays are the function's
/// own (one set per workgroup, whichever store it merges).
DYNG_DEV void tail_block(const merge_params& p, int block, int blocks) {
  __shared__ int32_t s_v[kMergeSeg];       // neighbour of each operation
  __shared__ int32_t s_pp[kMergeSeg + 1];  // pending entries before each operation
  __shared__ int32_t s_t[kTailMax];        // the alive tail entries, compacted
  __shared__ int s_tot[kTailPerThread * kMergeWaves + 1];
  const int count = p.list_count[kTailBlock];
  const int32_t* list = p.lists + kTailBlock * (p.N + 1);
  const u64 mask = (1ULL << p.vbits) - 1;
  const int tid = static_cast<int>(threadIdx.x);
  const int wid = tid / 64;
  const int K = p.K;
  for (int t = block; t < count; t += blocks) {
    const int32_t u = list[t];
    const int2 mt = p.meta[u];
    const int64_t a = p.row_a[u], b = p.row_b[u];
    const int nops = static_cast<int>(b - a);
    const int bl = p.base[u];
    const int tl = mt.y - bl;
    const int64_t at = mt.x + int64_t{bl};
    const int pa = p.pend_prefix[a];
    for (int j = tid; j < nops; j += kMergeBlock) {
      s_v[j] = static_cast<int32_t>(p.keys[a + j] & mask);
      s_pp[j] = p.pend_prefix[a + j] - pa;
    }
    if (tid == 0) s_pp[nops] = p.pend_prefix[b] - pa;
    int32_t x[kTailPerThread];
    int32_t wr[kRegWeights][kTailPerThread];
    int rank[kTailPerThread];
#pragma unroll
    for (int e = 0; e < kTailPerThread; ++e) {
      const int jx = e * kMergeBlock + tid;
      const bool in = jx < tl;
      x[e] = in ? p.nbr[at + jx] : -1;
#pragma unroll
      for (int k = 0; k < kRegWeights; ++k) wr[k][e] = (in && k < K) ? p.w[k * p.slot_cap + at + jx] : 0;
      const u64 ballot = __ballot(x[e] >= 0);
      rank[e] = __popcll(ballot & lanes_below());
      if (lane() == 0) s_tot[e * kMergeWaves + wid] = __popcll(ballot);
    }
    __syncthreads();
    if (tid == 0) {
      int run = 0;
      for (int i = 0; i < kTailPerThread * kMergeWaves; ++i) {
        const int c = s_tot[i];
        s_tot[i] = run;
        run += c;
      }
      s_tot[kTailPerThread * kMergeWaves] = run;
    }
    __syncthreads();
    const int alive_tail = s_tot[kTailPerThread * kMergeWaves];
    int apos[kTailPerThread];
#pragma unroll
    for (int e = 0; e < kTailPerThread; ++e) {
      apos[e] = s_tot[e * kMergeWaves + wid] + rank[e];
      if (x[e] >= 0) s_t[apos[e]] = x[e];
    }
    __syncthreads();
    // the stores, kRegWeights weight columns per pass (the first pass's weights were read with
    // the tail; a later pass reads its columns, then waits for the whole workgroup before writing)
    for (int k0 = 0; k0 == 0 || k0 < K; k0 += kRegWeights) {
      if (k0 > 0) {
#pragma unroll
        for (int e = 0; e < kTailPerThread; ++e) {
          const int jx = e * kMergeBlock + tid;
#pragma unroll
          for (int k = 0; k < kRegWeights; ++k) {
            wr[k][e] = (jx < tl && k0 + k < K) ? p.w[(k0 + k) * p.slot_cap + at + jx] : 0;
          }
        }
        __syncthreads();
      }
      // pending entries: the alive tail entries up to their neighbour, the pending ones before them
      for (int j = tid; j < nops; j += kMergeBlock) {
        if (s_pp[j + 1] == s_pp[j]) continue;  // not pending
        const int32_t v = s_v[j];
        const int64_t pos = at + lds_bound(s_t, alive_tail, v, true) + s_pp[j];
        if (k0 == 0) p.nbr[pos] = v;
        for (int k = 0; k < kRegWeights; ++k) {
          if (k0 + k < K) p.w[(k0 + k) * p.slot_cap + pos] = p.pend_w[(k0 + k) * p.N + a + j];
        }
      }
#pragma unroll
      for (int e = 0; e < kTailPerThread; ++e) {
        if (x[e] < 0) continue;
        const int64_t pos = at + apos[e] + s_pp[lds_bound(s_v, nops, x[e], false)];
        if (k0 == 0) p.nbr[pos] = x[e];
#pragma unroll
        for (int k = 0; k < kRegWeights; ++k) {
          if (k0 + k < K) p.w[(k0 + k) * p.slot_cap + pos] = wr[k][e];
        }
      }
    }
    if (tid == 0) p.meta[u] = make_int2(mt.x, bl + alive_tail + s_pp[nops]);
    __syncthreads();
  }
}

/// Count of the entries of a sorted run in global memory that are < v (or <= v when `upper`).
DYNG_DEV int global_bound(const int32_t* a, int len, int32_t v, bool upper) {
  int lo = 0, hi = len;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    const int32_t x = a[mid];
    if (x < v || (upper && x == v)) lo = mid + 1; else hi = mid;
  }
  return lo;
}

/// Compact the alive entries of [src, src + len) to dst (a workgroup; returns the count).
DYNG_DEV int compact_alive(const merge_params& p, int64_t src, int len, int64_t dst, int* s_tot) {
  const int tid = static_cast<int>(threadIdx.x);
  const int wid = tid / 64;
  int carry = 0;
  for (int base = 0; base < len; base += kMergeBlock) {
    const int jx = base + tid;
    const int32_t x = jx < len ? p.nbr[src + jx] : -1;
    const u64 ballot = __ballot(x >= 0);
    if (lane() == 0) s_tot[wid] = __popcll(ballot);
    __syncthreads();
    int before = 0, total = 0;
    for (int q = 0; q < kMergeWaves; ++q) {
      before += q < wid ? s_tot[q] : 0;
      total += s_tot[q];
    }
    if (x >= 0) {
      const int64_t pos = dst + carry + before + __popcll(ballot & lanes_below());
      p.stage_nbr[pos] = x;
      for (int k = 0; k < p.K; ++k) p.stage_w[k * p.stage_cap + pos] = p.w[k * p.slot_cap + src + jx];
    }
    carry += total;
    __syncthreads();
  }
  return carry;
}

/// One workgroup per row rewritten whole, staging from `stage_from` on (its tail or dead entries
/// outgrew their limits, or the row its capacity): the alive base (A) and the alive tail (B) are compacted into the staging
/// arena, then A, B and the pending entries (C) are merged into one base run, in place or at the
/// tail of the arena. An entry's place is its index in its run plus the entries of the other two
/// runs before it: A before B before C among equal neighbours.
DYNG_DEV void full_merge(const merge_params& p, int block, int blocks, long long stage_from) {
  __shared__ int32_t s_v[kMergeSeg];
  __shared__ int32_t s_pp[kMergeSeg + 1];
  __shared__ int32_t s_b[kTailMax];
  __shared__ int s_tot[kMergeWaves];
  __shared__ long long s_stage, s_dest;
  __shared__ int s_newcap;
  const int count = p.list_count[kFull];
  const int32_t* list = p.lists + kFull * (p.N + 1);
  const u64 mask = (1ULL << p.vbits) - 1;
  const int tid = static_cast<int>(threadIdx.x);
  const int K = p.K;
  for (int t = block; t < count; t += blocks) {
    const int32_t u = list[t];
    const int2 mt = p.meta[u];
    const int64_t a = p.row_a[u], b = p.row_b[u];
    const int nops = static_cast<int>(b - a);
    const row_plan r = plan_row(read_facts(p, u, static_cast<int32_t>(a), static_cast<int32_t>(b)));
    if (tid == 0) {
      s_stage = stage_from + static_cast<long long>(atomicAdd(reinterpret_cast<unsigned long long*>(p.stage_used),
                                                 static_cast<unsigned long long>(r.alive_base + r.alive_tail)));
      s_newcap = p.cap[u];
      s_dest = mt.x;
      if (s_stage + r.alive_base + r.alive_tail > p.stage_cap) {
        atomicOr(p.error_bits, static_cast<int>(DYNG_HIP_DEVICE_ERROR_CAPACITY));
        s_dest = -1;
      } else if (r.new_len > p.cap[u]) {
        const int nc = grown_cap(r.new_len, p.headroom);
        const long long d = static_cast<long long>(
            atomicAdd(reinterpret_cast<unsigned long long*>(p.tail), static_cast<unsigned long long>(nc)));
        if (d + nc > p.slot_cap) {
          atomicOr(p.error_bits, static_cast<int>(DYNG_HIP_DEVICE_ERROR_CAPACITY));
          s_dest = -1;
        } else {
          atomicAdd(reinterpret_cast<unsigned long long*>(p.garbage), static_cast<unsigned long long>(p.cap[u]));
          atomicAdd(p.relocated, 1ULL);
          s_dest = d;
          s_newcap = nc;
        }
      }
    }
    __syncthreads();
    if (s_dest < 0) {
      __syncthreads();
      continue;
    }
    const long long sa = s_stage;
    const long long dest = s_dest;
    const int pa = p.pend_prefix[a];
    const bool ops_lds = nops <= kMergeSeg;
    if (ops_lds) {
      for (int j = tid; j < nops; j += kMergeBlock) {
        s_v[j] = static_cast<int32_t>(p.keys[a + j] & mask);
        s_pp[j] = p.pend_prefix[a + j] - pa;
      }
      if (tid == 0) s_pp[nops] = p.pend_prefix[b] - pa;
    }
    const int A = compact_alive(p, mt.x, r.base_len, sa, s_tot);
    const int B = compact_alive(p, mt.x + int64_t{r.base_len}, r.tail_len, sa + A, s_tot);
    const int32_t* SA = p.stage_nbr + sa;
    const int32_t* SB = p.stage_nbr + sa + A;
    for (int j = tid; j < B; j += kMergeBlock) s_b[j] = SB[j];  // B <= kTailMax
    __syncthreads();  // the staged runs (and the row's old slots are free to overwrite)
    // pending entries before v (strictly smaller neighbour)
    auto pend_before = [&](int32_t v) -> int {
      if (ops_lds) return s_pp[lds_bound(s_v, nops, v, false)];
      const int64_t lt = lower_key(p.keys, a, b, (static_cast<u64>(u) << p.vbits) | static_cast<u64>(v));
      return p.pend_prefix[lt] - pa;
    };
    for (int i = tid; i < A; i += kMergeBlock) {
      const int32_t v = SA[i];
      const int64_t pos = dest + i + lds_bound(s_b, B, v, false) + pend_before(v);
      p.nbr[pos] = v;
      for (int k = 0; k < K; ++k) p.w[k * p.slot_cap + pos] = p.stage_w[k * p.stage_cap + sa + i];
    }
    for (int j = tid; j < B; j += kMergeBlock) {
      const int32_t v = s_b[j];
      const int64_t pos = dest + global_bound(SA, A, v, true) + j + pend_before(v);
      p.nbr[pos] = v;
      for (int k = 0; k < K; ++k) p.w[k * p.slot_cap + pos] = p.stage_w[k * p.stage_cap + sa + A + j];
    }
    for (int64_t q = a + tid; q < b; q += kMergeBlock) {
      if (!p.pend_alive[q]) continue;
      const int32_t v = static_cast<int32_t>(p.keys[q] & mask);
      const int64_t pos = dest + global_bound(SA, A, v, true) + lds_bound(s_b, B, v, true) + (p.pend_prefix[q] - pa);
      p.nbr[pos] = v;
      for (int k = 0; k < K; ++k) p.w[k * p.slot_cap + pos] = p.pend_w[k * p.N + q];
    }
    if (tid == 0) {
      const int len = A + B + r.pending;
      p.meta[u] = make_int2(static_cast<int32_t>(dest), len);
      p.base[u] = len;
      p.dead[u] = 0;
      p.cap[u] = s_newcap;
    }
    __syncthreads();
  }
}

/// The rows that take a workgroup each, of both stores: tails, then whole rows. The in-rows stage behind
/// what the plan says the out-rows take. One launch where three took 11 us for a batch of 10.
__global__ void __launch_bounds__(kMergeBlock) k_rows(merge_roles m) {
  if (m.gate != nullptr && m.gate->hold != 0) return;  // uniform: the merges did not fit
  int b = static_cast<int>(blockIdx.x), role = 0;
  while (role < 3 && b >= m.groups[role]) b -= m.groups[role++];
  const merge_params& p = m.side[role & 1];
  if (role < 2) {
    tail_block(p, b, m.groups[role]);
  } else {
    full_merge(p, b, m.groups[role], role == 3 ? *m.side[0].need_stage : 0);
  }
}

/// Copy one row store into a fresh arena (compaction): one wave per row.
__global__ void k_compact_rows(const int2* meta, const int32_t* nbr, const int32_t* w, int64_t slot_cap,
                               int64_t n, int K, const int64_t* new_off, int2* new_meta, int32_t* new_nbr,
                               int32_t* new_w, int64_t new_slot_cap) {
  const int64_t wave = (blockIdx.x * int64_t{blockDim.x} + threadIdx.x) / 64;
  const int64_t waves = (int64_t{gridDim.x} * blockDim.x) / 64;
  for (int64_t u = wave; u < n; u += waves) {
    const int2 mt = meta[u];
    const int64_t o = new_off[u];
    for (int j = lane(); j < mt.y; j += 64) {
      new_nbr[o + j] = nbr[mt.x + j];
      for (int k = 0; k < K; ++k) new_w[k * new_slot_cap + o + j] = w[k * slot_cap + mt.x + j];
    }
    if (lane() == 0) new_meta[u] = make_int2(static_cast<int32_t>(o), mt.y);
  }
}

/// A freshly built row is one base run.
__global__ void k_base_from_len(const int2* meta, int64_t n, int32_t* base, int32_t* dead) {
  for (int64_t u = blockIdx.x * int64_t{blockDim.x} + threadIdx.x; u < n; u += int64_t{gridDim.x} * blockDim.x) {
    base[u] = meta[u].y;
    dead[u] = 0;
  }
}

__global__ void k_caps_from_len(const int2* meta, int64_t n, double headroom, int32_t* cap, int64_t* cap64) {
  for (int64_t u = blockIdx.x * int64_t{blockDim.x} + threadIdx.x; u < n; u += int64_t{gridDim.x} * blockDim.x) {
    const int len = meta[u].y;
    const int c = len + static_cast<int>(ceil(len * headroom)) + 2;
    cap[u] = c;
    cap64[u] = c;
  }
}

// ---------------------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------------------

hipStream_t as_stream(void* s) { return static_cast<hipStream_t>(s); }

int64_t arena_slots(int64_t rows_slots, int64_t m, int64_t extra) {
  return rows_slots + std::max<int64_t>(m + m / 2, 1 << 16) + extra;
}

void check_slots(int64_t slots) {
  if (slots >= (int64_t{1} << 31) - 1) {
    fail(DYNG_HIP_NOT_SUPPORTED,
         "dyng: the HIP device graph holds at most 2^31 - 1 edge slots per direction (needed " +
             std::to_string(slots) + ")");
  }
}

/// Build one row store from sorted keys (u << b | v) with keep flags and weights.
void build_store(dyng_hip_graph* g, row_store& rs, const u64* keys, const uint32_t* vals, int64_t N,
                 const int32_t* keep, int vbits, int stride, const int32_t* w_in, int from_slots,
                 int64_t in_slot_cap, hipStream_t s) {
  const int64_t n = g->n_cap;
  dbuf<int32_t> keep_prefix;
  keep_prefix.reserve(N + 1);
  exclusive_scan<int32_t>(g->scan_tmp, keep, keep_prefix.p, N + 1, s);
  rs.meta.reserve(n);
  rs.cap.reserve(n);
  rs.base.reserve(n);
  rs.dead.reserve(n);
  fill<int2>(rs.meta.p, n, make_int2(0, 0), s);
  fill<int32_t>(rs.cap.p, n, 0, s);
  fill<int32_t>(rs.base.p, n, 0, s);
  fill<int32_t>(rs.dead.p, n, 0, s);
  dbuf<int64_t> cap64, off64;
  cap64.reserve(g->n + 1);
  off64.reserve(g->n + 1);
  fill<int64_t>(cap64.p, g->n + 1, 0, s);
  hipLaunchKernelGGL(k_row_degrees, dim3(blocks_for(g->n)), dim3(kBlock), 0, s, keys, N, keep_prefix.p,
                     g->n, vbits, g->props.headroom, rs.meta.p, rs.cap.p, cap64.p);
  DYNG_HIP_TRY(hipGetLastError());
  exclusive_scan<int64_t>(g->scan_tmp, cap64.p, off64.p, g->n + 1, s);
  int64_t rows_slots = 0;
  DYNG_HIP_TRY(hipMemcpyAsync(&rows_slots, off64.p + g->n, sizeof(int64_t), hipMemcpyDeviceToHost, s));
  DYNG_HIP_TRY(hipStreamSynchronize(s));
  hipLaunchKernelGGL(k_set_offsets, dim3(blocks_for(g->n)), dim3(kBlock), 0, s, off64.p, g->n, rs.meta.p);
  const int64_t slots = arena_slots(rows_slots, N, 0);
  check_slots(slots);
  rs.slot_cap = slots;
  rs.tail = rows_slots;
  rs.garbage = 0;
  rs.nbr.reserve(slots);
  rs.w.reserve(slots * g->K);
  hipLaunchKernelGGL(k_fill_rows, dim3(blocks_for(N)), dim3(kBlock), 0, s, keys, vals, N, keep,
                     keep_prefix.p, vbits, stride, rs.meta.p, rs.nbr.p, rs.w.p, rs.slot_cap, g->K, w_in,
                     from_slots, in_slot_cap);
  DYNG_HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_base_from_len, dim3(blocks_for(g->n)), dim3(kBlock), 0, s, rs.meta.p, g->n, rs.base.p,
                     rs.dead.p);
  DYNG_HIP_TRY(hipGetLastError());
}

/// In-rows from the out-rows.
void build_in_store(dyng_hip_graph* g, hipStream_t s) {
  const int64_t n = g->n;
  const int vbits = bits_for(std::max<int64_t>(n, 1));
  dbuf<int64_t> len64, pos64;
  len64.reserve(n + 1);
  pos64.reserve(n + 1);
  fill<int64_t>(len64.p, n + 1, 0, s);
  hipLaunchKernelGGL(k_len64, dim3(blocks_for(n)), dim3(kBlock), 0, s, g->out.meta.p, n, len64.p);
  exclusive_scan<int64_t>(g->scan_tmp, len64.p, pos64.p, n + 1, s);
  const int64_t M = g->m;
  dbuf<u64> ka, kb;
  dbuf<uint32_t> va, vb;
  dbuf<int32_t> keep;
  ka.reserve(M);
  kb.reserve(M);
  va.reserve(M);
  vb.reserve(M);
  keep.reserve(M + 1);
  hipLaunchKernelGGL(k_reverse_keys, dim3(blocks_for(n * 64)), dim3(kBlock), 0, s, g->out.meta.p, g->out.nbr.p, n,
                     vbits, ka.p, va.p, pos64.p);
  DYNG_HIP_TRY(hipGetLastError());
  sort_pairs(g->sort_tmp, ka.p, kb.p, va.p, vb.p, M, 2 * vbits, s);
  hipLaunchKernelGGL(k_keep, dim3(blocks_for(M + 1)), dim3(kBlock), 0, s, kb.p, M, 1, keep.p);
  build_store(g, g->in, kb.p, vb.p, M, keep.p, vbits, 1, g->out.w.p, 1, g->out.slot_cap, s);
  DYNG_HIP_TRY(hipStreamSynchronize(s));
}

/// Exact column summaries (max, sum, count of the max) of every objective.
void recompute_columns(dyng_hip_graph* g, hipStream_t s) {
  apply_control* c = g->host_ctl.p;
  std::memset(c, 0, sizeof(apply_control));
  DYNG_HIP_TRY(hipMemcpyAsync(g->ctl.p, c, sizeof(apply_control), hipMemcpyHostToDevice, s));
  // a bounded grid (one reduction per wave, then one atomic per wave and column)
  const unsigned grid = std::min(blocks_for(g->n), 2048u);
  hipLaunchKernelGGL(k_column_summary, dim3(grid), dim3(kBlock), 0, s, g->out.meta.p, g->out.nbr.p, g->out.w.p,
                     g->n, g->out.slot_cap, g->K, 0, g->ctl.p);
  DYNG_HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_column_summary, dim3(grid), dim3(kBlock), 0, s, g->out.meta.p, g->out.nbr.p, g->out.w.p,
                     g->n, g->out.slot_cap, g->K, 1, g->ctl.p);
  DYNG_HIP_TRY(hipGetLastError());
  DYNG_HIP_TRY(hipMemcpyAsync(c, g->ctl.p, sizeof(apply_control), hipMemcpyDeviceToHost, s));
  DYNG_HIP_TRY(hipStreamSynchronize(s));
  g->wmax.assign(g->K, 1);
  g->wsum.assign(g->K, 0);
  g->wmax_count.assign(g->K, 0);
  g->wmin.assign(g->K, 1);
  for (int k = 0; k < g->K; ++k) {
    g->wmin[k] = c->col_bad[k] == 0 ? 1 : 0;
    g->wmax[k] = std::max<long long>(1, c->col_max[k]);
    g->wsum[k] = c->col_dsum[k];
    g->wmax_count[k] = c->col_max[k] >= 1 ? c->col_dcount[k] : 0;
  }
}

void compact_store(dyng_hip_graph* g, row_store& rs, int64_t extra, hipStream_t s) {
  const int64_t n = g->n;
  dbuf<int64_t> cap64, off64;
  cap64.reserve(n + 1);
  off64.reserve(n + 1);
  fill<int64_t>(cap64.p, n + 1, 0, s);
  hipLaunchKernelGGL(k_caps_from_len, dim3(blocks_for(n)), dim3(kBlock), 0, s, rs.meta.p, n, g->props.headroom,
                     rs.cap.p, cap64.p);
  exclusive_scan<int64_t>(g->scan_tmp, cap64.p, off64.p, n + 1, s);
  int64_t rows_slots = 0;
  DYNG_HIP_TRY(hipMemcpyAsync(&rows_slots, off64.p + n, sizeof(int64_t), hipMemcpyDeviceToHost, s));
  DYNG_HIP_TRY(hipStreamSynchronize(s));
  const int64_t slots = arena_slots(rows_slots, g->m, extra);
  check_slots(slots);
  row_store fresh;
  fresh.meta.reserve(g->n_cap);
  fresh.nbr.reserve(slots);
  fresh.w.reserve(slots * g->K);
  fill<int2>(fresh.meta.p, g->n_cap, make_int2(0, 0), s);
  hipLaunchKernelGGL(k_compact_rows, dim3(blocks_for(n * 64)), dim3(kBlock), 0, s, rs.meta.p, rs.nbr.p, rs.w.p,
                     rs.slot_cap, n, g->K, off64.p, fresh.meta.p, fresh.nbr.p, fresh.w.p, slots);
  DYNG_HIP_TRY(hipGetLastError());
  DYNG_HIP_TRY(hipStreamSynchronize(s));
  std::swap(rs.meta.p, fresh.meta.p);
  std::swap(rs.meta.n, fresh.meta.n);
  std::swap(rs.nbr.p, fresh.nbr.p);
  std::swap(rs.nbr.n, fresh.nbr.n);
  std::swap(rs.w.p, fresh.w.p);
  std::swap(rs.w.n, fresh.w.n);
  rs.slot_cap = slots;
  rs.tail = rows_slots;
  rs.garbage = 0;
}

void grow_vertices(dyng_hip_graph* g, int64_t n_after, hipStream_t s) {
  if (n_after <= g->n) return;
  if (n_after > g->n_cap) {
    const int64_t cap = std::max<int64_t>(n_after, g->n_cap + g->n_cap / 2);
    for (row_store* rs : {&g->out, &g->in}) {
      rs->meta.reserve(cap, true, s);
      rs->cap.reserve(cap, true, s);
      rs->base.reserve(cap, true, s);
      rs->dead.reserve(cap, true, s);
    }
    g->mark_out.reserve(cap, true, s);
    g->mark_in.reserve(cap, true, s);
    fill<int32_t>(g->mark_out.p + g->n_cap, cap - g->n_cap, 0, s);
    fill<int32_t>(g->mark_in.p + g->n_cap, cap - g->n_cap, 0, s);
    g->n_cap = cap;
  }
  for (row_store* rs : {&g->out, &g->in}) {
    fill<int2>(rs->meta.p + g->n, n_after - g->n, make_int2(0, 0), s);
    fill<int32_t>(rs->cap.p + g->n, n_after - g->n, 0, s);
    fill<int32_t>(rs->base.p + g->n, n_after - g->n, 0, s);
    fill<int32_t>(rs->dead.p + g->n, n_after - g->n, 0, s);
  }
}

dyng_hip_graph* create_from_edge_list(int device, const dyng_hip_graph_props* props, int64_t n, int64_t count,
                                      int32_t K, const int32_t* src, const int32_t* dst, const int32_t* w,
                                      int32_t from_device, hipStream_t s) {
  if (props == nullptr) fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: graph properties are required");
  if (n < 0 || n >= INT32_MAX) fail(DYNG_HIP_NOT_SUPPORTED, "dyng: the HIP backend takes int32 vertex ids");
  if (K < 1 || K > max_weights) {
    fail(DYNG_HIP_NOT_SUPPORTED, "dyng: the HIP sssp backend takes 1.." + std::to_string(max_weights) +
                                     " weight columns, got " + std::to_string(K));
  }
  if (props->on_existing_insert < 0 || props->on_existing_insert > 2 || props->on_missing_delete < 0 ||
      props->on_missing_delete > 1) {
    fail(DYNG_HIP_INVALID_ARGUMENT,
         "dyng: on_existing_insert must be 0 (upsert), 1 (error) or 2 (ignore) and on_missing_delete 0 "
         "(ignore) or 1 (error)");
  }
  scoped_device guard(device);
  auto g = std::make_unique<dyng_hip_graph>();
  g->device = device;
  g->props = *props;
  if (!(g->props.headroom >= 0.0) || g->props.headroom > 16.0) g->props.headroom = 0.25;
  g->K = K;
  g->n = n;
  g->n_cap = std::max<int64_t>(n, 1);
  const int stride = props->directed ? 1 : 2;
  const int64_t N = count * stride;
  if (N >= (int64_t{1} << 32)) fail(DYNG_HIP_NOT_SUPPORTED, "dyng: too many edges for the HIP device graph");
  const int vbits = bits_for(std::max<int64_t>(n, 1));
  // stage the edge list on the device
  dbuf<int32_t> d_src, d_dst, d_w;
  const int32_t* ps = src;
  const int32_t* pd = dst;
  const int32_t* pw = w;
  if (!from_device) {
    d_src.reserve(count);
    d_dst.reserve(count);
    d_w.reserve(count * K);
    if (count > 0) {
      DYNG_HIP_TRY(hipMemcpyAsync(d_src.p, src, count * sizeof(int32_t), hipMemcpyHostToDevice, s));
      DYNG_HIP_TRY(hipMemcpyAsync(d_dst.p, dst, count * sizeof(int32_t), hipMemcpyHostToDevice, s));
      DYNG_HIP_TRY(hipMemcpyAsync(d_w.p, w, count * K * sizeof(int32_t), hipMemcpyHostToDevice, s));
    }
    ps = d_src.p;
    pd = d_dst.p;
    pw = d_w.p;
  }
  g->ctl.reserve(1);
  dbuf<u64> ka, kb;
  dbuf<uint32_t> va, vb;
  dbuf<int32_t> keep;
  ka.reserve(N);
  kb.reserve(N);
  va.reserve(N);
  vb.reserve(N);
  keep.reserve(N + 1);
  if (N > 0) {
    hipLaunchKernelGGL(k_edge_keys, dim3(blocks_for(N)), dim3(kBlock), 0, s, ps, pd, count, stride,
                       props->directed, props->on_self_loop == 1 ? 1 : 0, vbits, ka.p, va.p);
    DYNG_HIP_TRY(hipGetLastError());
    sort_pairs(g->sort_tmp, ka.p, kb.p, va.p, vb.p, N, 2 * vbits, s);
  }
  hipLaunchKernelGGL(k_keep, dim3(blocks_for(N + 1)), dim3(kBlock), 0, s, kb.p, N, props->allow_parallel, keep.p);
  DYNG_HIP_TRY(hipGetLastError());
  build_store(g.get(), g->out, kb.p, vb.p, N, keep.p, vbits, stride, pw, 0, 0, s);
  // edges kept
  {
    dbuf<int32_t> kp;
    kp.reserve(N + 1);
    exclusive_scan<int32_t>(g->scan_tmp, keep.p, kp.p, N + 1, s);
    int32_t mm = 0;
    DYNG_HIP_TRY(hipMemcpyAsync(&mm, kp.p + N, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    DYNG_HIP_TRY(hipStreamSynchronize(s));
    g->m = mm;
  }
  g->mark_out.reserve(g->n_cap);
  g->mark_in.reserve(g->n_cap);
  fill<int32_t>(g->mark_out.p, g->n_cap, 0, s);
  fill<int32_t>(g->mark_in.p, g->n_cap, 0, s);
  build_in_store(g.get(), s);
  recompute_columns(g.get(), s);
  static uint64_t next_state = 1;
  g->state_id = __atomic_fetch_add(&next_state, 1, __ATOMIC_RELAXED);
  return g.release();
}

void copy_rows_to_host(const row_store& rs, int64_t n, int K, int64_t* row_ptr, int32_t* col, int32_t* w) {
  std::vector<int2> meta(static_cast<size_t>(n));
  std::vector<int32_t> base(static_cast<size_t>(n));
  if (n > 0) {
    DYNG_HIP_TRY(hipMemcpy(meta.data(), rs.meta.p, n * sizeof(int2), hipMemcpyDeviceToHost));
    DYNG_HIP_TRY(hipMemcpy(base.data(), rs.base.p, n * sizeof(int32_t), hipMemcpyDeviceToHost));
  }
  std::vector<int32_t> nbr(static_cast<size_t>(rs.slot_cap));
  std::vector<int32_t> wt(static_cast<size_t>(rs.slot_cap) * K);
  if (rs.slot_cap > 0) {
    DYNG_HIP_TRY(hipMemcpy(nbr.data(), rs.nbr.p, rs.slot_cap * sizeof(int32_t), hipMemcpyDeviceToHost));
    DYNG_HIP_TRY(hipMemcpy(wt.data(), rs.w.p, rs.slot_cap * K * sizeof(int32_t), hipMemcpyDeviceToHost));
  }
  // each row in the reference's order: its base and tail runs merged by neighbour id (base
  // entries first among equal ones), dead entries dropped
  row_ptr[0] = 0;
  for (int64_t u = 0; u < n; ++u) {
    int64_t alive = 0;
    for (int j = 0; j < meta[u].y; ++j) alive += nbr[meta[u].x + j] >= 0 ? 1 : 0;
    row_ptr[u + 1] = row_ptr[u] + alive;
  }
  const int64_t m = row_ptr[n];
  for (int64_t u = 0; u < n; ++u) {
    const int64_t off = meta[u].x;
    int i = 0, j = base[u];
    const int bend = base[u], tend = meta[u].y;
    int64_t o = row_ptr[u];
    auto put = [&](int x) {
      col[o] = nbr[off + x];
      for (int k = 0; k < K; ++k) w[k * m + o] = wt[k * rs.slot_cap + off + x];
      ++o;
    };
    for (;;) {
      while (i < bend && nbr[off + i] < 0) ++i;
      while (j < tend && nbr[off + j] < 0) ++j;
      if (i == bend && j == tend) break;
      if (j == tend || (i < bend && nbr[off + i] <= nbr[off + j])) {
        put(i++);
      } else {
        put(j++);
      }
    }
  }
}

}  // namespace

// ---------------------------------------------------------------------------------------------
// The apply (host orchestration)
// ---------------------------------------------------------------------------------------------

namespace {

/// Whether the apply times its stages: DYNG_HIP_STAGE_TIMES=1 in the environment. Each timed
/// event costs the stream a few microseconds, so the stages are not timed by default.
bool stage_timing() {
  static const bool on = [] {
    const char* v = std::getenv("DYNG_HIP_STAGE_TIMES");
    return v != nullptr && v[0] == '1';
  }();
  return on;
}

void mark_stage(dyng_hip_graph* g, int i, hipStream_t s) {
  if (!stage_timing()) return;
  if (g->apply_ev[i] == nullptr) DYNG_HIP_TRY(hipEventCreate(&g->apply_ev[i]));
  DYNG_HIP_TRY(hipEventRecord(g->apply_ev[i], s));
}

/// Stage durations from the recorded events (after the stream has been synchronized).
void stage_times(dyng_hip_graph* g, bool rows, dyng_hip_apply_summary* out) {
  for (double& t : out->stage_ms) t = 0.0;
  if (!stage_timing()) return;
  float ms = 0.0f;
  if (hipEventElapsedTime(&ms, g->apply_ev[0], g->apply_ev[1]) == hipSuccess) out->stage_ms[0] = ms;
  if (!rows) return;
  for (int i = 2; i < 12; ++i) {
    if (hipEventElapsedTime(&ms, g->apply_ev[i], g->apply_ev[i + 1]) == hipSuccess) out->stage_ms[i - 1] = ms;
  }
}

}  // namespace

void graph_grow(dyng_hip_graph* g, int64_t n, hipStream_t s) {
  if (n <= g->n) return;
  if (n >= INT32_MAX) fail(DYNG_HIP_NOT_SUPPORTED, "dyng: the HIP backend takes int32 vertex ids");
  grow_vertices(g, n, s);
  g->n = n;
}

void scan_batch(dyng_hip_graph* g, const dyng_hip_batch* b, hipStream_t s, batch_scan& sc) {
  if (b == nullptr) fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: graph apply: no batch");
  mark_stage(g, 0, s);
  const int K = g->K;
  const int64_t num_ins = b->num_ins, num_del = b->num_del;
  if (num_ins < 0 || num_del < 0) fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: negative batch sizes");
  if (num_ins > 0 && b->num_weights != K) {
    fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: the batch has " + std::to_string(b->num_weights) +
                                        " weights per insertion but the graph has " + std::to_string(K));
  }
  // stage host batches on the device
  const int32_t *ins_src = b->ins_src, *ins_dst = b->ins_dst, *ins_w = b->ins_w, *del_src = b->del_src,
                *del_dst = b->del_dst;
  if (!b->on_device) {
    // one device buffer, each array from a 256-byte boundary on
    const int32_t* from[5] = {ins_src, ins_dst, ins_w, del_src, del_dst};
    const int64_t count[5] = {num_ins, num_ins, num_ins * K, num_del, num_del};
    int64_t at[5], total = 0;
    for (int i = 0; i < 5; ++i) {
      at[i] = total;
      total += (count[i] + 63) / 64 * 64;
    }
    g->b_batch.reserve(total);
    if (total * 4 <= kGatherBytes) {
      // a small batch: gathered in pinned memory (the last batch's copy ended before its scan was read)
      // and sent as one copy. Five copies from pageable memory took 23 us of a batch of 1,000.
      g->host_batch.reserve(static_cast<size_t>(total) * 4);
      for (int i = 0; i < 5; ++i) {
        if (count[i] > 0) std::memcpy(g->host_batch.p + at[i] * 4, from[i], static_cast<size_t>(count[i]) * 4);
      }
      if (total > 0) DYNG_HIP_TRY(hipMemcpyAsync(g->b_batch.p, g->host_batch.p, total * 4, hipMemcpyHostToDevice, s));
    } else {
      for (int i = 0; i < 5; ++i) {
        if (count[i] > 0) DYNG_HIP_TRY(hipMemcpyAsync(g->b_batch.p + at[i], from[i], count[i] * 4, hipMemcpyHostToDevice, s));
      }
    }
    ins_src = g->b_batch.p + at[0];
    ins_dst = g->b_batch.p + at[1];
    ins_w = g->b_batch.p + at[2];
    del_src = g->b_batch.p + at[3];
    del_dst = g->b_batch.p + at[4];
  }
  // ---- scan the batch (ids, self-loops, weights) before anything changes ----
  int min_id = INT32_MAX, max_id = -1, self_loops = 0;
  sc.wmax.assign(K, 0);
  sc.wmin.assign(K, 1);
  if (num_ins + num_del == 0) {
    mark_stage(g, 1, s);
  } else {
    const int blocks = static_cast<int>(std::min<unsigned>(blocks_for(std::max(num_ins, num_del), kScanBlock), kScanParts));
    scan_part* parts = g->host_scan.p->part;
    hipLaunchKernelGGL(k_batch_scan, dim3(static_cast<unsigned>(blocks)), dim3(kScanBlock), 0, s, ins_src, ins_dst, ins_w,
                       num_ins, del_src, del_dst, num_del, K, parts);
    DYNG_HIP_TRY(hipGetLastError());
    mark_stage(g, 1, s);
    DYNG_HIP_TRY(hipStreamSynchronize(s));
    for (int b = 0; b < blocks; ++b) {
      min_id = std::min(min_id, parts[b].id[0]);
      max_id = std::max(max_id, parts[b].id[1]);
      self_loops += parts[b].id[2] != 0 || parts[b].id[3] != 0 ? 1 : 0;
      for (int k = 0; k < K; ++k) {
        sc.wmax[k] = std::max<int64_t>(sc.wmax[k], parts[b].wmax[k]);
        sc.wmin[k] = std::min<int64_t>(sc.wmin[k], parts[b].wmin[k]);
      }
    }
  }
  if (min_id < 0) fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: the batch names a negative vertex id");
  if (g->props.on_self_loop == 2 && self_loops > 0) {
    fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: the batch has a self-loop and on_self_loop is error");
  }
  int64_t n_after = g->n;
  if (max_id >= 0) {
    if (!g->props.allow_vertex_growth && max_id >= g->n) {
      fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: an insertion names a vertex >= " + std::to_string(g->n) +
                                          " and allow_vertex_growth is false");
    }
    if (max_id >= INT32_MAX - 1) fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: an insertion names the largest vertex id");
    // a self-loop insertion that is dropped does not grow the vertex set; keep the rule simple by
    // growing only for kept insertions (the scan covers them all; drop is rare)
    n_after = std::max<int64_t>(n_after, static_cast<int64_t>(max_id) + 1);
  }
  sc.n_after = n_after;
  sc.num_ins = num_ins;
  sc.num_del = num_del;
  sc.ins_src = ins_src;
  sc.ins_dst = ins_dst;
  sc.ins_w = ins_w;
  sc.del_src = del_src;
  sc.del_dst = del_dst;
}

/// The merge parameters of one row store for a batch of N operations (keys of `vbits` bits).
merge_params merge_setup(dyng_hip_graph* g, bool outs, int64_t N, int vbits) {
  apply_control* dc = g->ctl.p;
  row_store& rs = outs ? g->out : g->in;
  merge_params mp{};
  mp.meta = rs.meta.p;
  mp.cap = rs.cap.p;
  mp.base = rs.base.p;
  mp.dead = rs.dead.p;
  mp.nbr = rs.nbr.p;
  mp.w = rs.w.p;
  mp.slot_cap = rs.slot_cap;
  mp.K = g->K;
  mp.keys = outs ? g->ops.keys_b : g->ops.keys_b + N;
  mp.N = N;
  mp.vbits = vbits;
  mp.pend_alive = outs ? g->ops.pend_alive : g->ops.ipend_alive;
  mp.pend_prefix = outs ? g->ops.pend_prefix : g->ops.ipend_prefix;
  mp.kill_prefix = outs ? g->ops.kill_prefix : g->ops.ikill_prefix;
  mp.pend_w = outs ? g->ops.pend_w : g->ops.ipend_w;
  mp.touched = outs ? g->ops.touched_out : g->ops.touched_in;
  mp.touched_count = outs ? &dc->touched_out : &dc->touched_in;
  mp.row_a = outs ? g->row_a_out.p : g->row_a_in.p;
  mp.row_b = outs ? g->row_b_out.p : g->row_b_in.p;
  mp.lane_rows = g->ops.lane_rows + (outs ? 0 : 2 * (N + 1));
  mp.lists = g->ops.merge_lists + (outs ? 0 : kModes * (N + 1));
  mp.list_count = outs ? dc->modes_out : dc->modes_in;
  mp.stage_nbr = g->stage_nbr.p;
  mp.stage_w = g->stage_w.p;
  mp.stage_cap = g->stage_cap;
  mp.stage_used = outs ? &dc->stage_out : &dc->stage_in;
  mp.tail = outs ? &dc->tail_out : &dc->tail_in;
  mp.garbage = outs ? &dc->garbage_out : &dc->garbage_in;
  mp.relocated = &dc->relocated_rows;
  mp.need_reloc = outs ? &dc->need_reloc_out : &dc->need_reloc_in;
  mp.need_stage = outs ? &dc->need_stage_out : &dc->need_stage_in;
  mp.error_bits = &dc->error_bits;
  mp.headroom = g->props.headroom;
  return mp;
}

unsigned plan_groups(int64_t N) { return static_cast<unsigned>((N + kPlanBlock - 1) / kPlanBlock); }  // rows <= N

/// Launch the merges: `rows` of each store's per mode (an upper bound, the merges loop over what the
/// plan listed), `cap` limiting the workgroups per role and store.
void launch_merges(dyng_hip_graph* g, int64_t P, int vbits, const int* out_rows, const int* in_rows, bool gated,
                   const int (&cap)[kModes], hipStream_t s) {
  merge_roles m{};
  m.side[0] = merge_setup(g, true, P, vbits);
  m.side[1] = merge_setup(g, false, P, vbits);
  m.gate = gated ? g->ctl.p : nullptr;
  auto groups = [&](int rows, int per_group, int mode) { return std::min((rows + per_group - 1) / per_group, cap[mode]); };
  auto launch = [&](void (*kernel)(merge_roles), int mode0, int per0, int mode1, int per1, int threads) {
    m.groups[0] = groups(out_rows[mode0], per0, mode0);
    m.groups[1] = groups(in_rows[mode0], per0, mode0);
    m.groups[2] = groups(out_rows[mode1], per1, mode1);
    m.groups[3] = groups(in_rows[mode1], per1, mode1);
    const int all = m.groups[0] + m.groups[1] + m.groups[2] + m.groups[3];
    if (all > 0) hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(all)), dim3(threads), 0, s, m);
    DYNG_HIP_TRY(hipGetLastError());
  };
  mark_stage(g, 10, s);
  launch(g->K == 1 ? k_tails<1> : k_tails<kRegWeights>, kTailWave, kTailsBlock / 64, kTailLane, kTailsBlock, kTailsBlock);
  mark_stage(g, 11, s);
  launch(k_rows, kTailBlock, 1, kFull, 1, kMergeBlock);
  mark_stage(g, 12, s);
}

/// The merge plan and the merges with the plan read back first: the launches sized from it, the
/// arenas compacted and the staging arena grown as it needs. kPlanAgain: a plan already ran (its
/// counts are cleared first); kPlanDone: it is the one to use.
enum plan_state { kPlanNone, kPlanAgain, kPlanDone };
void merges_exact(dyng_hip_graph* g, int64_t N, int vbits, hipStream_t s, dyng_hip_apply_summary* out, plan_state state) {
  apply_control* hc = g->host_ctl.p;
  apply_control* dc = g->ctl.p;
  const int K = g->K;
  for (int attempt = 0;; ++attempt) {
    const bool planned = attempt == 0 && state == kPlanDone;
    if (attempt > 0 || state == kPlanAgain) {
      // planning again: clear what the last plan counted (the first plan of a batch finds them
      // zero, as the control block was uploaded zeroed at the start of the apply)
      hc->need_reloc_out = hc->need_reloc_in = hc->need_stage_out = hc->need_stage_in = 0;
      for (int i = 0; i < kModes; ++i) hc->modes_out[i] = hc->modes_in[i] = 0;
      DYNG_HIP_TRY(hipMemcpyAsync(&dc->need_reloc_out, &hc->need_reloc_out, 4 * sizeof(long long),
                                  hipMemcpyHostToDevice, s));
      DYNG_HIP_TRY(hipMemcpyAsync(dc->modes_out, hc->modes_out, 2 * sizeof(hc->modes_out), hipMemcpyHostToDevice,
                                  s));
    }
    if (!planned) {
      merge_sides plan{};  // both stores' plans in one launch: out-rows first
      plan.side[0] = merge_setup(g, true, N, vbits);
      plan.side[1] = merge_setup(g, false, N, vbits);
      plan.split = static_cast<int>(plan_groups(N));
      hipLaunchKernelGGL(k_merge_plan, dim3(2 * plan_groups(N)), dim3(kPlanBlock), 0, s, plan);
      DYNG_HIP_TRY(hipGetLastError());
    }
    DYNG_HIP_TRY(hipMemcpyAsync(hc, dc, sizeof(apply_control), hipMemcpyDeviceToHost, s));
    DYNG_HIP_TRY(hipStreamSynchronize(s));
    if (out) out->host_plans += 1;
    if (hc->error_bits != 0 || hc->miss != 0) return;  // the caller's to report, or to sort and plan
    bool compacted = false;
    for (int side = 0; side < 2; ++side) {
      row_store& rs = side == 0 ? g->out : g->in;
      const int64_t need = (side == 0 ? hc->need_reloc_out : hc->need_reloc_in) + kArenaMargin;
      if (rs.slot_cap - rs.tail < need) {
        if (attempt > 2) fail(DYNG_HIP_RUNTIME_ERROR, "dyng: graph apply: the row arena cannot take the batch");
        compact_store(g, rs, 2 * need, s);
        if (out) out->compactions += 1;
        compacted = true;
      }
    }
    if (!compacted) break;
    // compaction recomputed the capacities: plan again on the fresh arenas
    hc->tail_out = g->out.tail;
    hc->tail_in = g->in.tail;
    hc->garbage_out = hc->garbage_in = 0;
    DYNG_HIP_TRY(hipMemcpyAsync(&dc->tail_out, &hc->tail_out, 2 * sizeof(long long), hipMemcpyHostToDevice, s));
    DYNG_HIP_TRY(hipMemcpyAsync(&dc->garbage_out, &hc->garbage_out, 2 * sizeof(long long), hipMemcpyHostToDevice, s));
  }
  const int64_t stage_need = hc->need_stage_out + hc->need_stage_in;
  if (stage_need > g->stage_cap) {
    g->stage_cap = stage_need + stage_need / 4 + 4096;
    g->stage_nbr.reserve(g->stage_cap);
    g->stage_w.reserve(g->stage_cap * K);
  }
  launch_merges(g, N, vbits, hc->modes_out, hc->modes_in, false, {32768, 4096, 4096, 8192}, s);
}

/// The merges of a small batch queued behind its plan, with no read-back in between: the device
/// checks that the arenas take what the plan asks (merges_fit) and holds the merges back otherwise;
/// the grids are sized for the batch (every touched row is one of its at most N + 1 rows per store)
/// and the merges loop over the rows the plan listed.
void merges_queued(dyng_hip_graph* g, int64_t N, int vbits, hipStream_t s) {
  int rows[kModes];
  std::fill(rows, rows + kModes, static_cast<int>(N + 1));
  launch_merges(g, N, vbits, rows, rows, true, {1024, 256, 256, 1024}, s);
}

/// The merge plan and the merges queued together (see merges_queued).
void merges_speculative(dyng_hip_graph* g, int64_t N, int vbits, hipStream_t s) {
  merge_sides plan{};
  plan.side[0] = merge_setup(g, true, N, vbits);
  plan.side[1] = merge_setup(g, false, N, vbits);
  plan.split = static_cast<int>(plan_groups(N));
  hipLaunchKernelGGL(k_merge_plan, dim3(2 * plan_groups(N)), dim3(kPlanBlock), 0, s, plan);
  DYNG_HIP_TRY(hipGetLastError());
  merges_queued(g, N, vbits, s);
}

/// Throw the invalid-argument error of the offending operation of rank `rank` (k_check_pairs):
/// the message names the operation's kind, batch index and (u, v), as apply_host.cpp:117-120 and
/// 222-225 do. Nothing has changed yet.
[[noreturn]] void report_batch_error(dyng_hip_graph* g, const batch_scan& sc, const op_layout& L,
                                     unsigned long long rank, hipStream_t s) {
  const bool row_phase = (rank >> 63) != 0;
  const int64_t j = static_cast<int64_t>(rank & 0x7fffffffULL);
  const bool second = ((rank >> 31) & 1ULL) != 0;
  const bool del = !row_phase || (second ? L.first_is_del == 0 : L.first_is_del != 0);
  int32_t uv[2] = {0, 0};
  const int32_t* src = del ? sc.del_src : sc.ins_src;
  const int32_t* dst = del ? sc.del_dst : sc.ins_dst;
  DYNG_HIP_TRY(hipMemcpyAsync(&uv[0], src + j, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  DYNG_HIP_TRY(hipMemcpyAsync(&uv[1], dst + j, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  DYNG_HIP_TRY(hipStreamSynchronize(s));
  if (row_phase) {
    // the arc of the row: (v, u) for the reverse arc of an undirected edge
    const int32_t row = static_cast<int32_t>((rank >> 32) & 0x7fffffffULL);
    if (row != uv[0]) std::swap(uv[0], uv[1]);
  }
  (void)g;
  const std::string op = std::string(del ? "deletion " : "insertion ") + std::to_string(j) + " (" +
                         std::to_string(uv[0]) + ", " + std::to_string(uv[1]) + ")";
  throw batch_refused(DYNG_HIP_INVALID_ARGUMENT,
                      "dyng: " + op +
                          (del ? " names a missing edge and batch_semantics::on_missing_delete is error"
                               : " names an existing edge and batch_semantics::on_existing_insert is error"));
}

/// The control block at the start of an apply: counters, tails, the column targets; the first
/// `num_counts` group counters cleared.
void begin_apply(dyng_hip_graph* g, const batch_scan& sc, int num_counts, hipStream_t s) {
  begin_params b{};
  b.tail_out = g->out.tail;
  b.tail_in = g->in.tail;
  for (int k = 0; k < g->K; ++k) b.col_max[k] = std::max<int64_t>(g->wmax[k], sc.wmax[k]);
  b.counts = g->ops.group_counts;
  b.num_counts = num_counts;
  hipLaunchKernelGGL(k_begin, dim3(1), dim3(1024), 0, s, g->ctl.p, b);
  DYNG_HIP_TRY(hipGetLastError());
}

scratch_pool& apply_scratch(int device) {
  struct pools {
    std::mutex lock;
    std::map<int, std::unique_ptr<scratch_pool>> of;
  };
  static pools* all = new pools();  // lives until the process ends
  std::lock_guard<std::mutex> hold(all->lock);
  std::unique_ptr<scratch_pool>& pool = all->of[device];
  if (!pool) {
    pool = std::make_unique<scratch_pool>(
        [](size_t bytes) -> void* {
          void* p = nullptr;
          if (hipMalloc(&p, bytes) == hipSuccess) return p;
          (void)hipGetLastError();
          return nullptr;
        },
        [](void* p) { (void)hipFree(p); });
  }
  return *pool;
}

/// Take the scratch of P places in sorted order, and of `groups` groups of both directions.
void take_ops(dyng_hip_graph* g, int64_t P, size_t groups) {
  const int K = g->K;
  op_scratch& o = g->ops;
  // the arrays from `base` on, each from a 256-byte boundary; returns their size
  auto lay_out = [&](unsigned char* base) {
    size_t at = 0;
    auto place = [&](auto*& p, size_t count) {
      p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(base + at);
      at += (count * sizeof(*p) + 255) / 256 * 256;
    };
    const size_t n = static_cast<size_t>(P);
    place(o.keys_b, 2 * n);  // out-row keys, then in-row keys
    place(o.vals_b, 2 * n);
    place(o.group_counts, groups);
    for (int32_t** p : {&o.pend_alive, &o.kill, &o.pend_prefix, &o.kill_prefix, &o.ipend_alive, &o.ikill,
                        &o.ipend_prefix, &o.ikill_prefix}) {
      place(*p, n + 1);
    }
    for (int32_t** p : {&o.pend_w, &o.ipend_w, &o.iop_wold, &o.iop_wnew}) place(*p, n * K);
    place(o.iop_type, n);
    place(o.touched_out, n + 1);
    place(o.touched_in, n + 1);
    place(o.lane_rows, 4 * (n + 1));
    place(o.merge_lists, 2 * kModes * (n + 1));
    place(o.group_entries, groups * kGroupCap);  // last: a small batch fills few places of many
    return at;
  };
  const size_t bytes = lay_out(nullptr);
  if (g->pool == nullptr) {
    scratch_pool& pool = apply_scratch(g->device);
    pool.join();
    g->pool = &pool;
  }
  // a block that a failed apply left with the graph is used again: its work is on the graph's stream
  if (o.block.bytes < bytes) {
    if (o.block.p != nullptr) DYNG_HIP_TRY(hipFree(o.block.p));
    o.block = {};
    o.block = g->pool->take(bytes);
    if (o.block.p == nullptr) {
      throw status_error(DYNG_HIP_OUT_OF_MEMORY, "dyng: out of device memory (" + std::to_string(bytes) + " bytes)");
    }
  }
  lay_out(static_cast<unsigned char*>(o.block.p));
}

/// The apply's work has ended: its scratch goes back.
void give_ops(dyng_hip_graph* g) {
  g->pool->give(g->ops.block);
  g->ops = op_scratch{};
}

/// Groups per direction for N operations, as a power of two's exponent.
int group_bits(int64_t N, int vbits) {
  int lb = 0;
  while (lb < kGroupBits && lb < vbits) {
    const int ops = lb < kGroupBitsFew ? kGroupOpsFew : lb < kGroupBitsSome ? kGroupOpsSome : kGroupOps;
    if ((N / ops) >> (lb + 1) == 0) break;
    ++lb;
  }
  return lb;
}

int op_bits(int64_t N) {
  int b = 1;
  while ((int64_t{1} << b) < N) ++b;
  return b;
}

/// Whether a batch takes the grouped apply: an operation's row within its group, neighbour and
/// batch place fit a word (less its top bit), the groups hold it on average, and no error mode wants
/// the operations checked before anything changes (k_check_pairs reads them in the order of the rows).
bool group_eligible(const dyng_hip_graph* g, int64_t N, int vbits, int lb) {
  return N > 0 && N <= kGroupMost && 2 * vbits - lb + op_bits(N) <= 63 &&
         g->props.on_missing_delete != 1 && g->props.on_existing_insert != 1;
}

out_pair_params out_setup(dyng_hip_graph* g, const batch_scan& sc, const op_layout& L, int64_t N, int64_t P, int vbits,
                          int64_t n_before) {
  out_pair_params op{};
  op.L = L;
  op.keys = g->ops.keys_b;
  op.vals = g->ops.vals_b;
  op.N = N;
  op.stride = P;
  op.vbits = vbits;
  op.K = g->K;
  op.n_before = n_before;
  op.upsert = g->props.on_existing_insert == 0 ? 1 : 0;
  op.ins_w = sc.ins_w;
  op.meta = g->out.meta.p;
  op.base = g->out.base.p;
  op.dead = g->out.dead.p;
  op.nbr = g->out.nbr.p;
  op.w = g->out.w.p;
  op.slot_cap = g->out.slot_cap;
  op.pend_alive = g->ops.pend_alive;
  op.kill = g->ops.kill;
  op.pend_w = g->ops.pend_w;
  op.e_inc = g->ins_inc.p;
  op.e_fw = g->props.allow_parallel ? nullptr : g->ins_fw.p;
  op.iop_type = g->ops.iop_type;
  op.iop_wold = g->ops.iop_wold;
  op.iop_wnew = g->ops.iop_wnew;
  op.mark = g->mark_out.p;
  op.mark_gen = g->mark_generation;
  op.touched = g->ops.touched_out;
  op.row_a = g->row_a_out.p;
  op.row_b = g->row_b_out.p;
  op.ctl = g->ctl.p;
  return op;
}

in_pair_params in_setup(dyng_hip_graph* g, const batch_scan& sc, const op_layout& L, int64_t N, int64_t P, int vbits) {
  in_pair_params ip{};
  ip.L = L;
  ip.ins_w = sc.ins_w;
  ip.upsert = g->props.on_existing_insert == 0 ? 1 : 0;
  ip.keys = g->ops.keys_b + P;
  ip.vals = g->ops.vals_b + P;
  ip.N = N;
  ip.stride = P;
  ip.vbits = vbits;
  ip.K = g->K;
  ip.iop_type = g->ops.iop_type;
  ip.iop_wold = g->ops.iop_wold;
  ip.iop_wnew = g->ops.iop_wnew;
  ip.meta = g->in.meta.p;
  ip.base = g->in.base.p;
  ip.dead = g->in.dead.p;
  ip.nbr = g->in.nbr.p;
  ip.w = g->in.w.p;
  ip.slot_cap = g->in.slot_cap;
  ip.pend_alive = g->ops.ipend_alive;
  ip.kill = g->ops.ikill;
  ip.pend_w = g->ops.ipend_w;
  ip.mark = g->mark_in.p;
  ip.mark_gen = g->mark_generation;
  ip.touched = g->ops.touched_in;
  ip.row_a = g->row_a_in.p;
  ip.row_b = g->row_b_in.p;
  ip.ctl = g->ctl.p;
  return ip;
}

op_layout layout_of(const dyng_hip_graph* g, const batch_scan& sc) {
  op_layout L;
  L.first_is_del = g->props.deletions_first ? 1 : 0;
  L.num_first = L.first_is_del ? sc.num_del : sc.num_ins;
  L.num_second = L.first_is_del ? sc.num_ins : sc.num_del;
  L.stride = g->props.directed ? 1 : 2;
  return L;
}

/// The rows' update behind a device-wide sort of the operations: the error modes, batches past the
/// groups' limits, and batches with more operations on one row than a group takes.
void rows_sorted(dyng_hip_graph* g, const batch_scan& sc, const op_layout& L, int64_t N, int vbits, int64_t n_before,
                 hipStream_t s, dyng_hip_apply_summary* out, hipEvent_t wait, apply_pending& ap) {
  apply_control* hc = g->host_ctl.p;
  apply_control* dc = g->ctl.p;
  const int K = g->K;
  const int64_t n_after = sc.n_after;
  const int32_t *ins_src = sc.ins_src, *ins_dst = sc.ins_dst, *del_src = sc.del_src, *del_dst = sc.del_dst;
  g->keys_a.reserve(2 * N);
  g->vals_a.reserve(2 * N);
  mark_stage(g, 2, s);
  hipLaunchKernelGGL(k_make_ops, dim3(blocks_for(N)), dim3(kBlock), 0, s, L, ins_src, ins_dst, del_src, del_dst,
                     g->props.directed, g->props.on_self_loop == 1 ? 1 : 0, n_after, vbits, g->keys_a.p,
                     g->vals_a.p, g->del_src.p, g->del_dst.p, g->ins_src.p, g->ins_dst.p, g->ins_inc.p,
                     g->props.allow_parallel ? nullptr : g->ins_fw.p, K, g->props.on_missing_delete == 1 ? 1 : 0,
                     dc);
  DYNG_HIP_TRY(hipGetLastError());
  mark_stage(g, 3, s);
  // one stable sort of both directions' keys (2N of them, 2 * vbits + 1 bits): one sort of 2N
  // keys costs little more than one of N, since rocPRIM's small-size path is launch-bound
  sort_pairs(g->sort_tmp, g->keys_a.p, g->ops.keys_b, g->vals_a.p, g->ops.vals_b, 2 * N, 2 * vbits + 1, s);
  hipLaunchKernelGGL(k_untag, dim3(std::min<unsigned>(blocks_for(2 * N), 1024)), dim3(kBlock), 0, s, g->ops.keys_b,
                     2 * N, vbits);
  if (g->props.on_missing_delete == 1 || g->props.on_existing_insert == 1) {
    // the error modes: every operation checked before anything changes (one more launch and
    // synchronization, only in these modes)
    hipLaunchKernelGGL(k_check_pairs, dim3(blocks_for(N)), dim3(kBlock), 0, s, L, g->ops.keys_b, g->ops.vals_b, N,
                       vbits, n_before, g->out.meta.p, g->out.base.p, g->out.nbr.p,
                       g->props.on_missing_delete == 1 ? 1 : 0, g->props.on_existing_insert == 1 ? 1 : 0, dc);
    DYNG_HIP_TRY(hipGetLastError());
    DYNG_HIP_TRY(hipMemcpyAsync(&hc->first_error, &dc->first_error, sizeof(hc->first_error),
                                hipMemcpyDeviceToHost, s));
    DYNG_HIP_TRY(hipStreamSynchronize(s));
    if (hc->first_error != kNoError) report_batch_error(g, sc, L, hc->first_error, s);
  }
  mark_stage(g, 4, s);
  const out_pair_params op = out_setup(g, sc, L, N, N, vbits, n_before);
  const in_pair_params ip = in_setup(g, sc, L, N, N, vbits);
  const unsigned pair_groups = blocks_for(N + 1);
  if (!g->props.allow_parallel) {
    // a simple graph: the in-row pass replays the operations itself, in the same launch
    mark_stage(g, 5, s);
    hipLaunchKernelGGL(k_pairs_simple, dim3(2 * pair_groups), dim3(kBlock), 0, s, op, ip,
                       static_cast<int>(pair_groups));
    DYNG_HIP_TRY(hipGetLastError());
    mark_stage(g, 6, s);
    mark_stage(g, 7, s);
  } else {
    mark_stage(g, 5, s);
    hipLaunchKernelGGL(k_out_pairs, dim3(pair_groups), dim3(kBlock), 0, s, op);
    DYNG_HIP_TRY(hipGetLastError());
    mark_stage(g, 6, s);
    mark_stage(g, 7, s);
    hipLaunchKernelGGL(k_in_pairs, dim3(pair_groups), dim3(kBlock), 0, s, ip);
    DYNG_HIP_TRY(hipGetLastError());
  }
  mark_stage(g, 8, s);
  exclusive_scan4(g->scan_tmp, g->ops.pend_alive, g->ops.kill, g->ops.ipend_alive, g->ops.ikill, g->ops.pend_prefix,
                  g->ops.kill_prefix, g->ops.ipend_prefix, g->ops.ikill_prefix, N + 1, s);
  mark_stage(g, 9, s);
  // ---- plan the merges: each row's mode, and the staging and tail slots they take ----
  if (wait != nullptr) DYNG_HIP_TRY(hipStreamWaitEvent(s, wait, 0));  // before the rows change
  ap.speculative = N <= kSpeculativeOps;
  if (ap.speculative) {
    merges_speculative(g, N, vbits, s);
  } else {
    merges_exact(g, N, vbits, s, out, kPlanNone);
  }
}

/// A batch whose groups could not take it (more operations on one row than a group's room) again
/// behind the device-wide sort; nothing changed yet. The graph's next batches go there directly: a
/// stream with such a batch has more of them, and each would pay for the attempt.
void resort(dyng_hip_graph* g, const batch_scan& sc, int64_t n_before, hipStream_t s, dyng_hip_apply_summary* out,
            apply_pending& ap) {
  g->group_pause = kGroupPause;
  begin_apply(g, sc, 0, s);
  ap.P = ap.N;
  rows_sorted(g, sc, layout_of(g, sc), ap.N, ap.vbits, n_before, s, out, ap.wait, ap);
}

/// The rows' update by groups (see k_group_front).
void rows_grouped(dyng_hip_graph* g, const batch_scan& sc, const op_layout& L, int64_t N, int64_t P, int vbits, int lb,
                  int64_t n_before, hipStream_t s, dyng_hip_apply_summary* out, hipEvent_t wait, apply_pending& ap) {
  apply_control* dc = g->ctl.p;
  const int groups = 1 << lb;
  mark_stage(g, 2, s);
  front_params f{};
  f.L = L;
  f.ins_src = sc.ins_src;
  f.ins_dst = sc.ins_dst;
  f.del_src = sc.del_src;
  f.del_dst = sc.del_dst;
  f.directed = g->props.directed;
  f.drop_self_loops = g->props.on_self_loop == 1 ? 1 : 0;
  f.n_after = sc.n_after;
  f.vbits = vbits;
  f.ebits = op_bits(N);
  f.lb = lb;
  f.K = g->K;
  f.groups = groups;
  f.room = kGroupCap;
  f.entries = g->ops.group_entries;
  f.counts = g->ops.group_counts;
  f.e_del_src = g->del_src.p;
  f.e_del_dst = g->del_dst.p;
  f.e_ins_src = g->ins_src.p;
  f.e_ins_dst = g->ins_dst.p;
  f.e_inc = g->ins_inc.p;
  f.e_fw = g->props.allow_parallel ? nullptr : g->ins_fw.p;
  f.ctl = dc;
  // one operation per thread while that fills the chip at most once; eight above, so that a
  // workgroup reserves a group's places for several operations at a time
  if (N <= 256 * 1024) {
    hipLaunchKernelGGL(k_group_front<1>, dim3(blocks_for(N, 1024)), dim3(1024), 0, s, f);
  } else {
    hipLaunchKernelGGL(k_group_front<8>, dim3(blocks_for(N, 8 * 1024)), dim3(1024), 0, s, f);
  }
  DYNG_HIP_TRY(hipGetLastError());
  mark_stage(g, 3, s);
  mark_stage(g, 4, s);
  group_params gp{};
  gp.entries = g->ops.group_entries;
  gp.counts = g->ops.group_counts;
  gp.groups = groups;
  gp.room = f.room;
  gp.vbits = vbits;
  gp.ebits = f.ebits;
  gp.lb = lb;
  uint32_t inverse = kGroupHash;  // Newton's iteration: right modulo 2^3, then 2^6, ... 2^48
  for (int i = 0; i < 4; ++i) inverse *= 2u - kGroupHash * inverse;
  gp.inverse = inverse;
  gp.keys = g->ops.keys_b;
  gp.vals = g->ops.vals_b;
  gp.P = P;
  gp.out = out_setup(g, sc, L, N, P, vbits, n_before);
  gp.in = in_setup(g, sc, L, N, P, vbits);
  gp.merge_out = merge_setup(g, true, P, vbits);
  gp.merge_in = merge_setup(g, false, P, vbits);
  gp.pend_prefix_out = g->ops.pend_prefix;
  gp.kill_prefix_out = g->ops.kill_prefix;
  gp.pend_prefix_in = g->ops.ipend_prefix;
  gp.kill_prefix_in = g->ops.ikill_prefix;
  gp.ctl = dc;
  mark_stage(g, 5, s);
  if (!g->props.allow_parallel) {
    hipLaunchKernelGGL(k_group_pairs<kGroupsBoth>, dim3(static_cast<unsigned>(2 * groups)), dim3(kGroupBlock), 0, s, gp);
    mark_stage(g, 6, s);
    mark_stage(g, 7, s);
  } else {
    hipLaunchKernelGGL(k_group_pairs<kGroupsOut>, dim3(static_cast<unsigned>(groups)), dim3(kGroupBlock), 0, s, gp);
    mark_stage(g, 6, s);
    mark_stage(g, 7, s);
    hipLaunchKernelGGL(k_group_pairs<kGroupsIn>, dim3(static_cast<unsigned>(groups)), dim3(kGroupBlock), 0, s, gp);
  }
  DYNG_HIP_TRY(hipGetLastError());
  mark_stage(g, 8, s);
  mark_stage(g, 9, s);
  ap.speculative = N <= kSpeculativeOps;
  if (wait != nullptr) DYNG_HIP_TRY(hipStreamWaitEvent(s, wait, 0));  // before the rows change
  if (ap.speculative) {
    merges_queued(g, P, vbits, s);
    return;
  }
  merges_exact(g, P, vbits, s, out, kPlanDone);
  if (g->host_ctl.p->miss != 0) resort(g, sc, n_before, s, out, ap);
}

apply_pending apply_launch(dyng_hip_graph* g, const batch_scan& sc, hipStream_t s, dyng_hip_apply_summary* out,
                           hipEvent_t wait) {
  const int K = g->K;
  // G_t as the batch found it (the repair of a result one apply behind reads it)
  g->last.valid = false;
  g->last.max_weight.assign(K, 1);
  g->last.batch_wmin.assign(K, 1);
  g->last.wsum.assign(K, 0);
  for (int k = 0; k < K; ++k) {
    g->last.max_weight[k] = std::max<int64_t>(std::max<int64_t>(sc.wmax[k], 1), g->wmax[k]);
    g->last.batch_wmin[k] = sc.wmin[k];
    g->last.wsum[k] = g->wsum[k];
  }
  g->last.m = g->m;
  g->last.n = g->n;
  g->last.num_ins = sc.num_ins;
  const int64_t num_ins = sc.num_ins, num_del = sc.num_del;
  const int64_t n_after = sc.n_after;
  const int64_t n_before = g->n;
  const int stride = g->props.directed ? 1 : 2;
  const int64_t N = (num_ins + num_del) * stride;
  if (N >= (int64_t{1} << 31)) fail(DYNG_HIP_NOT_SUPPORTED, "dyng: batch too large");
  grow_vertices(g, n_after, s);
  // deletions below the old vertex count that name vertices of the growth are fine; ids in the
  // batch >= n_after only occur in deletions (handled in Step 0)
  const int vbits = bits_for(std::max<int64_t>(n_after, 1));
  apply_pending ap;
  ap.n_before = n_before;
  ap.N = N;
  ap.vbits = vbits;
  ap.wait = wait;
  const op_layout L = layout_of(g, sc);
  g->num_del_slots = num_del * stride;
  g->num_ins_slots = num_ins * stride;
  g->del_src.reserve(g->num_del_slots);
  g->del_dst.reserve(g->num_del_slots);
  g->ins_src.reserve(g->num_ins_slots);
  g->ins_dst.reserve(g->num_ins_slots);
  g->ins_inc.reserve(g->num_ins_slots * K);
  if (!g->props.allow_parallel) g->ins_fw.reserve(g->num_ins_slots * K);
  // P: places of the sorted operations (the grouped apply leaves one behind each group)
  const int lb = group_bits(N, vbits);
  const bool grouped = group_eligible(g, N, vbits, lb) && g->group_pause == 0;
  if (g->group_pause > 0) g->group_pause -= 1;
  const int64_t P = ap.P = grouped ? N + (int64_t{1} << lb) : N;
  take_ops(g, P, grouped ? size_t{2} << lb : 0);
  g->row_a_out.reserve(g->n_cap);
  g->row_b_out.reserve(g->n_cap);
  g->row_a_in.reserve(g->n_cap);
  g->row_b_in.reserve(g->n_cap);
  if (++g->mark_generation == INT32_MAX) {
    fill<int32_t>(g->mark_out.p, g->n_cap, 0, s);
    fill<int32_t>(g->mark_in.p, g->n_cap, 0, s);
    g->mark_generation = 1;
  }
  begin_apply(g, sc, grouped ? 2 << lb : 0, s);
  if (N > 0) {
    if (grouped) {
      rows_grouped(g, sc, L, N, P, vbits, lb, n_before, s, out, wait, ap);
    } else {
      rows_sorted(g, sc, L, N, vbits, n_before, s, out, wait, ap);
    }
  }
  if (wait != nullptr) DYNG_HIP_TRY(hipStreamWaitEvent(s, wait, 0));
  // from here on the graph has the batch's vertices (work queued behind reads them)
  g->n = n_after;
  return ap;
}

void apply_finish(dyng_hip_graph* g, const batch_scan& sc, apply_pending& ap, hipStream_t s,
                  dyng_hip_apply_summary* out) {
  const int K = g->K;
  apply_control* hc = g->host_ctl.p;
  apply_control* dc = g->ctl.p;
  const int64_t n_before = ap.n_before;
  const int64_t n_after = g->n;
  if (!ap.published) DYNG_HIP_TRY(hipMemcpyAsync(hc, dc, sizeof(apply_control), hipMemcpyDeviceToHost, s));
  DYNG_HIP_TRY(hipStreamSynchronize(s));
  if (hc->miss != 0 && hc->error_bits == 0) {
    resort(g, sc, n_before, s, out, ap);
    DYNG_HIP_TRY(hipMemcpyAsync(hc, dc, sizeof(apply_control), hipMemcpyDeviceToHost, s));
    DYNG_HIP_TRY(hipStreamSynchronize(s));
    ap.replanned = true;
  }
  if (ap.speculative && hc->hold != 0 && hc->error_bits == 0) {
    // the arenas could not take the merges as the device planned them: plan again with the
    // host's compaction and staging growth (nothing was merged; the rows are as the pairing left
    // them)
    hc->hold = 0;
    DYNG_HIP_TRY(hipMemcpyAsync(&dc->hold, &hc->hold, sizeof(int), hipMemcpyHostToDevice, s));
    merges_exact(g, ap.P, ap.vbits, s, out, kPlanAgain);
    if (ap.wait != nullptr) DYNG_HIP_TRY(hipStreamWaitEvent(s, ap.wait, 0));
    DYNG_HIP_TRY(hipMemcpyAsync(hc, dc, sizeof(apply_control), hipMemcpyDeviceToHost, s));
    DYNG_HIP_TRY(hipStreamSynchronize(s));
    ap.replanned = true;
  }
  give_ops(g);
  if (hc->error_bits != 0) {
    g->n = n_before;
    throw status_error(DYNG_HIP_DEVICE_ERROR, "dyng: the device apply reported an internal error",
                       static_cast<uint32_t>(hc->error_bits));
  }
  g->m += static_cast<int64_t>(hc->inserted_edges) - static_cast<int64_t>(hc->deleted_edges);
  for (int k = 0; k < K; ++k) g->wmin[k] = std::min<int64_t>(g->wmin[k], sc.wmin[k]);
  g->out.tail = hc->tail_out;
  g->in.tail = hc->tail_in;
  g->out.garbage += hc->garbage_out;
  g->in.garbage += hc->garbage_in;
  bool dirty = false;
  for (int k = 0; k < K; ++k) {
    const int64_t target = hc->col_max[k];
    const int64_t before = target == g->wmax[k] ? g->wmax_count[k] : 0;
    g->wsum[k] += hc->col_dsum[k];
    g->wmax[k] = target;
    g->wmax_count[k] = before + hc->col_dcount[k];
    if (g->wmax_count[k] <= 0) dirty = true;
  }
  g->version += 1;
  if (out != nullptr) {
    out->inserted_edges = static_cast<int64_t>(hc->inserted_edges);
    out->updated_edges = static_cast<int64_t>(hc->updated_edges);
    out->deleted_edges = static_cast<int64_t>(hc->deleted_edges);
    out->ignored_deletions = static_cast<int64_t>(hc->ignored_deletions);
    out->dropped_self_loops = static_cast<int64_t>(hc->dropped_self_loops);
    out->ignored_insertions = static_cast<int64_t>(hc->ignored_insertions);
    out->inserted_vertices = n_after - n_before;
    out->num_vertices_after = n_after;
    out->relocated_rows = static_cast<int64_t>(hc->relocated_rows);
    stage_times(g, ap.N > 0 && hc->error_bits == 0, out);
    g->last.summary = *out;
  }
  g->last.valid = true;
  // the last edge of the largest weight left: recompute the column summaries (reuses the control
  // block, so only after the counters above were read)
  if (dirty) recompute_columns(g, s);
}

void apply_scanned(dyng_hip_graph* g, const batch_scan& sc, hipStream_t s, dyng_hip_apply_summary* out,
                   hipEvent_t wait) {
  apply_pending ap = apply_launch(g, sc, s, out, wait);
  apply_finish(g, sc, ap, s, out);
}


}  // namespace dyng_hip

// ---------------------------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------------------------

using namespace dyng_hip;

extern "C" int dyng_hip_graph_create_from_edges(int device, const dyng_hip_graph_props* props, int64_t n,
                                                int64_t count, int32_t num_weights, const int32_t* src,
                                                const int32_t* dst, const int32_t* w, int32_t from_device,
                                                void* stream, dyng_hip_graph** out) {
  return guarded([&] {
    if (out == nullptr) fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: null output handle");
    for (int64_t i = 0; !from_device && i < count; ++i) {
      if (src[i] < 0 || src[i] >= n || dst[i] < 0 || dst[i] >= n) {
        fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: edge " + std::to_string(i) + " (" + std::to_string(src[i]) + ", " +
                                            std::to_string(dst[i]) + ") is out of range [0, " + std::to_string(n) + ")");
      }
    }
    *out = create_from_edge_list(device, props, n, count, num_weights, src, dst, w, from_device, as_stream(stream));
  });
}

extern "C" int dyng_hip_graph_create(int device, const dyng_hip_graph_props* props, int64_t n, int64_t m,
                                     int32_t num_weights, const int64_t* row_ptr, const int32_t* col,
                                     const int32_t* w, int32_t from_device, void* stream, dyng_hip_graph** out) {
  return guarded([&] {
    if (from_device) fail(DYNG_HIP_NOT_SUPPORTED, "dyng: graph_create takes host rows (use create_from_edges)");
    if (n < 0 || m < 0) fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: negative sizes");
    if (row_ptr[0] != 0 || row_ptr[n] != m) fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: row offsets do not span the edges");
    std::vector<int32_t> src(static_cast<size_t>(m));
    std::vector<int32_t> wl(static_cast<size_t>(m) * num_weights);
    for (int64_t u = 0; u < n; ++u) {
      if (row_ptr[u + 1] < row_ptr[u]) fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: row offsets decrease");
      for (int64_t e = row_ptr[u]; e < row_ptr[u + 1]; ++e) src[e] = static_cast<int32_t>(u);
    }
    for (int64_t e = 0; e < m; ++e) {
      if (col[e] < 0 || col[e] >= n) fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: neighbour out of range");
      for (int k = 0; k < num_weights; ++k) wl[e * num_weights + k] = w[k * m + e];
    }
    *out = create_from_edge_list(device, props, n, m, num_weights, src.data(), col, wl.data(), 0, as_stream(stream));
  });
}

extern "C" int dyng_hip_graph_destroy(dyng_hip_graph* g) {
  return guarded([&] { delete g; });
}

extern "C" int dyng_hip_graph_num_vertices(const dyng_hip_graph* g, int64_t* n) {
  return guarded([&] { *n = g->n; });
}

extern "C" int dyng_hip_graph_num_edges(const dyng_hip_graph* g, int64_t* m) {
  return guarded([&] { *m = g->m; });
}

extern "C" int dyng_hip_graph_version(const dyng_hip_graph* g, uint64_t* version) {
  return guarded([&] { *version = g->version; });
}

extern "C" int dyng_hip_graph_column(const dyng_hip_graph* g, int32_t k, int64_t* max_weight, int64_t* weight_sum) {
  return guarded([&] {
    if (k < 0 || k >= g->K) fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: objective out of range");
    *max_weight = g->wmax[k];
    *weight_sum = g->wsum[k];
  });
}

extern "C" int dyng_hip_graph_download(const dyng_hip_graph* g, int64_t* row_ptr, int32_t* col, int32_t* w) {
  return guarded([&] {
    scoped_device guard(g->device);
    DYNG_HIP_TRY(hipDeviceSynchronize());
    copy_rows_to_host(g->out, g->n, g->K, row_ptr, col, w);
  });
}

extern "C" int dyng_hip_graph_download_in(const dyng_hip_graph* g, int64_t* row_ptr, int32_t* col, int32_t* w) {
  return guarded([&] {
    scoped_device guard(g->device);
    DYNG_HIP_TRY(hipDeviceSynchronize());
    copy_rows_to_host(g->in, g->n, g->K, row_ptr, col, w);
  });
}

extern "C" int dyng_hip_graph_apply(dyng_hip_graph* g, const dyng_hip_batch* batch, void* stream,
                                    dyng_hip_apply_summary* summary) {
  return guarded([&] {
    if (g == nullptr) fail(DYNG_HIP_INVALID_ARGUMENT, "dyng: null graph");
    scoped_device guard(g->device);
    dyng_hip_apply_summary tmp{};
    batch_scan sc;
    scan_batch(g, batch, as_stream(stream), sc);
    apply_scanned(g, sc, as_stream(stream), &tmp);
    if (summary != nullptr) *summary = tmp;
  });
}

extern "C" int dyng_hip_graph_changes(const dyng_hip_graph* g, dyng_hip_changes* out) {
  return guarded([&] {
    out->del_src = g->del_src.p;
    out->del_dst = g->del_dst.p;
    out->num_del = g->num_del_slots;
    out->ins_src = g->ins_src.p;
    out->ins_dst = g->ins_dst.p;
    out->ins_increased = g->ins_inc.p;
    out->num_ins = g->num_ins_slots;
    out->num_weights = g->K;
  });
}
