// Stand-ins for what device code uses of HIP, so that a host compiler can build a kernel whose workgroups
// are single threads of the host: each workgroup's place, its LDS (per thread of the host) and the atomics.
// Lane-to-lane moves fold into the one lane.
#pragma once

#include <cstdint>

#define __device__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static thread_local
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_load(p, order, scope) __atomic_load_n(p, __ATOMIC_SEQ_CST)
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n(p, v, __ATOMIC_SEQ_CST)
#define __hip_atomic_fetch_add(p, v, order, scope) __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST)

struct host_dim {
  unsigned int x;
};
inline thread_local host_dim blockIdx{0}, threadIdx{0}, blockDim{1}, gridDim{1};

/// The real-time counter, the pause of a poll and the workgroup barrier: the program that includes this
/// defines them.
unsigned long long __builtin_amdgcn_s_memrealtime();
void __builtin_amdgcn_s_sleep(int);
void __syncthreads();

inline void __builtin_amdgcn_s_waitcnt(int) {}
inline void __builtin_amdgcn_fence(int, const char*) {}
inline int __builtin_amdgcn_readfirstlane(int v) { return v; }
inline int __builtin_amdgcn_readlane(int v, int) { return v; }
inline int __builtin_amdgcn_update_dpp(int old, int, int, int, int, bool) { return old; }
inline unsigned int __lane_id() { return 0; }
inline unsigned long long __ballot(bool p) { return p ? 1 : 0; }
inline int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
inline int __ffsll(long long v) { return __builtin_ffsll(v); }
template <class T>
T __shfl_xor(T v, int) {
  return v;
}
template <class T>
T atomicAdd(T* p, T v) {
  return __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST);
}
inline int __syncthreads_count(int p) { return p; }
