// Device helpers shared by the cbx kernels (wave64 scans, block scans,
// error checks).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "cbx_internal.h"

#define CBX_HIP(call)                                                                  \
  do {                                                                                 \
    hipError_t e_ = (call);                                                            \
    if (e_ != hipSuccess)                                                              \
      return ::cbx::set_error(CBX_ERR_HIP, "%s failed: %s (%s:%d)", #call,            \
                              hipGetErrorString(e_), __FILE__, __LINE__);             \
  } while (0)

namespace cbx {

constexpr int kWave = 64;

// Index of this wave in a 1-D or 2-D grid of 1-D blocks (a 2-D grid keeps
// the per-dimension work-item count of wave-per-column launches below 2^32).
__device__ __forceinline__ int64_t global_wave() {
  return (((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * blockDim.x + threadIdx.x) / kWave;
}

// Grid with one wave per item for blocks of `bs` threads.
inline dim3 wave_grid(int64_t nwaves, int bs = 256) {
  int64_t blocks = (nwaves * kWave + bs - 1) / bs;
  if (blocks < 1) blocks = 1;
  const int64_t X = (int64_t)1 << 22;
  return blocks <= X ? dim3((unsigned)blocks) : dim3((unsigned)X, (unsigned)((blocks + X - 1) / X));
}

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & (kWave - 1)); }
__device__ __forceinline__ int wave_id() { return (int)(threadIdx.x >> 6); }

// v + the value of the lane that the DPP control names (0 where it names none
// or the row mask leaves the lane out).
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_add(int v) {
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}

// Inclusive prefix sum over the 64 lanes of a wave (all must be active): row
// shifts by 1, 2, 4 and 8 within rows of 16 lanes, then the rows' last lanes
// broadcast to the rows after them.  Six VALU instructions; shuffles went
// through LDS and a compare each step.
__device__ __forceinline__ int wave_incl_scan(int v) {
  v = dpp_add<0x111, 0xf>(v);
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);
  v = dpp_add<0x143, 0xc>(v);
  return v;
}

// Holds v in a register at this point, so that a load of v (and of what its
// address comes from) is issued before it even where v is only used under a
// condition: the compiler otherwise sinks the load into the branch, and a
// lane's independent loads then wait for each other.
template <class T>
__device__ __forceinline__ void pin(T& v) {
  if constexpr (sizeof(T) < 4) {
    uint32_t x = (uint32_t)v;
    asm volatile("" : "+v"(x));
    v = (T)x;
  } else {
    asm volatile("" : "+v"(v));
  }
}

// The wave's index in its workgroup, in a scalar register.
__device__ __forceinline__ int wave_id_uniform() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

__device__ __forceinline__ long long wave_sum_ll(long long v) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, kWave);
  return v;
}

// Exclusive prefix sum over a block of NT threads; `wsum` is LDS scratch of
// NT/64 ints.  Returns this thread's exclusive prefix and the block total.
// Contains barriers: every thread of the block must call it.
template <int NT>
__device__ __forceinline__ int block_excl_scan(int v, int* wsum, int& total) {
  constexpr int NW = NT / kWave;
  const int lane = lane_id(), w = wave_id_uniform();
  const int inc = wave_incl_scan(v);
  if (lane == kWave - 1) wsum[w] = inc;
  __syncthreads();
  const int x = wave_incl_scan(lane < NW ? wsum[lane] : 0);  // every wave scans the waves' sums
  const int base = w ? __builtin_amdgcn_readlane(x, w - 1) : 0;
  total = __builtin_amdgcn_readlane(x, NW - 1);
  __syncthreads();
  return base + inc - v;
}

template <int CTRL, int ROWS>
__device__ __forceinline__ long long dpp_add_ll(long long v) {
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)v, CTRL, ROWS, 0xf, false);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, ROWS, 0xf, false);
  return v + (long long)(((unsigned long long)hi << 32) | lo);
}

__device__ __forceinline__ long long wave_incl_scan_ll(long long v) {
  v = dpp_add_ll<0x111, 0xf>(v);
  v = dpp_add_ll<0x112, 0xf>(v);
  v = dpp_add_ll<0x114, 0xf>(v);
  v = dpp_add_ll<0x118, 0xf>(v);
  v = dpp_add_ll<0x142, 0xa>(v);
  v = dpp_add_ll<0x143, 0xc>(v);
  return v;
}

__device__ __forceinline__ long long readlane_ll(long long v, int lane) {
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), lane);
  return (long long)(((unsigned long long)hi << 32) | lo);
}

// 64-bit exclusive prefix sum over a block of NT threads (wsum: NT/64 slots).
template <int NT>
__device__ __forceinline__ long long block_excl_scan_ll(long long v, long long* wsum, long long& total) {
  constexpr int NW = NT / kWave;
  const int lane = lane_id(), w = wave_id_uniform();
  const long long inc = wave_incl_scan_ll(v);
  if (lane == kWave - 1) wsum[w] = inc;
  __syncthreads();
  const long long x = wave_incl_scan_ll(lane < NW ? wsum[lane] : 0);
  const long long base = w ? readlane_ll(x, w - 1) : 0;
  total = readlane_ll(x, NW - 1);
  __syncthreads();
  return base + inc - v;
}

// Sum over a block of NT threads (result valid in every thread).
template <int NT>
__device__ __forceinline__ long long block_sum_ll(long long v, long long* wsum) {
  constexpr int NW = NT / kWave;
  v = wave_sum_ll(v);
  if (lane_id() == 0) wsum[wave_id()] = v;
  __syncthreads();
  long long t = 0;
#pragma unroll
  for (int i = 0; i < NW; ++i) t += wsum[i];
  __syncthreads();
  return t;
}

// Adds two per-thread counts into *pa and *pb with one device atomic each per
// workgroup (same-address device atomics serialise, so reduce first).
// Contains a barrier: every thread of the workgroup must call it.
template <int NT>
__device__ __forceinline__ void block_add_counts(long long a, long long b, unsigned long long* pa,
                                                 unsigned long long* pb) {
  __shared__ long long s[2][NT / kWave];
  a = wave_sum_ll(a);
  b = wave_sum_ll(b);
  if (lane_id() == 0) {
    s[0][wave_id()] = a;
    s[1][wave_id()] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    long long x = 0, y = 0;
    for (int w = 0; w < NT / kWave; ++w) {
      x += s[0][w];
      y += s[1][w];
    }
    if (x) atomicAdd(pa, (unsigned long long)x);
    if (y) atomicAdd(pb, (unsigned long long)y);
  }
}

}  // namespace cbx
