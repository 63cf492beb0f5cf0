// Device-side reduction helpers shared by the HIP translation units of
// libcfdla.  A reducing kernel sums its values per block (wave64 shuffle
// tree, then LDS across the 4 waves of a 256-thread block) and stores one
// partial per block with a plain store.  A single-block kernel launched next
// on the same stream sums the partials in block order and advances the
// solver scalars.  No atomics, no fences: the kernel boundary orders the
// partial stores before their loads, and the fixed summation order makes
// results bitwise reproducible run to run.
#pragma once

#include <hip/hip_runtime.h>

#include "internal.hpp"

namespace cfdla {

// v of the lane CTRL names within its row of 16 (a DPP move: VALU latency, no
// LDS crossbar).
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// v of this lane plus v of the lane W (16 or 32) away.
template <int W>
__device__ __forceinline__ auto lane_swap(unsigned v) {
  if constexpr (W == 32) return __builtin_amdgcn_permlane32_swap(v, v, false, false);
  else return __builtin_amdgcn_permlane16_swap(v, v, false, false);
}
template <int W>
__device__ __forceinline__ double add_across(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const auto lo = lane_swap<W>((unsigned)b), hi = lane_swap<W>((unsigned)(b >> 32));
  return __builtin_bit_cast(double, ((unsigned long long)hi[0] << 32) | lo[0]) +
         __builtin_bit_cast(double, ((unsigned long long)hi[1] << 32) | lo[1]);
}
template <int W>
__device__ __forceinline__ double max_across(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const auto lo = lane_swap<W>((unsigned)b), hi = lane_swap<W>((unsigned)(b >> 32));
  return fmax(__builtin_bit_cast(double, ((unsigned long long)hi[0] << 32) | lo[0]),
              __builtin_bit_cast(double, ((unsigned long long)hi[1] << 32) | lo[1]));
}
template <int W>
__device__ __forceinline__ float add_across(float v) {
  const auto p = lane_swap<W>(__builtin_bit_cast(unsigned, v));
  const unsigned a = p[0], b = p[1];  // (a bit cast of a vector's element reads its first one)
  return __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
}

// v is computed, and loaded, by here.
template <typename T>
__device__ __forceinline__ void pin(T &v) {
  asm volatile("" : "+v"(v));
}

// Sum of a wavefront, in every lane: the xor tree 32, 16, 8, 4, 2, 1 without
// LDS traffic.  The lane swaps of gfx950 add the halves (lane ^ 32) and then
// the rows (lane ^ 16); within a row the partial sums repeat with the period
// just added, so a rotation by 8, 4, 2, 1 brings the xor partner's value.
// Every addition pairs the same two values as __shfl_xor does, so the sum is
// the same bit for bit.  A tree of 6 shuffles is 12 dependent ds_bpermutes,
// about 0.5 us of latency (Jacobi-PCG on 16,384 rows, two reductions per
// iteration: 10.5 -> 8.8 ms for 750 iterations; 600 networks of 30-700 nodes
// with their adjoint: 6.41 -> 5.75 ms).
__device__ __forceinline__ double wave_sum(double v) {
  v = add_across<32>(v);
  v = add_across<16>(v);
  v += dpp_move<0x128>(v);  // row_ror:8
  v += dpp_move<0x124>(v);  // row_ror:4
  v += dpp_move<0x122>(v);  // row_ror:2
  v += dpp_move<0x121>(v);  // row_ror:1
  return v;
}

// Every thread of the block must call this; partial i of this block lands at
// partials[i * kMaxBlocks + blockIdx.x].
template <int NV>
__device__ __forceinline__ void block_partials(double (&v)[NV], double *partials) {
  __shared__ double sh[NV][kBlock / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    double t = wave_sum(v[i]);
    if (lane == 0) sh[i][wid] = t;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      double t = 0.0;
#pragma unroll
      for (int w = 0; w < kBlock / 64; ++w) t += sh[i][w];
      partials[i * kMaxBlocks + blockIdx.x] = t;
    }
  }
}

// One block of kBlock threads sums nblocks partials per value; the totals are
// valid in thread 0.
template <int NV>
__device__ __forceinline__ void sum_partials(int nblocks, const double *partials, double (&tot)[NV]) {
  __shared__ double sh[NV][kBlock / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  double acc[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) acc[i] = 0.0;
  // unrolled so up to 8 loads per value are in flight (same summation order)
#pragma unroll 8
  for (int b = threadIdx.x; b < nblocks; b += kBlock) {
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] += partials[i * kMaxBlocks + b];
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    double t = wave_sum(acc[i]);
    if (lane == 0) sh[i][wid] = t;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) t += sh[i][w];
    tot[i] = t;
  }
}

inline int blocks_for(int64_t work_items, int per_block) {
  int64_t b = (work_items + per_block - 1) / per_block;
  if (b < 1) b = 1;
  if (b > kGridCap) b = kGridCap;
  return (int)b;
}

}  // namespace cfdla
