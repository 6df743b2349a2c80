// Scans over a 256-thread block, shared by the dispatch and permute kernels.
#pragma once
#include <hip/hip_runtime.h>

namespace moe {

// Exclusive scan of 256 ints held one per thread; returns the exclusive prefix
// and the block total.  Wave scans by __shfl_up, then a 4-entry carry.
__device__ __forceinline__ int block_exclusive_scan(int v, int* sh4, int& total) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int n = __shfl_up(inc, o, 64);
    if (lane >= o) inc += n;
  }
  if (lane == 63) sh4[wave] = inc;
  __syncthreads();
  int carry = 0;
  for (int w = 0; w < wave; ++w) carry += sh4[w];
  total = sh4[0] + sh4[1] + sh4[2] + sh4[3];
  __syncthreads();
  return carry + inc - v;
}

// Exclusive scan of cnt[0..E) into offs[0..E] held in LDS (E <= 1024).
__device__ __forceinline__ void lds_offsets(const int* __restrict__ cnt, int E, int* offs,
                                            int* sh4) {
  const int tid = threadIdx.x;
  int v[4];
  int s = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int idx = tid * 4 + i;
    v[i] = idx < E ? cnt[idx] : 0;
    s += v[i];
  }
  int total;
  int ex = block_exclusive_scan(s, sh4, total);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int idx = tid * 4 + i;
    if (idx < E) offs[idx] = ex;
    ex += v[i];
  }
  if (tid == 0) offs[E] = total;
}

}  // namespace moe
