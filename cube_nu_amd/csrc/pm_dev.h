// pm_dev.h -- device helpers shared by the particle-mesh kernels.
#pragma once
#include "pm.h"

namespace cube {
namespace {

constexpr float kFixF = 4294967296.0f;  // 2^32: weights are < 0.43, so w * 2^32 fits a u32

// FP32 TSC weight product as a 2^-32 fixed-point integer (round to nearest).
__device__ inline unsigned long long fix32(float cw) { return (unsigned long long)__float2uint_rn(cw * kFixF); }

__device__ inline int floor_div(int a, int b) {
  int q = a / b;
  if ((a % b != 0) && ((a < 0) != (b < 0))) --q;
  return q;
}

template <int IZ>
using XT = typename XP<IZ>::T;


// Exclusive block scan of cnt[0..n) into pre[0..n] (pre[n] = total), n <= 1024.
__device__ inline void block_scan(const int* cnt, int* pre, int n, int* wsum) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int b0 = 4 * threadIdx.x;
  int loc[4], s = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    loc[k] = (b0 + k < n) ? cnt[b0 + k] : 0;
    s += loc[k];
  }
  int incl = s;
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(incl, o, 64);
    if (lane >= o) incl += v;
  }
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  int wbase = 0;
  for (int w = 0; w < wave; ++w) wbase += wsum[w];
  int run = wbase + incl - s;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (b0 + k < n) pre[b0 + k] = run;
    run += loc[k];
  }
  if (threadIdx.x == blockDim.x - 1) {
    int tot = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) tot += wsum[w];
    pre[n] = tot;
  }
  __syncthreads();
}

// largest c with pre[c] <= i
__device__ inline int find_cell(const int* pre, int nC, int i) {
  int lo = 0, hi = nC - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (pre[mid] <= i) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__device__ inline void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace
}  // namespace cube
