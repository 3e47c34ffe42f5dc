// fft_zlines.h -- the z pass of the size-specialised convolutions: lines along
// z of the half-complex mesh, forward, times G, inverse, in one kernel.
#pragma once
#include "fft_radix.h"

namespace cube {
namespace fftr {

template <typename R>
using CP = typename Cplx<R>::T;

constexpr int cmax(int a, int b) { return a > b ? a : b; }
constexpr int round64(int a) { return (a + 63) / 64 * 64; }

// Columns per workgroup W (64: one j per wavefront, its twiddles scalar; less
// where the lines are long) and one thread per column and butterfly.
template <typename R, int N>
struct ZPlan {
  static constexpr Split col = split2(N);
  static constexpr int R1 = col.r1, R2 = col.r2, NC = N * (N / 2 + 1);
  static constexpr int bytes = N * (int)sizeof(CP<R>);
  static constexpr int W = 64 * cmax(R1, R2) <= 1024 && 64 * bytes <= 53248 ? 64 : (32 * bytes <= 73728 ? 32 : 16);
  static constexpr int NB = (NC + W - 1) / W, NT = round64(W * cmax(R1, R2));
};

// W columns (of the N P columns of a box, contiguous in memory) along
// z: forward, times G, inverse.
template <typename R, int N>
static __global__ void __launch_bounds__((ZPlan<R, N>::NT)) k_zlines(CP<R>* __restrict__ data, const float* __restrict__ G,
                                                             const CP<R>* __restrict__ tw) {
  using C = CP<R>;
  using L = ZPlan<R, N>;
  constexpr int R1 = L::R1, R2 = L::R2, W = L::W, NC = L::NC, NB = L::NB;
  __shared__ C buf[N * W];
  const int c = threadIdx.x % W;
  int j = threadIdx.x / W;
  if constexpr (W == 64) j = __builtin_amdgcn_readfirstlane(j);  // twiddles by scalar loads
  const int64_t box = blockIdx.x / NB;
  const int col = (int)(blockIdx.x % NB) * W + c;
  const bool ok = col < NC;
  C* base = data + box * (int64_t)N * NC + col;
  if (j < R2) {
    C v[R1];
#pragma unroll
    for (int r = 0; r < R1; ++r) v[r] = ok ? base[(j + r * R2) * NC] : CT<C>::mk((R)0, (R)0);
    bfly<-1, R1>(v);
#pragma unroll
    for (int k = 0; k < R1; ++k) buf[(j * R1 + k) * W + c] = v[k];
  }
  __syncthreads();
  C x[R2];
  if (j < R1) {
    R g[R2];
#pragma unroll
    for (int k = 0; k < R2; ++k) g[k] = ok ? (R)G[(j + k * R1) * NC + col] : (R)0;
#pragma unroll
    for (int r = 0; r < R2; ++r) {
      x[r] = buf[(j + r * R1) * W + c];
      if (r > 0) x[r] = mulw<-1>(x[r], tw[r * j]);
    }
    bfly<-1, R2>(x);
#pragma unroll
    for (int k = 0; k < R2; ++k) x[k] = scl(x[k], g[k]);  // cxyz*tf (kick.f90:698)
    bfly<+1, R2>(x);
  }
  __syncthreads();
  if (j < R1) {
#pragma unroll
    for (int k = 0; k < R2; ++k) buf[(j * R2 + k) * W + c] = x[k];
  }
  __syncthreads();
  if (j < R2) {
    C v[R1];
#pragma unroll
    for (int r = 0; r < R1; ++r) {
      v[r] = buf[(j + r * R2) * W + c];
      if (r > 0) v[r] = mulw<+1>(v[r], tw[r * j]);
    }
    bfly<+1, R1>(v);
    if (ok) {
#pragma unroll
      for (int k = 0; k < R1; ++k) base[(j + k * R2) * NC] = v[k];
    }
  }
}

template <typename R, int N>
void launch_zlines(CP<R>* work, const float* G, const CP<R>* tw, int64_t nbox, hipStream_t s) {
  using L = ZPlan<R, N>;
  hipLaunchKernelGGL((k_zlines<R, N>), dim3((unsigned)(nbox * L::NB)), dim3(L::NT), 0, s, work, G, tw);
  CUBE_HIP(hipGetLastError());
}

}  // namespace fftr
}  // namespace cube
