// fft_box.hip -- size-specialised one-pass FFT convolution for many small cubes whose
// half-complex values fit in LDS whole: one workgroup per cube, rows (r2c),
// columns along y, lines along z (forward, times G, inverse), columns, rows (c2r
// and normalisation).
//
// A thread holds a whole line in registers (radices up to 32, twiddles in the
// code), so a value crosses LDS four times and global memory only as input and
// output, where the plane form's three passes move it six times; both ends go
// through LDS so that lanes run along the rows.  Bound by the latency of the phases
// (two workgroups of 24^3 share a CU, one of 32^3).  Measured on MI355X: 4096
// windows of 24^3 0.187 ms against 0.307 as planes, of 32^3 0.40 against 0.74; 512
// cubes are the two workgroups of every CU, and half as many take as long as their
// planes.
#include "fft.h"
#include "fft_radix.h"
#include "timing.h"

namespace cube {
namespace {

using namespace fftr;

template <int N>
struct BPlan {
  static constexpr int H = N / 2, P = H + 1, LS = P % 2 ? P : P + 1;
  static constexpr int NT = N * N;  // a thread per row
};

// W_N^q, forward
template <int N>
__device__ inline float2 root(int q) {
  constexpr Roots<N> W = roots<N>();
  return make_float2((float)W.c[q], (float)-W.s[q]);
}

template <int N, bool WIN>
__global__ void __launch_bounds__((BPlan<N>::NT)) k_box(float* __restrict__ rho, FFTWindow win,
                                                       const float* __restrict__ G, float div3, float div1) {
  using L = BPlan<N>;
  constexpr int H = L::H, P = L::P, LS = L::LS, NT = L::NT;
  __shared__ float2 buf[N * N * LS];
  const int64_t box = WIN ? xcd_block(blockIdx.x, gridDim.x) : (int64_t)blockIdx.x;
  float* cube = rho + box * (N * N * N);
  // in: lanes along the rows, eight loads in flight
  constexpr int NV = N * N * H, KV = (NV + NT - 1) / NT, KR = (N * N + NT - 1) / NT;
  float2 ends[KR];  // WIN: the face values that end this thread's rows
  const uintptr_t* from = nullptr;
  int ox = 0;
  if constexpr (WIN) {
    // each row's address, one thread a row; odd: a row of the mesh
    __shared__ uintptr_t rows[N * N];
    from = rows;
    const float* fb = win.faces + box * (6 * N * N);
    const int4 o = win.org[box];
    ox = o.x;
#pragma unroll
    for (int k = 0; k < KR; ++k) {
      const int row = min(k * NT + (int)threadIdx.x, N * N - 1), z = row / N, y = row - z * N;
      ends[k] = make_float2(fb[row], fb[N * N + row]);
      if (z == 0 || z == N - 1 || y == 0 || y == N - 1) {
        const bool zf = z == 0 || z == N - 1;
        rows[row] = (uintptr_t)(fb + (zf ? (z == 0 ? 4 : 5) * N + y : (y == 0 ? 2 : 3) * N + z) * N);
      } else {
        int gz = o.z + z, gy = o.y + y;
        gz = gz >= win.n ? gz - win.n : gz;
        gy = gy >= win.n ? gy - win.n : gy;
        rows[row] = (uintptr_t)(win.mesh + ((int64_t)gz * win.n + gy) * win.n) | 1;
      }
    }
    __syncthreads();
  }
  const float2* src = reinterpret_cast<const float2*>(cube);
#pragma unroll
  for (int k0 = 0; k0 < KV; k0 += 8) {
    float2 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int i = min((k0 + k) * NT + (int)threadIdx.x, NV - 1);
      if (k0 + k >= KV) continue;
      if constexpr (WIN) {
        const int row = i / H, j = i - row * H;
        const uintptr_t a = from[row];
        const int xm = 2 * j + ox, x = (a & 1) ? (xm >= win.n ? xm - win.n : xm) : 2 * j;
        v[k] = *reinterpret_cast<const float2*>(reinterpret_cast<const float*>(a & ~(uintptr_t)1) + x);
      } else {
        v[k] = src[i];
      }
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int i = (k0 + k) * NT + (int)threadIdx.x, row = i / H;
      if (k0 + k < KV && i < NV) buf[row * LS + i - row * H] = v[k];
    }
  }
  __syncthreads();
  // rows: N reals as H complex, and the split X[q] = (Z[q] + conj Z[H-q])/2 - i/2 W_N^q (Z[q] - conj Z[H-q])
#pragma unroll
  for (int k = 0; k < KR; ++k) {
    const int row = k * NT + (int)threadIdx.x;
    if (row >= N * N) break;
    float2* o = buf + row * LS;
    float2 v[H];
#pragma unroll
    for (int r = 0; r < H; ++r) v[r] = o[r];
    if (WIN) {
      const int z = row / N, y = row - z * N;
      if (z > 0 && z < N - 1 && y > 0 && y < N - 1) {
        v[0].x = ends[k].x;
        v[H - 1].y = ends[k].y;
      }
    }
    bfly<-1, H>(v);
    o[0] = make_float2(v[0].x + v[0].y, 0.0f);
    o[H] = make_float2(v[0].x - v[0].y, 0.0f);
#pragma unroll
    for (int q = 1; q <= H / 2; ++q) {
      const float2 p = cj(v[H - q]);
      const float2 xe = scl(add(v[q], p), 0.5f), d = scl(sub(v[q], p), 0.5f);
      const float2 t = mul(root<N>(q), mi<-1>(d));
      o[q] = add(xe, t);
      if (2 * q != H) o[H - q] = cj(sub(xe, t));
    }
  }
  __syncthreads();
  const int x = threadIdx.x % P, l = threadIdx.x / P;  // a line at x of plane z = l, then of row y = l
  const bool ok = l < N;
  if (ok) {
    float2 v[N];
#pragma unroll
    for (int r = 0; r < N; ++r) v[r] = buf[(l * N + r) * LS + x];
    bfly<-1, N>(v);
#pragma unroll
    for (int r = 0; r < N; ++r) buf[(l * N + r) * LS + x] = v[r];
  }
  __syncthreads();
  if (ok) {
    float g[N];
#pragma unroll
    for (int r = 0; r < N; ++r) g[r] = G[(r * N + l) * P + x];
    float2 v[N];
#pragma unroll
    for (int r = 0; r < N; ++r) v[r] = buf[(r * N + l) * LS + x];
    bfly<-1, N>(v);
#pragma unroll
    for (int r = 0; r < N; ++r) v[r] = scl(v[r], g[r]);  // cxyz*tf (kick.f90:698)
    bfly<+1, N>(v);
#pragma unroll
    for (int r = 0; r < N; ++r) buf[(r * N + l) * LS + x] = v[r];
  }
  __syncthreads();
  if (ok) {
    float2 v[N];
#pragma unroll
    for (int r = 0; r < N; ++r) v[r] = buf[(l * N + r) * LS + x];
    bfly<+1, N>(v);
#pragma unroll
    for (int r = 0; r < N; ++r) buf[(l * N + r) * LS + x] = v[r];
  }
  __syncthreads();
  // rows: the merge Z[q] = E + iO, E = X[q] + conj X[H-q], O = (X[q] - conj X[H-q]) W_N^-q, and the inverse
  for (int row = threadIdx.x; row < N * N; row += NT) {
    float2* o = buf + row * LS;
    float2 v[H];
    {
      const float2 a = o[0], b = o[H];
      v[0] = make_float2(a.x + b.x, a.x - b.x);
    }
#pragma unroll
    for (int q = 1; q <= H / 2; ++q) {
      const float2 a = o[q], p = cj(o[H - q]);
      const float2 e = add(a, p), od = mi<+1>(mulw<+1>(sub(a, p), root<N>(q)));
      v[q] = add(e, od);
      if (2 * q != H) v[H - q] = cj(sub(e, od));
    }
    bfly<+1, H>(v);
#pragma unroll
    for (int r = 0; r < H; ++r) o[r] = v[r];
  }
  __syncthreads();
  // out: lanes along the rows
  const float inv = 1.0f / (div3 != 0.0f ? div3 : div1);
  float2* dst = reinterpret_cast<float2*>(cube);
#pragma unroll 4
  for (int i = threadIdx.x; i < N * N * H; i += NT) {
    const int row = i / H;
    float2 v = buf[row * LS + i - row * H];
    if (div3 != 0.0f) {
      v = make_float2(div_by(v.x, div3, inv), div_by(v.y, div3, inv));
    } else {
      v.x = div_by(div_by(div_by(v.x, div1, inv), div1, inv), div1, inv);
      v.y = div_by(div_by(div_by(v.y, div1, inv), div1, inv), div1, inv);
    }
    dst[i] = v;
  }
}

template <int N>
void run_box(float* rho, const float* G, int64_t nbox, float div3, float div1, hipStream_t s, KTimer* tm,
             const std::string& t, const FFTWindow* win) {
  KScope k(tm, (t + "fft_box").c_str(), 2.0 * N * N * N * sizeof(float) * nbox);
  if (win)
    hipLaunchKernelGGL((k_box<N, true>), dim3((unsigned)nbox), dim3(BPlan<N>::NT), 0, s, rho, *win, G, div3, div1);
  else
    hipLaunchKernelGGL((k_box<N, false>), dim3((unsigned)nbox), dim3(BPlan<N>::NT), 0, s, rho, FFTWindow{}, G, div3,
                       div1);
  CUBE_HIP(hipGetLastError());
}

}  // namespace

// Returns false for other sizes, and for levels of fewer cubes than keep the chip's
// CUs busy (the plane form spreads one over several).
bool fft_convolve_boxes(int n, float* rho, const float* G, int64_t nbox, int64_t total, float div3, float div1,
                        hipStream_t s, KTimer* tm, const char* tag, const FFTWindow* win) {
  if (total < 512) return false;
  switch (n) {
    case 16: run_box<16>(rho, G, nbox, div3, div1, s, tm, tag, win); return true;
    case 24: run_box<24>(rho, G, nbox, div3, div1, s, tm, tag, win); return true;
    case 32: run_box<32>(rho, G, nbox, div3, div1, s, tm, tag, win); return true;
    default: return false;
  }
}

}  // namespace cube
