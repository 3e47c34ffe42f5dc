// fft_line.hip -- size-specialised 5-pass FFT convolution for cubes whose
// z-plane does not fit in LDS (and for the coarse mesh beside the second
// stream's kernels, where a workgroup that needs half a CU's LDS waits):
// rows along x (r2c), columns along y, lines along z (forward, G, inverse),
// columns along y, rows along x (c2r and normalisation).
//
// As in fft_plane.hip every line is two radices held in registers, the first
// read from and the last written to global memory directly, so a value crosses
// LDS once per direction (rows: twice with the split or merge).  Each pass
// reads and writes the mesh once and is bound by HBM: 4 meshes of 256^3, 0.54
// GB a pass, 0.13-0.14 ms each (4 TB/s), 0.68 ms a convolution against 1.84 on
// the generic line passes; one coarse mesh of 128^3 0.06 ms alone.
#include "fft.h"
#include "fft_zlines.h"
#include "timing.h"

namespace cube {
namespace {

using namespace fftr;

template <typename R, int N>
struct LPlan {
  static constexpr int H = N / 2, P = H + 1;
  static constexpr Split row = split2(H), col = split2(N);
  static constexpr int RB = cmax(row.r1, row.r2), RS = H / RB, TP = RB / 2 + 1;
  static constexpr int R1 = col.r1, R2 = col.r2;
  static constexpr int LS = H % 2 ? H : H + 1;
  static constexpr int RT = cmax(RS, TP);                  // threads per row
  static constexpr int NR = cmax(1, 256 / RT);             // rows per workgroup
  static constexpr int NT = round64(NR * RT);
  // y columns: W adjacent x per workgroup
  static constexpr int W = 32, NX = (P + W - 1) / W, NTY = round64(W * cmax(R1, R2));
};

// rows of N reals -> N/2+1 complex; the stages and the split as in k_plane_fwd
template <typename R, int N>
__global__ void __launch_bounds__((LPlan<R, N>::NT)) k_line_r2c(const R* __restrict__ in, CP<R>* __restrict__ out,
                                                               int64_t nrows, const CP<R>* __restrict__ tw) {
  using C = CP<R>;
  using L = LPlan<R, N>;
  constexpr int H = L::H, LS = L::LS, A1 = L::RB, A2 = L::RS;
  __shared__ C buf[L::NR * LS];
  const int lr = threadIdx.x / L::RT, j = threadIdx.x % L::RT;
  const int64_t row = (int64_t)blockIdx.x * L::NR + lr;
  const bool ok = lr < L::NR && row < nrows;
  if (ok && j < A2) {
    const C* src = reinterpret_cast<const C*>(in + row * N);
    C v[A1];
#pragma unroll
    for (int r = 0; r < A1; ++r) v[r] = src[j + r * A2];
    bfly<-1, A1>(v);
#pragma unroll
    for (int k = 0; k < A1; ++k) buf[lr * LS + j * A1 + k] = v[k];
  }
  __syncthreads();
  if (!ok || j >= L::TP) return;
  const int j2 = j == 0 ? 0 : A1 - j;
  C v[A2], u[A2];
#pragma unroll
  for (int r = 0; r < A2; ++r) {
    v[r] = buf[lr * LS + j + r * A1];
    u[r] = buf[lr * LS + j2 + r * A1];
    if (r > 0) {
      v[r] = mulw<-1>(v[r], tw[2 * r * j]);
      u[r] = mulw<-1>(u[r], tw[2 * r * j2]);
    }
  }
  bfly<-1, A2>(v);
  bfly<-1, A2>(u);
  C* dst = out + row * (H + 1);
  const R half = (R)0.5;
#pragma unroll
  for (int k = 0; k < A2; ++k) {
    const C p = cj(j == 0 ? v[(A2 - k) % A2] : u[A2 - 1 - k]);
    const C xe = scl(add(v[k], p), half), d = scl(sub(v[k], p), half);
    const C t = mul(tw[j + k * A1], mi<-1>(d));
    dst[j + k * A1] = add(xe, t);
    if (j != 0 || k == 0) dst[H - j - k * A1] = cj(sub(xe, t));
  }
}

// N/2+1 complex -> rows of N reals, normalised; merge and stages as in k_plane_inv
template <typename R, int N>
__global__ void __launch_bounds__((LPlan<R, N>::NT)) k_line_c2r(const CP<R>* __restrict__ in, R* __restrict__ out,
                                                               int64_t nrows, const CP<R>* __restrict__ tw, R div3,
                                                               R div1) {
  using C = CP<R>;
  using L = LPlan<R, N>;
  constexpr int H = L::H, LS = L::LS, A1 = L::RS, A2 = L::RB;
  __shared__ C buf[L::NR * LS];
  const int lr = threadIdx.x / L::RT, j = threadIdx.x % L::RT;
  const int64_t row = (int64_t)blockIdx.x * L::NR + lr;
  const bool ok = lr < L::NR && row < nrows;
  if (ok && j < L::TP) {
    const C* rp = in + row * (H + 1);
    const int j2 = j == 0 ? 0 : A2 - j;
    C v[A1], u[A1], zb[A1];
#pragma unroll
    for (int r = 0; r < A1; ++r) {
      v[r] = rp[j + r * A2];
      u[r] = rp[j2 + r * A2];
    }
    const C xh = rp[H];
    C za[A1];
#pragma unroll
    for (int r = 0; r < A1; ++r) {
      const C p = cj(j == 0 ? (r == 0 ? xh : v[(A1 - r) % A1]) : u[A1 - 1 - r]);
      const C e = add(v[r], p), o = mi<+1>(mulw<+1>(sub(v[r], p), tw[j + r * A2]));
      za[r] = add(e, o);
      zb[A1 - 1 - r] = cj(sub(e, o));
    }
    bfly<+1, A1>(za);
    bfly<+1, A1>(zb);
#pragma unroll
    for (int k = 0; k < A1; ++k) {
      buf[lr * LS + j * A1 + k] = za[k];
      if (j2 != j) buf[lr * LS + j2 * A1 + k] = zb[k];
    }
  }
  __syncthreads();
  if (!ok || j >= A1) return;
  C v[A2];
#pragma unroll
  for (int r = 0; r < A2; ++r) {
    v[r] = buf[lr * LS + j + r * A1];
    if (r > 0) v[r] = mulw<+1>(v[r], tw[2 * r * j]);
  }
  bfly<+1, A2>(v);
  C* dst = reinterpret_cast<C*>(out + row * N);
  const R inv = (R)1 / (div3 != (R)0 ? div3 : div1);
#pragma unroll
  for (int k = 0; k < A2; ++k) {
    R a = v[k].x, b = v[k].y;
    if (div3 != (R)0) {
      a = div_by(a, div3, inv);
      b = div_by(b, div3, inv);
    } else {
      a = div_by(div_by(div_by(a, div1, inv), div1, inv), div1, inv);
      b = div_by(div_by(div_by(b, div1, inv), div1, inv), div1, inv);
    }
    dst[j + k * A1] = CT<C>::mk(a, b);
  }
}

// columns along y, in place: W adjacent x of one z-plane per workgroup
template <typename R, int N, int SIGN>
__global__ void __launch_bounds__((LPlan<R, N>::NTY)) k_line_y(CP<R>* __restrict__ data,
                                                              const CP<R>* __restrict__ tw) {
  using C = CP<R>;
  using L = LPlan<R, N>;
  constexpr int P = L::P, R1 = L::R1, R2 = L::R2, W = L::W;
  __shared__ C buf[N * W];
  const int c = threadIdx.x % W, j = threadIdx.x / W;
  const int64_t plane = blockIdx.x / L::NX;
  const int x = (int)(blockIdx.x % L::NX) * W + c;
  const bool ok = x < P;
  C* base = data + plane * N * P + x;
  if (j < R2) {
    C v[R1];
#pragma unroll
    for (int r = 0; r < R1; ++r) v[r] = ok ? base[(j + r * R2) * P] : CT<C>::mk((R)0, (R)0);
    bfly<SIGN, R1>(v);
#pragma unroll
    for (int k = 0; k < R1; ++k) buf[(j * R1 + k) * W + c] = v[k];
  }
  __syncthreads();
  if (j >= R1 || !ok) return;
  C v[R2];
#pragma unroll
  for (int r = 0; r < R2; ++r) {
    v[r] = buf[(j + r * R1) * W + c];
    if (r > 0) v[r] = mulw<SIGN>(v[r], tw[r * j]);
  }
  bfly<SIGN, R2>(v);
#pragma unroll
  for (int k = 0; k < R2; ++k) base[(j + k * R1) * P] = v[k];
}

template <typename R, int N>
bool run_lines(const FFTCube<R>& c, R* rho, CP<R>* work, const float* G, int64_t nbox, R div3, R div1,
               hipStream_t s, KTimer* tm, const std::string& t) {
  using L = LPlan<R, N>;
  const int64_t nrows = nbox * N * N;
  const dim3 rows((unsigned)ceil_div(nrows, L::NR)), cols((unsigned)(nbox * N * L::NX));
  const double Gb = (double)N * N * N * sizeof(R) * nbox;
  const double Kb = (double)N * N * L::P * sizeof(CP<R>) * nbox;
  const double Gk = (double)N * N * L::P * sizeof(float);
  {
    KScope k(tm, (t + "fft_x_r2c").c_str(), Gb + Kb);
    hipLaunchKernelGGL((k_line_r2c<R, N>), rows, dim3(L::NT), 0, s, rho, work, nrows, c.tw);
    CUBE_HIP(hipGetLastError());
  }
  {
    KScope k(tm, (t + "fft_y_fwd").c_str(), 2 * Kb);
    hipLaunchKernelGGL((k_line_y<R, N, -1>), cols, dim3(L::NTY), 0, s, work, c.tw);
    CUBE_HIP(hipGetLastError());
  }
  {
    KScope k(tm, (t + "fft_z_green").c_str(), 2 * Kb + Gk);
    launch_zlines<R, N>(work, G, c.tw, nbox, s);
  }
  {
    KScope k(tm, (t + "fft_y_inv").c_str(), 2 * Kb);
    hipLaunchKernelGGL((k_line_y<R, N, +1>), cols, dim3(L::NTY), 0, s, work, c.tw);
    CUBE_HIP(hipGetLastError());
  }
  {
    KScope k(tm, (t + "fft_x_c2r").c_str(), Gb + Kb);
    hipLaunchKernelGGL((k_line_c2r<R, N>), rows, dim3(L::NT), 0, s, work, rho, nrows, c.tw, div3, div1);
    CUBE_HIP(hipGetLastError());
  }
  return true;
}

}  // namespace

// Returns false when n has no specialised form (the caller then uses the
// generic line passes).
template <typename R>
bool fft_convolve_lines(const FFTCube<R>& c, R* rho, typename Cplx<R>::T* work, const float* G, int64_t nbox,
                        R div3, R div1, hipStream_t s, KTimer* tm, const char* tag) {
  if constexpr (std::is_same<R, float>::value) {
    const std::string t(tag);
    // below 208 the plane form's sizes beyond 88 points, for coarse meshes beside another
    // stream (with generic line passes: 104 0.042 / 0.096 ms alone, 144 0.063 / 0.122,
    // 192 0.092 / 0.210); above, where no plane form is
    switch (c.n) {
#define CUBE_FFT_SIZE(n) \
  case n: return run_lines<R, n>(c, rho, work, G, nbox, div3, div1, s, tm, t);
      CUBE_FFT_SIZE(96)
      CUBE_FFT_SIZE(104)
      CUBE_FFT_SIZE(112)
      CUBE_FFT_SIZE(120)
      CUBE_FFT_SIZE(128)
      CUBE_FFT_SIZE(144)
      CUBE_FFT_SIZE(160)
      CUBE_FFT_SIZE(168)
      CUBE_FFT_SIZE(176)
      CUBE_FFT_SIZE(192)
      CUBE_FFT_SIZE(208)
      CUBE_FFT_SIZE(210)
      CUBE_FFT_SIZE(216)
      CUBE_FFT_SIZE(224)
      CUBE_FFT_SIZE(234)
      CUBE_FFT_SIZE(240)
      CUBE_FFT_SIZE(252)
      CUBE_FFT_SIZE(256)
      CUBE_FFT_SIZE(288)
#undef CUBE_FFT_SIZE
      default: break;
    }
  }
  return false;
}

template bool fft_convolve_lines<float>(const FFTCube<float>&, float*, float2*, const float*, int64_t, float, float,
                                        hipStream_t, KTimer*, const char*);
template bool fft_convolve_lines<double>(const FFTCube<double>&, double*, double2*, const float*, int64_t, double,
                                         double, hipStream_t, KTimer*, const char*);

}  // namespace cube
