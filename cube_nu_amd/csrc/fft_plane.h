// fft_plane.h -- size-specialised 3-pass FFT convolution for cubes whose
// z-plane of half-complex values fits in LDS: (A) per z-plane, r2c along x and
// forward c2c along y; (B) lines along z: forward, times G, inverse; (C) per
// z-plane, inverse along y and c2r along x, with the normalisation.
//
// Every line length is split in two radices N = R1 R2 (half-length rows: A1
// A2) held in registers, and the ends of a pass work on registers directly:
// the first stage reads global memory, the last one writes it, the r2c split
// and the c2r merge ride on the row stage next to them (a task owns butterflies
// j and A1-j, whose elements are each other's conjugate partners), and in pass
// B the inverse starts with the radix the forward transform ended with, on the
// same registers.  A plane value crosses LDS 3 times per pass (write + read)
// and a z value twice, instead of 6 and 6 times with each stage, the split and
// the kernel product as LDS round trips of their own.  The passes move
// 8 bytes per mesh point and pass, and are bound by HBM and by the barriers
// between the stages: the more workgroups share a CU, the better.  Measured on
// MI355X: 4096 boxes of 80^3, 16.9 GB a pass, 3.1 + 3.5 + 4.0 ms (5.5, 4.9 and
// 4.2 TB/s; 4.1 + 5.5 + 4.3 ms with a stage per LDS round trip; a large copy
// reaches 4.9 TB/s), 64 boxes of 160^3 0.52 + 0.51 + 0.62 ms (1.01 + 1.20 +
// 1.07); 4096 boxes of 40^3 1.3 ms in all and of 56^3 3.5 ms, against 9.4 and
// 18 ms on the generic line passes.
#pragma once
#include "fft.h"
#include "fft_zlines.h"
#include "timing.h"

namespace cube {
namespace {

using namespace fftr;

// Work split of one size: planes per workgroup and threads of the plane passes.
template <typename R, int N>
struct Plan {
  static constexpr int H = N / 2, P = H + 1;
  static constexpr Split row = split2(H), col = split2(N);
  static constexpr int R1 = col.r1, R2 = col.r2;
  // rows: the stage that pairs butterflies has half the tasks, so it takes the larger number of
  // them: forward A1 = RB, A2 = RS (split stage A1/2+1 tasks), inverse A1 = RS, A2 = RB (merge A2/2+1)
  static constexpr int RB = cmax(row.r1, row.r2), RS = H / RB, TP = RB / 2 + 1;
  static constexpr int LS = P % 2 ? P : P + 1;  // odd row stride: rows start in different banks
  static constexpr int tasks = cmax(N * cmax(RS, TP), P * cmax(R1, R2));
  static constexpr int bytes = N * LS * (int)sizeof(CP<R>);
  // small planes: several per workgroup, up to about 512 tasks and 32 KB
  static constexpr int fit(int pb) { return N % pb == 0 && pb * tasks <= 512 && pb * bytes <= 32768 ? pb : 0; }
  static constexpr int PB = fit(8) ? 8 : (fit(4) ? 4 : (fit(2) ? 2 : 1));
  static constexpr int NT = round64(PB * tasks) < 1024 ? round64(PB * tasks) : 1024;
};

// Pass A: PB z-planes: rho (N x N reals) -> complex (N rows of N/2+1).
// WIN: the planes are read from the windows of a larger mesh (FFTWindow), in
// an order that gives each XCD a run of neighbouring boxes: their windows
// overlap, and the overlaps come from its L2.  Writing the windows out as
// cubes first cost 4.0 ms for 4096 of 80^3 (a pass over 8.4 GB and its read);
// here the pass takes 3.8 ms against 3.2.
template <typename R, int N, bool WIN>
__global__ void __launch_bounds__((Plan<R, N>::NT)) k_plane_fwd(const R* __restrict__ rho, FFTWindow win,
                                                                CP<R>* __restrict__ out,
                                                                const CP<R>* __restrict__ twg) {
  using C = CP<R>;
  using L = Plan<R, N>;
  constexpr int H = L::H, P = L::P, LS = L::LS, A1 = L::RB, A2 = L::RS, R1 = L::R1, R2 = L::R2, PB = L::PB,
                NT = L::NT;
  __shared__ C buf[PB * N * LS];
  __shared__ C tw[N];
  const int64_t plane0 = (WIN ? xcd_block(blockIdx.x, gridDim.x) : (int64_t)blockIdx.x) * PB;
  const C* src = reinterpret_cast<const C*>(rho + plane0 * N * N);
  for (int i = threadIdx.x; i < N; i += NT) tw[i] = twg[i];
  // rows, first stage: global -> registers -> LDS
#pragma unroll
  for (int i0 = 0; i0 < PB * N * A2; i0 += NT) {
    const int i = i0 + threadIdx.x;
    if (i < PB * N * A2) {
      const int row = i / A2, j = i % A2;
      C v[A1];
      if constexpr (WIN) {
        const uint32_t p = (uint32_t)plane0 + row / N, box = p / N;
        const int z = (int)(p % N), y = row % N;
        const float* fb = win.faces + (int64_t)box * (6 * N * N);
        const float* rp;
        int ox = 0, wrap = 1 << 30;
        const bool zf = z == 0 || z == N - 1, yf = y == 0 || y == N - 1;
        if (zf || yf) {
          rp = fb + (zf ? (z == 0 ? 4 : 5) * N + y : (y == 0 ? 2 : 3) * N + z) * N;
        } else {
          const int4 o = win.org[box];
          int gz = o.z + z, gy = o.y + y;
          gz = gz >= win.n ? gz - win.n : gz;
          gy = gy >= win.n ? gy - win.n : gy;
          rp = win.mesh + ((int64_t)gz * win.n + gy) * win.n;
          ox = o.x;
          wrap = win.n;
        }
#pragma unroll
        for (int r = 0; r < A1; ++r) {
          int x = ox + 2 * (j + r * A2);
          x = x >= wrap ? x - wrap : x;
          v[r] = *reinterpret_cast<const C*>(rp + x);
        }
        if (!zf && !yf) {
          if (j == 0) v[0].x = fb[z * N + y];
          if (j == A2 - 1) v[A1 - 1].y = fb[(N + z) * N + y];
        }
      } else {
#pragma unroll
        for (int r = 0; r < A1; ++r) v[r] = src[row * H + j + r * A2];
      }
      bfly<-1, A1>(v);
#pragma unroll
      for (int k = 0; k < A1; ++k) buf[row * LS + j * A1 + k] = v[k];
    }
  }
  __syncthreads();
  // rows, second stage, and the split X[q] = (Z[q] + conj Z[H-q])/2 - i/2 W_N^q (Z[q] - conj Z[H-q]):
  // butterflies j and A1-j hold each other's partners q and H-q
  {
    constexpr int T = PB * N * L::TP, MB = (T + NT - 1) / NT;
    C xa[MB][A2], xb[MB][A2];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int i = b * NT + threadIdx.x;
      if (i < T) {
        const int row = i / L::TP, j = i % L::TP, j2 = j == 0 ? 0 : A1 - j;
        C v[A2], u[A2];
#pragma unroll
        for (int r = 0; r < A2; ++r) {
          v[r] = buf[row * LS + j + r * A1];
          u[r] = buf[row * LS + j2 + r * A1];
          if (r > 0) {
            v[r] = mulw<-1>(v[r], tw[2 * r * j]);
            u[r] = mulw<-1>(u[r], tw[2 * r * j2]);
          }
        }
        bfly<-1, A2>(v);
        bfly<-1, A2>(u);
        const R half = (R)0.5;
#pragma unroll
        for (int k = 0; k < A2; ++k) {
          const C p = cj(j == 0 ? v[(A2 - k) % A2] : u[A2 - 1 - k]);
          const C xe = scl(add(v[k], p), half), d = scl(sub(v[k], p), half);
          const C t = mul(tw[j + k * A1], mi<-1>(d));
          xa[b][k] = add(xe, t);
          xb[b][k] = cj(sub(xe, t));
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int i = b * NT + threadIdx.x;
      if (i < T) {
        const int row = i / L::TP, j = i % L::TP;
#pragma unroll
        for (int k = 0; k < A2; ++k) {
          buf[row * LS + j + k * A1] = xa[b][k];
          // j = 0 holds q and H-q both: only X[H] is written from the partner side
          if (j != 0 || k == 0) buf[row * LS + H - j - k * A1] = xb[b][k];
        }
      }
    }
  }
  __syncthreads();
  // columns, first stage, in place
  {
    constexpr int T = PB * P * R2, MB = (T + NT - 1) / NT;
    C v[MB][R1];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int i = b * NT + threadIdx.x;
      if (i < T) {
        const int x = i % P, j = (i / P) % R2, pl = i / (P * R2);
#pragma unroll
        for (int r = 0; r < R1; ++r) v[b][r] = buf[(pl * N + j + r * R2) * LS + x];
        bfly<-1, R1>(v[b]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int i = b * NT + threadIdx.x;
      if (i < T) {
        const int x = i % P, j = (i / P) % R2, pl = i / (P * R2);
#pragma unroll
        for (int k = 0; k < R1; ++k) buf[(pl * N + j * R1 + k) * LS + x] = v[b][k];
      }
    }
  }
  __syncthreads();
  // columns, second stage: LDS -> registers -> global
  C* dst = out + plane0 * N * P;
#pragma unroll
  for (int i0 = 0; i0 < PB * P * R1; i0 += NT) {
    const int i = i0 + threadIdx.x;
    if (i < PB * P * R1) {
      const int x = i % P, j = (i / P) % R1, pl = i / (P * R1);
      C v[R2];
#pragma unroll
      for (int r = 0; r < R2; ++r) {
        v[r] = buf[(pl * N + j + r * R1) * LS + x];
        if (r > 0) v[r] = mulw<-1>(v[r], tw[r * j]);
      }
      bfly<-1, R2>(v);
#pragma unroll
      for (int k = 0; k < R2; ++k) dst[(pl * N + j + k * R1) * P + x] = v[k];
    }
  }
}

// Pass C: PB z-planes: inverse along y, c2r along x, normalisation.
template <typename R, int N>
__global__ void __launch_bounds__((Plan<R, N>::NT)) k_plane_inv(const CP<R>* __restrict__ in, R* __restrict__ phi,
                                                                const CP<R>* __restrict__ twg, R div3, R div1) {
  using C = CP<R>;
  using L = Plan<R, N>;
  constexpr int H = L::H, P = L::P, LS = L::LS, A1 = L::RS, A2 = L::RB, R1 = L::R1, R2 = L::R2, PB = L::PB,
                NT = L::NT;
  __shared__ C buf[PB * N * LS];
  __shared__ C tw[N];
  const int64_t plane0 = (int64_t)blockIdx.x * PB;
  const C* src = in + plane0 * N * P;
  for (int i = threadIdx.x; i < N; i += NT) tw[i] = twg[i];
  // columns, first stage: global -> registers -> LDS
#pragma unroll
  for (int i0 = 0; i0 < PB * P * R2; i0 += NT) {
    const int i = i0 + threadIdx.x;
    if (i < PB * P * R2) {
      const int x = i % P, j = (i / P) % R2, pl = i / (P * R2);
      C v[R1];
#pragma unroll
      for (int r = 0; r < R1; ++r) v[r] = src[(pl * N + j + r * R2) * P + x];
      bfly<+1, R1>(v);
#pragma unroll
      for (int k = 0; k < R1; ++k) buf[(pl * N + j * R1 + k) * LS + x] = v[k];
    }
  }
  __syncthreads();
  // columns, second stage, in place
  {
    constexpr int T = PB * P * R1, MB = (T + NT - 1) / NT;
    C v[MB][R2];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int i = b * NT + threadIdx.x;
      if (i < T) {
        const int x = i % P, j = (i / P) % R1, pl = i / (P * R1);
#pragma unroll
        for (int r = 0; r < R2; ++r) {
          v[b][r] = buf[(pl * N + j + r * R1) * LS + x];
          if (r > 0) v[b][r] = mulw<+1>(v[b][r], tw[r * j]);
        }
        bfly<+1, R2>(v[b]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int i = b * NT + threadIdx.x;
      if (i < T) {
        const int x = i % P, j = (i / P) % R1, pl = i / (P * R1);
#pragma unroll
        for (int k = 0; k < R2; ++k) buf[(pl * N + j + k * R1) * LS + x] = v[b][k];
      }
    }
  }
  __syncthreads();
  // rows: the merge Z[q] = E + iO, E = X[q] + conj X[H-q], O = (X[q] - conj X[H-q]) W_N^-q, and the
  // first stage of the half-length inverse (inputs q = j + r A2; partners H-q belong to A2-j)
  {
    constexpr int T = PB * N * L::TP, MB = (T + NT - 1) / NT;
    C za[MB][A1], zb[MB][A1];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int i = b * NT + threadIdx.x;
      if (i < T) {
        const int row = i / L::TP, j = i % L::TP, j2 = j == 0 ? 0 : A2 - j;
        const C* rp = buf + row * LS;
        C v[A1], u[A1];
#pragma unroll
        for (int r = 0; r < A1; ++r) {
          v[r] = rp[j + r * A2];
          u[r] = rp[j2 + r * A2];
        }
        const C xh = rp[H];
#pragma unroll
        for (int r = 0; r < A1; ++r) {
          const C p = cj(j == 0 ? (r == 0 ? xh : v[(A1 - r) % A1]) : u[A1 - 1 - r]);
          const C e = add(v[r], p), o = mi<+1>(mulw<+1>(sub(v[r], p), tw[j + r * A2]));
          za[b][r] = add(e, o);
          zb[b][A1 - 1 - r] = cj(sub(e, o));
        }
        bfly<+1, A1>(za[b]);
        bfly<+1, A1>(zb[b]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int i = b * NT + threadIdx.x;
      if (i < T) {
        const int row = i / L::TP, j = i % L::TP, j2 = j == 0 ? 0 : A2 - j;
#pragma unroll
        for (int k = 0; k < A1; ++k) {
          buf[row * LS + j * A1 + k] = za[b][k];
          if (j2 != j) buf[row * LS + j2 * A1 + k] = zb[b][k];
        }
      }
    }
  }
  __syncthreads();
  // rows, second stage: LDS -> registers -> global, normalised
  C* dst = reinterpret_cast<C*>(phi + plane0 * N * N);
  const R inv = (R)1 / (div3 != (R)0 ? div3 : div1);
#pragma unroll
  for (int i0 = 0; i0 < PB * N * A1; i0 += NT) {
    const int i = i0 + threadIdx.x;
    if (i < PB * N * A1) {
      const int row = i / A1, j = i % A1;
      C v[A2];
#pragma unroll
      for (int r = 0; r < A2; ++r) {
        v[r] = buf[row * LS + j + r * A1];
        if (r > 0) v[r] = mulw<+1>(v[r], tw[2 * r * j]);
      }
      bfly<+1, A2>(v);
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
        dst[row * H + j + k * A1] = CT<C>::mk(a, b);
      }
    }
  }
}

template <typename R, int N>
bool run_plane(const FFTCube<R>& c, R* rho, CP<R>* work, const float* G, int64_t nbox, R div3, R div1,
               hipStream_t s, KTimer* tm, const std::string& t, const FFTWindow* win) {
  using L = Plan<R, N>;
  const double Gb = (double)N * N * N * sizeof(R) * nbox;
  const double Kb = (double)N * N * L::P * sizeof(CP<R>) * nbox;
  const double Gk = (double)N * N * L::P * sizeof(float);
  const dim3 planes((unsigned)(nbox * (N / L::PB)));
  {
    KScope k(tm, (t + "fft_xy_fwd").c_str(), Gb + Kb);
    if (!win) {
      hipLaunchKernelGGL((k_plane_fwd<R, N, false>), planes, dim3(L::NT), 0, s, rho, FFTWindow{}, work, c.tw);
    } else {
      if constexpr (std::is_same<R, float>::value && N % 8 == 0)
        hipLaunchKernelGGL((k_plane_fwd<R, N, true>), planes, dim3(L::NT), 0, s, rho, *win, work, c.tw);
    }
    CUBE_HIP(hipGetLastError());
  }
  {
    KScope k(tm, (t + "fft_z_green").c_str(), 2 * Kb + Gk);
    launch_zlines<R, N>(work, G, c.tw, nbox, s);
  }
  {
    KScope k(tm, (t + "fft_xy_inv").c_str(), Gb + Kb);
    hipLaunchKernelGGL((k_plane_inv<R, N>), planes, dim3(L::NT), 0, s, work, rho, c.tw, div3, div1);
    CUBE_HIP(hipGetLastError());
  }
  return true;
}

}  // namespace
}  // namespace cube
