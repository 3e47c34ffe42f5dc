// fft.h -- batched 3-D real FFT convolution on cubes (LDS-staged Stockham).
//
// Replaces the FFTW plans of cubefft.f90:5-38 (tile / sub-tile meshes) and
// pencil_fft.f90:23-79, 327-338 (coarse mesh at nn=1).  Conventions follow
// FFTW: forward r2c e^{-i}, backward c2r e^{+i}, both unnormalised.
#pragma once
#include "common.h"

namespace cube {

struct FFTStages {
  int n;             // line length
  int nst;           // number of radix stages
  int rad[16];
};

FFTStages make_stages(int n);

// One cube size: twiddle tables for n (full, used by r2c post-processing and
// the y/z passes) and the stage factorisations of n and n/2.
template <typename R>
struct FFTCube {
  int n = 0;
  FFTStages full{}, half{};
  typename Cplx<R>::T* tw = nullptr;  // e^{-2 pi i t / n}, t = 0..n-1
  void init(int n_);
  void release();
};

// Convolve `nbox` real cubes in place with a real kernel G(kx,ky,kz):
//   phi = c2r( G * r2c(rho) ) / div
// rho/phi: [box][z][y][x] real (n^3 per box); work: complex scratch of
// nbox * n*n*(n/2+1) elements.  The division follows the reference: one FP
// division by div3 when div3 != 0, else three divisions by div1.
// A convolution's input cut from one larger periodic mesh instead of cubes of
// its own: box b's point (x, y, z) is mesh[(org[b] + (x, y, z)) mod n], except
// on the window's faces, which are given: face 2 axis + side of box b at
// faces[(6 b + face) c^2] (c the cube size), rows along the lower of the other
// two axes.  org.x and n are even.
struct FFTWindow {
  const float* mesh = nullptr;
  const float* faces = nullptr;
  const int4* org = nullptr;
  int n = 0;
};
// True when cubes of n points take the plane passes (the only ones that read
// windows).
template <typename R>
bool fft_reads_windows(int n);

// Sizes with a specialised form take it: one pass (fft_box.hip) where a small
// cube fits in LDS and there are many, plane passes (fft_plane.h) where a z-plane
// fits, line passes (fft_line.hip) for larger ones; the others take the generic
// line passes.  small_lds: no pass that needs more than about 40 KB of LDS per
// workgroup (a launch beside another stream's kernels).  total: the cubes of the
// whole level, of which nbox are a batch (0: nbox); the form follows it, so that
// the workspace's batches give the same bits.
template <typename R>
void fft_convolve(const FFTCube<R>& c, R* rho, typename Cplx<R>::T* work, const float* G, int64_t nbox, R div3,
                  R div1, hipStream_t s, KTimer* tm = nullptr, const char* tag = "", bool small_lds = false,
                  const FFTWindow* win = nullptr, int64_t total = 0);

// The specialised forms; false when n has none.
template <typename R>
bool fft_convolve_plane(const FFTCube<R>& c, R* rho, typename Cplx<R>::T* work, const float* G, int64_t nbox,
                        R div3, R div1, hipStream_t s, KTimer* tm, const char* tag, const FFTWindow* win);
bool fft_plane_size(int n);  // FP32
bool fft_convolve_boxes(int n, float* rho, const float* G, int64_t nbox, int64_t total, float div3, float div1,
                        hipStream_t s, KTimer* tm, const char* tag, const FFTWindow* win);
bool fft_convolve_plane_even(const FFTCube<float>& c, float* rho, float2* work, const float* G, int64_t nbox,
                             float div3, float div1, hipStream_t s, KTimer* tm, const char* tag);
template <typename R>
bool fft_convolve_lines(const FFTCube<R>& c, R* rho, typename Cplx<R>::T* work, const float* G, int64_t nbox,
                        R div3, R div1, hipStream_t s, KTimer* tm, const char* tag);

// Forward-only and inverse-only pieces (used by the input maker and tests).
template <typename R>
void fft_r2c3d(const FFTCube<R>& c, const R* rho, typename Cplx<R>::T* out, int64_t nbox, hipStream_t s);
template <typename R>
void fft_c2r3d(const FFTCube<R>& c, typename Cplx<R>::T* in, R* out, int64_t nbox, hipStream_t s);

}  // namespace cube
