// fft_plane.hip -- the plane convolutions (fft_plane.h) of multiples of 8.
#include "fft_plane.h"

namespace cube {

// Returns false when n has no specialised kernel (the caller then uses the
// generic line passes).  The sizes here are the multiples of 8 that tile and
// sub-tile meshes take (16k + 32 and 8k + 16, and their finer levels) whose
// plane fits in LDS; fft_plane2.hip has the other even ones.
template <typename R>
bool fft_convolve_plane(const FFTCube<R>& c, R* rho, typename Cplx<R>::T* work, const float* G, int64_t nbox,
                        R div3, R div1, hipStream_t s, KTimer* tm, const char* tag, const FFTWindow* win) {
  const std::string t(tag);
  switch (c.n) {
#define CUBE_FFT_SIZE(n) \
  case n: return run_plane<R, n>(c, rho, work, G, nbox, div3, div1, s, tm, t, win);
    CUBE_FFT_SIZE(16)
    CUBE_FFT_SIZE(24)
    CUBE_FFT_SIZE(32)
    CUBE_FFT_SIZE(40)
    CUBE_FFT_SIZE(48)
    CUBE_FFT_SIZE(56)
    CUBE_FFT_SIZE(64)
    CUBE_FFT_SIZE(72)
    CUBE_FFT_SIZE(80)
    CUBE_FFT_SIZE(88)
    CUBE_FFT_SIZE(96)
    CUBE_FFT_SIZE(104)
    CUBE_FFT_SIZE(112)
    CUBE_FFT_SIZE(120)
    CUBE_FFT_SIZE(128)
    default: break;
  }
  // FP64 planes beyond 128 points do not fit in LDS
  if constexpr (std::is_same<R, float>::value) {
    switch (c.n) {
      CUBE_FFT_SIZE(144)
      CUBE_FFT_SIZE(160)
      CUBE_FFT_SIZE(168)
      CUBE_FFT_SIZE(176)
      CUBE_FFT_SIZE(192)
      default: break;
    }
  }
#undef CUBE_FFT_SIZE
  if constexpr (std::is_same<R, float>::value) {
    if (!win) return fft_convolve_plane_even(c, rho, work, G, nbox, div3, div1, s, tm, tag);
  }
  return false;
}

template bool fft_convolve_plane<float>(const FFTCube<float>&, float*, float2*, const float*, int64_t, float, float,
                                        hipStream_t, KTimer*, const char*, const FFTWindow*);
template bool fft_convolve_plane<double>(const FFTCube<double>&, double*, double2*, const float*, int64_t, double,
                                         double, hipStream_t, KTimer*, const char*, const FFTWindow*);

bool fft_plane_size(int n) {
  switch (n) {
    case 16: case 24: case 32: case 40: case 48: case 56: case 64: case 72: case 80: case 88: case 96: case 104:
    case 112: case 120: case 128: case 144: case 160: case 168: case 176: case 192: return true;
    default: return false;
  }
}

}  // namespace cube
