// fft_plane2.hip -- the plane convolutions (fft_plane.h) of the other even sizes: the
// meshes of the differentiable path are free to be any.  FP32, no windows; every
// size up to 198 whose lines and half lines split into two radices and whose
// plane fits in LDS (three meshes of 90^3 0.027 ms against 0.098 on the generic line
// passes).
#include <utility>

#include "fft_plane.h"

namespace cube {
namespace {

constexpr int kFrom = 18, kTo = 198;
constexpr bool plane_ok(int n) {
  if (n % 8 == 0 || fftr::split2(n).r1 == 0 || fftr::split2(n / 2).r1 == 0) return false;
  const int p = n / 2 + 1, ls = p % 2 ? p : p + 1;
  return (n * ls + n) * 8 <= 160 * 1024;
}

struct Args {
  const FFTCube<float>& c;
  float* rho;
  float2* work;
  const float* G;
  int64_t nbox;
  float div3, div1;
  hipStream_t s;
  KTimer* tm;
  const char* tag;
};
template <int N>
bool one(const Args& a) {
  if constexpr (plane_ok(N))
    return run_plane<float, N>(a.c, a.rho, a.work, a.G, a.nbox, a.div3, a.div1, a.s, a.tm, a.tag, nullptr);
  return false;
}
template <int... I>
bool any(const Args& a, std::integer_sequence<int, I...>) {
  return ((a.c.n == kFrom + 2 * I && one<kFrom + 2 * I>(a)) || ...);
}

}  // namespace

bool fft_convolve_plane_even(const FFTCube<float>& c, float* rho, float2* work, const float* G, int64_t nbox,
                             float div3, float div1, hipStream_t s, KTimer* tm, const char* tag) {
  return any(Args{c, rho, work, G, nbox, div3, div1, s, tm, tag},
             std::make_integer_sequence<int, (kTo - kFrom) / 2 + 1>{});
}

}  // namespace cube
