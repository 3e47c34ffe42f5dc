// pmdiff.hip -- differentiable PM-only force on periodic meshes and its
// vector-Jacobian products (the C-ABI of include/cube_pm.h).
//
// Forward:  rho = TSC deposit, phi = c2r(G r2c(rho))/n^3, F_d = D_d phi (the
// 4-point stencil of particle_mesh.f90:237-242), acc = TSC interpolation of F.
// Adjoint of acc with respect to the positions, given g = dL/dacc:
//   Fbar_d   = TSC deposit of g_d                     (transpose of interpolation)
//   phibar   = sum_d D_d^T Fbar_d = -sum_d D_d Fbar_d (D_d is antisymmetric)
//   rhobar   = c2r(G r2c(phibar))/n^3                 (G real and even: self-adjoint)
//   dL/dx_p  = sum_m grad W(x_p - m) [F(m).g_p + rhobar(m)]
// Mesh sums use integer atomics on fixed-point values: 2^-32 units for the
// TSC density, 2^-31 for the CIC density, and for the signed adjoint
// deposits a power-of-two scale chosen from max|g| so that every
// contribution is a 32-bit integer and no sum can overflow.  Integer addition is
// associative, so every output is independent of thread order.
#include <algorithm>
#include <cmath>
#include <initializer_list>
#include <mutex>
#include <string>

#include "../../include/cube_p3m.h"
#include "../../include/cube_pm.h"
#include "common.h"
#include "fft.h"
#include "grid.h"
#include "growbuf.h"
#include "pm.h"

// The allocation-free CIC entry point's device scratch (sized and explained
// with kScratchCells below).
static __device__ __align__(256) unsigned long long scratch[(int64_t)1 << 23];

namespace cube {
namespace {

struct DeviceMem {
  static void* alloc(size_t bytes) {
    void* p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess)
      throw Error(CUBE_ERR_HIP, "hipMalloc of " + std::to_string(bytes) + " bytes failed");
    return p;
  }
  static void free(void* p) { (void)hipFree(p); }
};
template <typename T>
using PMBuf = GrowBuf<T, DeviceMem>;

constexpr double kFix = 4294967296.0;  // 2^32

// Fixed device scratch of cube_pm_cic_noalloc: the fixed-point CIC
// accumulator (batch * nw^3 64-bit cells, at most kScratchCells = 64 MiB).
// Each GPU the library runs on holds its own copy of the array, at its own
// address, until the process ends.  In host code `scratch` names a host-side
// stand-in, never the device memory: host code uses only the per-device
// address from hipGetSymbolAddress (scratch_address below).
constexpr int64_t kScratchCells = (int64_t)1 << 23;
constexpr int kMaxDevices = 64;

std::mutex g_scratch_mu;
unsigned long long* g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on `device` (which must be current),
// looked up once per device.
unsigned long long* scratch_address(int device) {
  if (device < 0 || device >= kMaxDevices) throw Error(CUBE_ERR_ARG, "device ordinal out of range");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    void* ptr = nullptr;
    static_assert(sizeof(::scratch) == sizeof(unsigned long long) * kScratchCells, "scratch size");
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(::scratch));
    if (e != hipSuccess || !ptr)
      throw Error(CUBE_ERR_HIP, std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
    g_scratch_ptr[device] = (unsigned long long*)ptr;
  }
  return g_scratch_ptr[device];
}

__device__ inline int wrapi(int i, int n) {
  if ((unsigned)i < (unsigned)n) return i;
  i %= n;
  return i < 0 ? i + n : i;
}
__device__ inline int up1(int i, int n) { return i + 1 == n ? 0 : i + 1; }
__device__ inline int dn1(int i, int n) { return i == 0 ? n - 1 : i - 1; }

// Particle positions: absolute mesh coordinates (L = 0), or displacements
// from a Lagrangian lattice of L^3 sites per mesh (L > 0): particle p of a
// batch sits at site q = p mod L^3 (x fastest) whose position along each
// axis is (i + 1/2) n / L, plus its displacement.  With displacements the
// floor index and the fraction come from the integer and fractional parts of
// the site position (exact in FP64) plus the FP32 displacement, so their
// rounding is that of the displacement (|s| of a few cells), not of the
// absolute coordinate (up to n cells).
struct Lattice {
  int L = 0;          // sites per dimension; 0 = absolute positions
  double step = 0.0;  // n / L mesh cells between sites
};

// Batch of particle p and its site along the three axes.  All indices fit 32
// bits (checked on the host); a 64-bit division is about 100 instructions.
__device__ inline uint32_t site_of(uint32_t p, uint32_t np, const Lattice& lt, uint32_t c[3]) {
  const uint32_t b = p / np;
  if (lt.L > 0) {
    const uint32_t q = p - b * np, L = (uint32_t)lt.L, qyz = q / L;
    c[0] = q - qyz * L;
    c[2] = qyz / L;
    c[1] = qyz - c[2] * L;
  }
  return b;
}

// One coordinate times `scale`, split: integer part ip and the rest (the whole
// coordinate for absolute positions).
__device__ inline float coord(const float* __restrict__ x, uint32_t p, int d, const uint32_t c[3], const Lattice& lt,
                              double scale, int& ip) {
  ip = 0;
  const float v = x[3 * (int64_t)p + d];
  if (lt.L == 0) return v * (float)scale;
  const double s = ((double)c[d] + 0.5) * lt.step * scale, f = floor(s);
  ip = (int)f;
  return (float)(s - f) + v * (float)scale;
}

// TSC: nearest point i = floor(x + 1/2) in [0, n) and d = x - i.
__device__ inline void tsc_point(const float* __restrict__ x, uint32_t p, uint32_t np, int n, const Lattice& lt,
                                 uint32_t& b, int i[3], float dd[3]) {
  uint32_t c[3];
  b = site_of(p, np, lt, c);
  for (int d = 0; d < 3; ++d) {
    int ip;
    const float v = coord(x, p, d, c, lt, 1.0, ip);
    const float fi = floorf(v + 0.5f);
    dd[d] = v - fi;
    i[d] = wrapi((int)fi + ip, n);
  }
}
// Weights on points i-1, i, i+1 and their derivatives.
__device__ inline void tsc_w(float d, float w[3]) {
  const float a = 0.5f - d, b = 0.5f + d;
  w[0] = 0.5f * a * a;
  w[1] = 0.75f - d * d;
  w[2] = 0.5f * b * b;
}
__device__ inline void tsc_dw(float d, float dw[3]) {
  dw[0] = -(0.5f - d);
  dw[1] = -2.0f * d;
  dw[2] = 0.5f + d;
}

// CIC: cell i = floor(x scale) in [0, nw) and f = x scale - i; weights 1 - f, f on
// points i, i+1.
__device__ inline void cic_point(const float* __restrict__ x, uint32_t p, uint32_t np, int nw, float scale,
                                 const Lattice& lt, uint32_t& b, int i[3], float f[3]) {
  uint32_t c[3];
  b = site_of(p, np, lt, c);
  for (int d = 0; d < 3; ++d) {
    int ip;
    const float y = coord(x, p, d, c, lt, (double)scale, ip);
    const float fi = floorf(y);
    i[d] = wrapi((int)fi + ip, nw);
    f[d] = y - fi;
  }
}
__device__ inline void cic_w(float f, float w[2]) {
  w[0] = 1.0f - f;
  w[1] = f;
}

// The point of either kind (scale is of CIC alone).
template <bool CIC>
__device__ inline void point(const float* __restrict__ x, uint32_t p, uint32_t np, int n, float scale,
                             const Lattice& lt, uint32_t& b, int i[3], float d[3]) {
  if (CIC) cic_point(x, p, np, n, scale, lt, b, i, d);
  else tsc_point(x, p, np, n, lt, b, i, d);
}

__global__ void k_zero_u32(unsigned int* a, int64_t n) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) a[t] = 0;
}

__global__ void k_zero_u64(unsigned long long* a, int64_t n) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) a[t] = 0;
}

// max|g| of a call, in slots one cache line apart (float bits: non-negative
// floats order as integers).
constexpr int kSlots = 64, kSlotStride = 32;

// Power-of-two scale S with max|g| * S in [2^30, 2^31): every contribution
// W g S (W <= 0.42) rounds to a 32-bit integer, and a mesh sum of at most
// 27 * ntot of them stays far inside 64 bits.  The rounding is 2^-31 of
// max|g| per contribution.  All lanes of a wavefront take part.
__device__ inline double fix_scale(const unsigned int* gmax) {
  float m = __uint_as_float(gmax[(threadIdx.x & 63) * kSlotStride]);
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if (!(m > 0)) return 1.0;
  return ldexp(1.0, 30 - ilogbf(m));
}

// max |g| of a block's threads, valid in thread 0.
template <int NT>
__device__ inline float block_max(float v) {
  __shared__ float red[NT / 64];
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int k = 1; k < NT / 64; ++k) v = fmaxf(v, red[k]);
  return v;
}

// The slots of max |g|: block k writes slot k, block 0 clears those of no block.
__global__ void __launch_bounds__(1024) k_absmax(const float* __restrict__ g, int64_t n, unsigned int* __restrict__ gmax) {
  float v = 0.0f;
  for (int64_t t = (int64_t)blockIdx.x * 1024 + threadIdx.x; t < n; t += (int64_t)gridDim.x * 1024)
    v = fmaxf(v, fabsf(g[t]));
  v = block_max<1024>(v);
  if (threadIdx.x == 0) gmax[blockIdx.x * kSlotStride] = __float_as_uint(v);
  if (blockIdx.x == 0 && threadIdx.x >= gridDim.x && threadIdx.x < kSlots) gmax[threadIdx.x * kSlotStride] = 0;
}

// Deposits of few particles: global atomics, three threads per particle, one a
// z-plane of taps (bound by the latency of a wave's chain of atomics; blocks of
// one wavefront spread them over the chip).  NC = 1: rho += W (fixed point
// 2^-32); NC = 3: Fbar[b][d] += W g_d at scale S.
constexpr int kFew = 63;  // threads of a block that work: 21 particles
// This thread's particle of a launch from p0 on (past the last one, none; below 2^32 either way).
__device__ inline uint32_t few_particle(uint32_t p0) { return p0 + blockIdx.x * (kFew / 3) + threadIdx.x / 3u; }
template <int NC>
__global__ void __launch_bounds__(64) k_tsc_deposit(const float* __restrict__ x, const float* __restrict__ g, uint32_t p0, uint32_t np, uint32_t ntot,
                              int n, Lattice lt, const unsigned int* __restrict__ gmax,
                              unsigned long long* __restrict__ acc) {
  const double S = NC == 3 ? fix_scale(gmax) : 1.0;
  const uint32_t p = few_particle(p0);
  const int k3 = (int)(threadIdx.x % 3u);
  if (threadIdx.x >= kFew || p >= ntot) return;
  uint32_t b;
  int i[3];
  float d[3], w[3][3], gs[3] = {0, 0, 0};
  tsc_point(x, p, np, n, lt, b, i, d);
  for (int k = 0; k < 3; ++k) tsc_w(d[k], w[k]);
  if (NC == 3) {
    for (int k = 0; k < 3; ++k) gs[k] = (float)(g[3 * (int64_t)p + k] * S);
  }
  const int64_t n3 = (int64_t)n * n * n;
  const int xi[3] = {dn1(i[0], n), i[0], up1(i[0], n)}, yi[3] = {dn1(i[1], n), i[1], up1(i[1], n)};
  const int z = k3 == 0 ? dn1(i[2], n) : (k3 == 1 ? i[2] : up1(i[2], n));
  const float wz = k3 == 0 ? w[2][0] : (k3 == 1 ? w[2][1] : w[2][2]);
  unsigned long long* a = acc + (int64_t)b * NC * n3;
  for (int k2 = 0; k2 < 3; ++k2) {
    unsigned long long* row = a + ((int64_t)z * n + yi[k2]) * n;
    for (int k1 = 0; k1 < 3; ++k1) {
      if (NC == 1) {
        const float wyz32 = (w[1][k2] * wz) * 4294967296.0f;  // weights <= 0.42: fits a u32
        atomicAdd(&row[xi[k1]], (unsigned long long)__float2uint_rn(w[0][k1] * wyz32));
      } else {
        const float wt = w[0][k1] * (w[1][k2] * wz);
        for (int k = 0; k < NC; ++k) {
          const int c = __float2int_rn(wt * gs[k]);
          if (c != 0) atomicAdd(&row[k * n3 + xi[k1]], (unsigned long long)(long long)c);
        }
      }
    }
  }
}

// out = acc * unit (as float), acc cleared for the next use.
__global__ void k_fix_to_float(unsigned long long* __restrict__ acc, int64_t n, double unit, float* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  out[t] = (float)((double)acc[t] * unit);
  acc[t] = 0;
}

// out = (signed) acc / S, acc cleared.
__global__ void k_sfix_to_float(unsigned long long* __restrict__ acc, int64_t n, const unsigned int* __restrict__ gmax,
                                float* __restrict__ out) {
  const double S = fix_scale(gmax);
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  out[t] = (float)((double)(long long)acc[t] / S);
  acc[t] = 0;
}

// Order of many particles: a counting sort by pieces of the mesh's rows.  Every
// (z, y) row is cut into segments of 16 cells, each segment into three bins: its
// first cell, the cells between, its last cell; so a tile that spans one segment
// along x and needs the cells next to it reads, of each row, one run of the
// order (two or three at the row's ends).  k_pm_count takes every particle's
// place in its bin (one atomic per run of lanes in the same bin; the order
// within a bin is free, as everything summed over a bin is a sum of integers),
// k_pm_sums and k_pm_scan the bins' starts, k_pm_sort the sorted records: the
// fractions and the cell along x (its row is the bin's), and the particle.  Four meshes of
// 256^3 with 128^3 particles each: 60 + 10 + 28 + 72 us, where lists by tile, each
// particle under the up to eight tiles its taps reach, by an atomic per listing
// in two passes, took 1.6 ms.
constexpr int TX = 16, TY = 8, TZ = 8;  // cells of a tile
constexpr int kBins = 3;                // bins of a segment

__device__ inline uint32_t bin_of(uint32_t b, const int i[3], int n) {
  const int seg = i[0] / TX, c = i[0] % TX, w = min(TX, n - seg * TX);
  return ((b * n + i[2]) * n + i[1]) * ((n + TX - 1) / TX * kBins) + seg * kBins + (c == 0 ? 0 : (c == w - 1 ? 2 : 1));
}

template <bool CIC>
__global__ void __launch_bounds__(256) k_pm_count(const float* __restrict__ x, uint32_t np, uint32_t ntot, int n,
                                                  float scale, Lattice lt, unsigned int* __restrict__ count,
                                                  unsigned int* __restrict__ rank) {
  const uint32_t p = blockIdx.x * 256u + threadIdx.x;
  const int lane = threadIdx.x & 63;
  uint32_t bin = 0xffffffffu;
  if (p < ntot) {
    uint32_t b;
    int i[3];
    float d[3];
    point<CIC>(x, p, np, n, scale, lt, b, i, d);
    bin = bin_of(b, i, n);
  }
  // the first lane of each run of equal bins adds the run's length
  const uint32_t prev = __shfl_up(bin, 1, 64);
  const bool head = lane == 0 || bin != prev;
  const unsigned long long heads = __builtin_amdgcn_ballot_w64(head);
  const unsigned long long upto = heads & (~0ull >> (63 - lane));
  const int first = 63 - __clzll(upto);
  unsigned int base = 0;
  if (head && p < ntot) {
    const unsigned long long later = heads & ~(~0ull >> (63 - lane));
    const int len = (later ? __ffsll((long long)later) - 1 : 64) - lane;
    base = atomicAdd(&count[bin], (unsigned)len);
  }
  base = __shfl(base, first, 64);
  if (p < ntot) rank[p] = base + (unsigned)(lane - first);
}

// Exclusive scan of the counts, which are cleared for the next call: the sums of
// the blocks' chunks of NT * 8, then each chunk after the sum of those before it
// (chunks of 1024 up to 2^20 bins, where blocks are few, else of 8192, where the
// sums before a chunk are many).
__device__ inline unsigned block_exclusive(unsigned v, unsigned* tmp, unsigned& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned s = v;
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned u = __shfl_up(s, o, 64);
    if (lane >= o) s += u;
  }
  if (lane == 63) tmp[wave] = s;
  __syncthreads();
  unsigned before = 0;
  total = 0;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
    before += w < wave ? tmp[w] : 0;
    total += tmp[w];
  }
  __syncthreads();
  return before + s - v;
}

struct alignas(16) Counts {
  unsigned v[8];
};
__device__ inline Counts counts_at(const unsigned int* __restrict__ count, int64_t i, int64_t n) {
  Counts c;
  if (i + 8 <= n) {
    c = *reinterpret_cast<const Counts*>(count + i);
  } else {
    for (int k = 0; k < 8; ++k) c.v[k] = i + k < n ? count[i + k] : 0;
  }
  return c;
}

template <int NT>
__global__ void __launch_bounds__(NT) k_pm_sums(const unsigned int* __restrict__ count, int64_t n,
                                                unsigned int* __restrict__ sums) {
  __shared__ unsigned tmp[NT / 64];
  const Counts c = counts_at(count, ((int64_t)blockIdx.x * NT + threadIdx.x) * 8, n);
  unsigned s = 0, total;
  for (int k = 0; k < 8; ++k) s += c.v[k];
  block_exclusive(s, tmp, total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

template <int NT>
__global__ void __launch_bounds__(NT) k_pm_scan(unsigned int* __restrict__ count, int64_t n,
                                                const unsigned int* __restrict__ sums,
                                                unsigned int* __restrict__ start, unsigned int ntot,
                                                unsigned int* __restrict__ gmax) {
  __shared__ unsigned tmp[NT / 64];
  const int64_t i = ((int64_t)blockIdx.x * NT + threadIdx.x) * 8;
  Counts c = counts_at(count, i, n);
  unsigned before, total, s = 0;
  for (unsigned k = threadIdx.x; k < blockIdx.x; k += NT) s += sums[k];
  block_exclusive(s, tmp, before);
  s = 0;
  for (int k = 0; k < 8; ++k) s += c.v[k];
  unsigned e = before + block_exclusive(s, tmp, total);
  for (int k = 0; k < 8; ++k) {
    const unsigned v = c.v[k];
    c.v[k] = e;
    e += v;
  }
  if (i + 8 <= n) {
    *reinterpret_cast<Counts*>(start + i) = c;
    *reinterpret_cast<Counts*>(count + i) = Counts{};
  } else {
    for (int k = 0; k < 8; ++k)
      if (i + k < n) {
        start[i + k] = c.v[k];
        count[i + k] = 0;
      }
  }
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) start[n] = ntot;
    if (threadIdx.x < kSlots) gmax[threadIdx.x * kSlotStride] = 0;
  }
}

// The records in order, with the particles, or with them and their cotangents (and
// the slots of max |g|), or alone (CIC).
enum class Sort { kPart, kCotangent, kCIC };
template <Sort M>
__global__ void __launch_bounds__(256) k_pm_sort(const float* __restrict__ x, const float* __restrict__ g, uint32_t np,
                                                 uint32_t ntot, int n, float scale, Lattice lt,
                                                 const unsigned int* __restrict__ start,
                                                 const unsigned int* __restrict__ rank, float4* __restrict__ rec,
                                                 unsigned int* __restrict__ part, float4* __restrict__ grec,
                                                 unsigned int* __restrict__ gmax) {
  const uint32_t p = blockIdx.x * 256u + threadIdx.x;
  float m = 0.0f;
  if (p < ntot) {
    uint32_t b;
    int i[3];
    float d[3];
    point<M == Sort::kCIC>(x, p, np, n, scale, lt, b, i, d);
    const uint32_t at = start[bin_of(b, i, n)] + rank[p];
    rec[at] = make_float4(d[0], d[1], d[2], __uint_as_float((uint32_t)i[0]));
    if constexpr (M == Sort::kCotangent) {
      const float* gp = g + 3 * (int64_t)p;
      grec[at] = make_float4(gp[0], gp[1], gp[2], __uint_as_float(p));
      m = fmaxf(fabsf(gp[0]), fmaxf(fabsf(gp[1]), fabsf(gp[2])));
    } else if constexpr (M == Sort::kPart) {
      part[at] = p;
    }
  }
  if constexpr (M == Sort::kCotangent) {
    m = block_max<256>(m);
    unsigned int* slot = gmax + (blockIdx.x % kSlots) * kSlotStride;
    if (threadIdx.x == 0 && __float_as_uint(m) > *(volatile unsigned int*)slot) atomicMax(slot, __float_as_uint(m));
  }
}

// a / d for a < 2^31, d < 2^31, by a multiplication.
struct FastDiv {
  uint32_t d, m, s;
  explicit FastDiv(uint32_t d_) : d(d_), m(0), s(0) {
    uint32_t l = 1;
    while (l < 31 && (1u << l) < d) ++l;
    m = (uint32_t)((((uint64_t)1 << (31 + l)) / d) + 1);
    s = l - 1;
  }
  __device__ uint32_t div(uint32_t a) const { return d == 1 ? a : __umulhi(a, m) >> s; }
};

// The tiles of a batch of meshes.  Workgroups go to the eight XCDs in turn; each
// XCD takes a run of tiles, so that the rows which neighbouring tiles share are
// read into one L2.
struct Tiles {
  FastDiv nx, ny, nz;
  uint32_t n, per;  // tiles, tiles of an XCD
  Tiles(int mesh, int batch)
      : nx((uint32_t)ceil_div(mesh, TX)), ny((uint32_t)ceil_div(mesh, TY)), nz((uint32_t)ceil_div(mesh, TZ)),
        n(nx.d * ny.d * nz.d * (uint32_t)batch), per((uint32_t)ceil_div(n, 8)) {}
  unsigned blocks() const { return 8 * per; }
};

// This workgroup's tile: its origin and width, and its batch (negative: none).
struct Tile {
  int b, tx, o[3], w[3];
};
__device__ inline Tile tile_of(const Tiles& ts, int n) {
  Tile r;
  uint32_t t = (blockIdx.x & 7) * ts.per + (blockIdx.x >> 3), q;
  const bool none = t >= ts.n;
  q = ts.nx.div(t);
  r.tx = (int)(t - q * ts.nx.d);
  r.o[0] = r.tx * TX;
  t = ts.ny.div(q);
  r.o[1] = (int)(q - t * ts.ny.d) * TY;
  q = ts.nz.div(t);
  r.o[2] = (int)(t - q * ts.nz.d) * TZ;
  r.b = none ? -1 : (int)q;
  r.w[0] = min(TX, n - r.o[0]);
  r.w[1] = min(TY, n - r.o[1]);
  r.w[2] = min(TZ, n - r.o[2]);
  return r;
}

// i in [-n, 2n) wrapped
__device__ inline int wrap1(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// The last of `rows` rows whose first entry pre[row] is at or before k.
__device__ inline int row_of(const unsigned* pre, int rows, unsigned k) {
  int lo = 0, hi = rows - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (pre[mid] <= k) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Deposits of many particles: one workgroup per tile sums the taps that fall
// inside it in LDS (u64; signed values as two's complement) and writes its
// cells once.  Contributors are the particles of the tile's cells and of one cell
// around: of each (z, y) row the run of the tile's own bins with the last bin
// before and the first after.  The rows' lengths are scanned in LDS and the
// threads share the whole list, so that a dense tile keeps all of them busy; the
// next record is loaded while the taps of one are added.  NC = 1: the density
// (contribution u32(W 2^32), out = sum / 2^32); NC = 3: the adjoint's vector
// (contribution int(W g S), out = sum / S).  The integers are those of
// k_tsc_deposit: the outputs are the same bit for bit.  Bound by the latency of a
// particle's chain of loads, weights and LDS adds, no pipe being full (four meshes
// of 256^3: 51 % of the vector issue slots, LDS busy 55 % of the cycles, a third of
// it with conflicts, the texture data unit 84 %; NC = 3 39, 61 and 77 %; CIC, four of 128^3,
// 56, 43 and 72 %): 16 x 8 x 8 cells are read by 1.8 times their particles, 8^3 by 2.0
// times.  Few dense tiles (90^3) leave all of them below 60 %.
// Four meshes of 256^3 with 128^3 particles each: 0.24 ms, NC = 3 0.53 ms (lists by
// tile of 8^3: 0.46 and 1.12); three of 90^3, 750 000 particles: 0.060 and 0.11 ms
// (global atomics with their pass to floats: 0.5 and 1.4).  CIC: the density of cube_pm_cic (contribution
// u32(W 2^31)); four meshes of 128^3 with as many particles: 0.07 ms, with the sort
// 0.18 (global atomics 0.65).
template <int NC, bool CIC>
__global__ void __launch_bounds__(256) k_pm_deposit(const float4* __restrict__ rec, const float4* __restrict__ grec,
                                                    int n, Tiles ts, const unsigned int* __restrict__ start,
                                                    const unsigned int* __restrict__ gmax, float* __restrict__ out) {
  constexpr int NT = 256, SY = TX + 1, SZ = TY * SY, NR = (TY + 2) * (TZ + 2);
  constexpr int K = CIC ? 2 : 3, LO = K - 2;  // taps per axis; those below the point (CIC: only cells before reach in)
  constexpr double kUnit = CIC ? 2147483648.0 : kFix;
  __shared__ __align__(16) unsigned long long acc[NC][TZ * SZ];
  __shared__ unsigned beg[3][NR], len[2][NR], pre[NR], wsum[NT / 64];
  const Tile t = tile_of(ts, n);
  if (t.b < 0) return;
  const int ry = t.w[1] + 1 + LO, rows = ry * (t.w[2] + 1 + LO), nseg = (n + TX - 1) / TX;
  static_assert(NC * TZ * SZ % 2 == 0, "cleared in pairs");
  for (int q = threadIdx.x; q < NC * TZ * SZ / 2; q += NT) reinterpret_cast<ulonglong2*>(&acc[0][0])[q] = ulonglong2{};
  unsigned l[3] = {0, 0, 0};
  const int r = threadIdx.x;
  if (r < rows) {
    const int lz = r / ry, ly = r - lz * ry, y = wrap1(t.o[1] + ly - 1, n), z = wrap1(t.o[2] + lz - 1, n);
    const unsigned int* s = start + (((int64_t)t.b * n + z) * n + y) * nseg * kBins;
    const int sb = dn1(t.tx, nseg), sa = up1(t.tx, nseg);
    const int bb = sb * kBins + (n - sb * TX == 1 ? 0 : 2);  // a segment of one cell has it in its first bin
    beg[0][r] = s[bb];
    l[0] = s[bb + 1] - s[bb];
    beg[1][r] = s[t.tx * kBins];
    l[1] = s[(t.tx + 1) * kBins] - s[t.tx * kBins];
    if (!CIC) {
      beg[2][r] = s[sa * kBins];
      l[2] = s[sa * kBins + 1] - s[sa * kBins];
    }
    len[0][r] = l[0];
    len[1][r] = l[1];
  }
  unsigned total, e = block_exclusive(l[0] + l[1] + l[2], wsum, total);
  if (r < rows) pre[r] = e;
  const double S = NC == 3 ? fix_scale(gmax) : 1.0;
  __syncthreads();
  auto fetch = [&](unsigned k, int& row, int& cx, float4& v, float4& g) {
    row = row_of(pre, rows, k);
    unsigned o = k - pre[row];
    int m = 0;
    if (o >= len[0][row]) {
      o -= len[0][row];
      m = 1;
      if (o >= len[1][row]) {
        o -= len[1][row];
        m = 2;
      }
    }
    const unsigned q = beg[m][row] + o;
    v = rec[q];
    if (NC == 3) g = grec[q];
    cx = m;
  };
  int row = 0, m = 0;
  float4 v{}, g{};
  // Long lists (above a particle a cell) in 32 segments, eight to a wavefront and eight
  // lanes to a segment: the 64 particles of a dense row would meet in the same few cells
  // (three meshes of 90^3, 750 000 clustered particles, NC = 3: 151 us with consecutive
  // lanes, 108 so; four of 256^3 with 225 entries a tile 529 and 584).
  unsigned k = threadIdx.x, k1 = total, step = NT;
  if (total > 8 * NT) {
    const unsigned seg = (threadIdx.x >> 6) * 8 + (threadIdx.x & 7);
    k1 = (unsigned)((uint64_t)total * (seg + 1) / 32);
    k = (unsigned)((uint64_t)total * seg / 32) + ((threadIdx.x & 63) >> 3);
    step = 8;
  }
  if (k < k1) fetch(k, row, m, v, g);
  for (; k < k1; k += step) {
    const int lz = row / ry, cy = row - lz * ry - 1, cz = lz - 1;
    const int cx = m == 1 ? (int)__float_as_uint(v.w) - t.o[0] : (m == 0 ? -1 : t.w[0]);
    float w[3][K], gs[3] = {0, 0, 0};
    const float d[3] = {v.x, v.y, v.z};
    for (int c = 0; c < 3; ++c) {
      if constexpr (CIC) cic_w(d[c], w[c]);
      else tsc_w(d[c], w[c]);
    }
    if (NC == 3) {
      gs[0] = (float)(g.x * S);
      gs[1] = (float)(g.y * S);
      gs[2] = (float)(g.z * S);
    }
    if (k + step < k1) fetch(k + step, row, m, v, g);
#pragma unroll
    for (int k3 = 0; k3 < K; ++k3) {
      const int z = cz - LO + k3;
      if ((unsigned)z >= (unsigned)t.w[2]) continue;
#pragma unroll
      for (int k2 = 0; k2 < K; ++k2) {
        const int y = cy - LO + k2;
        if ((unsigned)y >= (unsigned)t.w[1]) continue;
        const float wyz = w[1][k2] * w[2][k3];
#pragma unroll
        for (int k1 = 0; k1 < K; ++k1) {
          const int xx = cx - LO + k1;
          if ((unsigned)xx >= (unsigned)t.w[0]) continue;
          const int c = z * SZ + y * SY + xx;
          if constexpr (CIC) {
            const float wt = w[0][k1] * w[1][k2] * w[2][k3];
            atomicAdd(&acc[0][c], (unsigned long long)__float2uint_rn(wt * 2147483648.0f));
          } else if constexpr (NC == 1) {
            atomicAdd(&acc[0][c], (unsigned long long)__float2uint_rn(w[0][k1] * (wyz * 4294967296.0f)));
          } else {
            const float wt = w[0][k1] * wyz;
            for (int d = 0; d < NC; ++d)
              atomicAdd(&acc[d][c], (unsigned long long)(long long)__float2int_rn(wt * gs[d]));
          }
        }
      }
    }
  }
  __syncthreads();
  // unit is a power of two: the product is the quotient by S
  const double unit = NC == 1 ? 1.0 / kUnit : 1.0 / S;
  const int64_t n3 = (int64_t)n * n * n;
  const int lx = threadIdx.x % TX, ly = (threadIdx.x / TX) % TY, lz0 = threadIdx.x / (TX * TY);
  if (lx >= t.w[0] || ly >= t.w[1]) return;
  float* o = out + (int64_t)t.b * NC * n3 + ((int64_t)(t.o[2] + lz0) * n + (t.o[1] + ly)) * n + (t.o[0] + lx);
  constexpr int DZ = NT / (TX * TY);
#pragma unroll
  for (int lz = 0; lz < TZ; lz += DZ) {
    if (lz + lz0 < t.w[2])
      for (int d = 0; d < NC; ++d) {
        const unsigned long long a = acc[d][(lz + lz0) * SZ + ly * SY + lx];
        o[d * n3] = NC == 1 ? (float)((double)a * unit) : (float)((double)(long long)a * unit);
      }
    o += (int64_t)DZ * n * n;
  }
}

// F[b][d] = D_d phi[b] (periodic); its time is that of its bytes (a 64-bit division
// per index held it to a third of that rate).  V = 4: four cells along x per thread (n a
// multiple of 4, 16-byte aligned meshes).
template <int V>
struct alignas(4 * V) Vec {
  float v[V];
};
template <int V>
__device__ inline Vec<V> ldv(const float* p) {
  return *reinterpret_cast<const Vec<V>*>(p);
}
// At a cell of a mesh of fewer than 2^32: a scalar base and a 32-bit offset of bytes up
// to 1024^3 (!FAR), else of cells.
template <int V, bool FAR>
__device__ inline Vec<V> at_cell(const float* base, uint32_t cell) {
  if constexpr (FAR) return ldv<V>(base + cell);
  else return *reinterpret_cast<const Vec<V>*>(reinterpret_cast<const char*>(base) + 4u * cell);
}
// x-2 .. x+V+1 of a periodic row
template <int V>
__device__ inline void load_row(const float* __restrict__ r, int x, int n, float e[V + 4]) {
  if constexpr (V == 4) {
    const Vec<4> l = ldv<4>(r + (x == 0 ? n - 4 : x - 4)), c = ldv<4>(r + x), h = ldv<4>(r + (x + 4 == n ? 0 : x + 4));
    e[0] = l.v[2];
    e[1] = l.v[3];
    for (int k = 0; k < 4; ++k) e[2 + k] = c.v[k];
    e[6] = h.v[0];
    e[7] = h.v[1];
  } else {
    e[0] = r[x < 2 ? x - 2 + n : x - 2];
    e[1] = r[x < 1 ? x - 1 + n : x - 1];
    e[2] = r[x];
    e[3] = r[x + 1 >= n ? x + 1 - n : x + 1];
    e[4] = r[x + 2 >= n ? x + 2 - n : x + 2];
  }
}

template <int V>
__global__ void __launch_bounds__(256) k_fd_force(const float* __restrict__ phi, int n, uint32_t nthr, float* __restrict__ F) {
  const uint32_t nq = (uint32_t)(n / V), t = blockIdx.x * 256u + threadIdx.x;
  if (t >= nthr) return;
  const uint32_t row = t / nq, plane = row / (uint32_t)n;  // (b, z, y), (b, z)
  const int x = (int)(t - row * nq) * V, y = (int)(row - plane * (uint32_t)n);
  const int64_t b = plane / (uint32_t)n, n2 = (int64_t)n * n, n3 = n2 * n;
  const int z = (int)(plane - (uint32_t)b * (uint32_t)n);
  const float* ph = phi + b * n3;
  const FDWeights<float> W;
  const float c[4] = {W.w0, W.w1, W.w2, W.w3};
  const int s[4] = {-2, -1, 1, 2};
  float e[V + 4], f[3][V];
  load_row<V>(ph + z * n2 + (int64_t)y * n, x, n, e);
  for (int k = 0; k < V; ++k) {
    f[0][k] = e[k] * c[0] + e[k + 1] * c[1] + e[k + 3] * c[2] + e[k + 4] * c[3];
    f[1][k] = f[2][k] = 0;
  }
  for (int q = 0; q < 4; ++q) {
    int yy = y + s[q], zz = z + s[q];
    yy = yy < 0 ? yy + n : (yy >= n ? yy - n : yy);
    zz = zz < 0 ? zz + n : (zz >= n ? zz - n : zz);
    const Vec<V> a = ldv<V>(ph + z * n2 + (int64_t)yy * n + x), d = ldv<V>(ph + zz * n2 + (int64_t)y * n + x);
    for (int k = 0; k < V; ++k) {
      f[1][k] += a.v[k] * c[q];
      f[2][k] += d.v[k] * c[q];
    }
  }
  const int64_t m = z * n2 + (int64_t)y * n + x;
  for (int d = 0; d < 3; ++d) {
    Vec<V> o;
    for (int k = 0; k < V; ++k) o.v[k] = f[d][k];
    *reinterpret_cast<Vec<V>*>(F + (b * 3 + d) * n3 + m) = o;
  }
}

// phibar[b] = -sum_d D_d Fbar[b][d] (transpose of k_fd_force).
template <int V>
__global__ void __launch_bounds__(256) k_fd_adjoint(const float* __restrict__ Fb, int n, uint32_t nthr, float* __restrict__ phib) {
  const uint32_t nq = (uint32_t)(n / V), t = blockIdx.x * 256u + threadIdx.x;
  if (t >= nthr) return;
  const uint32_t row = t / nq, plane = row / (uint32_t)n;  // (b, z, y), (b, z)
  const int x = (int)(t - row * nq) * V, y = (int)(row - plane * (uint32_t)n);
  const int64_t b = plane / (uint32_t)n, n2 = (int64_t)n * n, n3 = n2 * n;
  const int z = (int)(plane - (uint32_t)b * (uint32_t)n);
  const FDWeights<float> W;
  const float c[4] = {W.w0, W.w1, W.w2, W.w3};
  const int s[4] = {-2, -1, 1, 2};
  const float *f0 = Fb + (b * 3 + 0) * n3, *f1 = Fb + (b * 3 + 1) * n3, *f2 = Fb + (b * 3 + 2) * n3;
  float e[V + 4], v[V];
  load_row<V>(f0 + z * n2 + (int64_t)y * n, x, n, e);
  for (int k = 0; k < V; ++k) v[k] = e[k] * c[0] + e[k + 1] * c[1] + e[k + 3] * c[2] + e[k + 4] * c[3];
  for (int q = 0; q < 4; ++q) {
    int yy = y + s[q], zz = z + s[q];
    yy = yy < 0 ? yy + n : (yy >= n ? yy - n : yy);
    zz = zz < 0 ? zz + n : (zz >= n ? zz - n : zz);
    const Vec<V> a = ldv<V>(f1 + z * n2 + (int64_t)yy * n + x), d = ldv<V>(f2 + zz * n2 + (int64_t)y * n + x);
    for (int k = 0; k < V; ++k) v[k] += a.v[k] * c[q] + d.v[k] * c[q];
  }
  Vec<V> o;
  for (int k = 0; k < V; ++k) o.v[k] = -v[k];
  *reinterpret_cast<Vec<V>*>(phib + b * n3 + z * n2 + (int64_t)y * n + x) = o;
}

// The three x taps around cell i of a periodic row: one 12-byte load away from
// the row's ends.
struct __attribute__((packed, aligned(4))) Tap3 {
  float v[3];
};
__device__ inline Tap3 taps(const float* __restrict__ row, int i, int n) {
  if (i > 0 && i < n - 1) return *reinterpret_cast<const Tap3*>(row + i - 1);
  return Tap3{{row[dn1(i, n)], row[i], row[up1(i, n)]}};
}

// Interpolations of few particles, three threads per particle (as in
// k_tsc_deposit), one a z-plane of taps; the first adds the three.
__device__ inline float add3(float v) {
  const float a = __shfl_down(v, 1, 64), b = __shfl_down(v, 2, 64);
  return (v + a) + b;
}

// acc_p = sum W F.
__global__ void __launch_bounds__(64) k_tsc_interp(const float* __restrict__ x, uint32_t p0, uint32_t np, uint32_t ntot, int n,
                                                   Lattice lt, const float* __restrict__ F, float* __restrict__ acc) {
  const uint32_t q = few_particle(p0), p = min(q, ntot - 1);
  const int k3 = (int)(threadIdx.x % 3u);
  uint32_t b;
  int i[3];
  float d[3], w[3][3];
  tsc_point(x, p, np, n, lt, b, i, d);
  for (int k = 0; k < 3; ++k) tsc_w(d[k], w[k]);
  const int64_t n3 = (int64_t)n * n * n;
  const float* Fb = F + (int64_t)b * 3 * n3;
  const int yi[3] = {dn1(i[1], n), i[1], up1(i[1], n)};
  const int z = k3 == 0 ? dn1(i[2], n) : (k3 == 1 ? i[2] : up1(i[2], n));
  const float wz = k3 == 0 ? w[2][0] : (k3 == 1 ? w[2][1] : w[2][2]);
  float a[3] = {0, 0, 0};
#pragma unroll
  for (int k2 = 0; k2 < 3; ++k2) {
    const int64_t row = ((int64_t)z * n + yi[k2]) * n;
    const float wyz = w[1][k2] * wz;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const Tap3 f = taps(Fb + c * n3 + row, i[0], n);
      a[c] = fmaf(wyz, fmaf(w[0][2], f.v[2], fmaf(w[0][1], f.v[1], w[0][0] * f.v[0])), a[c]);
    }
  }
  for (int c = 0; c < 3; ++c) a[c] = add3(a[c]);
  if (k3 == 0 && threadIdx.x < kFew && q < ntot)
    for (int c = 0; c < 3; ++c) acc[3 * (int64_t)p + c] = a[c];
}

// g_x = sum grad W (F.g + rhobar).
__global__ void __launch_bounds__(64) k_tsc_vjp(const float* __restrict__ x, uint32_t p0, uint32_t np, uint32_t ntot, int n,
                                                Lattice lt, const float* __restrict__ F, const float* __restrict__ g,
                                                const float* __restrict__ rhob, float* __restrict__ gx) {
  const uint32_t q = few_particle(p0), p = min(q, ntot - 1);
  const int k3 = (int)(threadIdx.x % 3u);
  uint32_t b;
  int i[3];
  float d[3], w[3][3], dw[3][3];
  tsc_point(x, p, np, n, lt, b, i, d);
  for (int k = 0; k < 3; ++k) {
    tsc_w(d[k], w[k]);
    tsc_dw(d[k], dw[k]);
  }
  const float* gp = g + 3 * (int64_t)p;
  const float g0 = gp[0], g1 = gp[1], g2 = gp[2];
  const int64_t n3 = (int64_t)n * n * n;
  const float *Fb = F + (int64_t)b * 3 * n3, *rb = rhob + (int64_t)b * n3;
  const int yi[3] = {dn1(i[1], n), i[1], up1(i[1], n)};
  const int z = k3 == 0 ? dn1(i[2], n) : (k3 == 1 ? i[2] : up1(i[2], n));
  const float wz = k3 == 0 ? w[2][0] : (k3 == 1 ? w[2][1] : w[2][2]);
  const float dwz = k3 == 0 ? dw[2][0] : (k3 == 1 ? dw[2][1] : dw[2][2]);
  float o[3] = {0, 0, 0};
#pragma unroll
  for (int k2 = 0; k2 < 3; ++k2) {
    const int64_t row = ((int64_t)z * n + yi[k2]) * n;
    const Tap3 f0 = taps(Fb + row, i[0], n), f1 = taps(Fb + n3 + row, i[0], n), f2 = taps(Fb + 2 * n3 + row, i[0], n),
               r = taps(rb + row, i[0], n);
    float sw = 0, sd = 0;  // sums along x with the weights and their derivatives
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float s = fmaf(f0.v[k], g0, fmaf(f1.v[k], g1, fmaf(f2.v[k], g2, r.v[k])));
      sw = fmaf(w[0][k], s, sw);
      sd = fmaf(dw[0][k], s, sd);
    }
    o[0] = fmaf(w[1][k2] * wz, sd, o[0]);
    o[1] = fmaf(dw[1][k2] * wz, sw, o[1]);
    o[2] = fmaf(w[1][k2] * dwz, sw, o[2]);
  }
  for (int c = 0; c < 3; ++c) o[c] = add3(o[c]);
  if (k3 == 0 && threadIdx.x < kFew && q < ntot)
    for (int c = 0; c < 3; ++c) gx[3 * (int64_t)p + c] = o[c];
}

// Interpolations of many particles: one workgroup per tile holds the force of its
// cells and of one cell around in LDS, as one float4 per cell (with the
// convolved adjoint density in VJP), and its particles, sorted, read 27 of
// them each.  F is the meshes (phi == nullptr), or formed here from the tile's
// part of phi: then no force mesh is read, or written, at all.  V = 4: quads
// along x (n a multiple of 4, aligned meshes).  VJP: g_x = sum grad W (F.g +
// rhobar); else acc = sum W F.  Bound by the latency of its three phases (three
// workgroups of 49 KB share a CU; LDS is busy 65 % of the cycles, half of it with
// conflicts, the vector pipe 28 % of its issue slots, the texture data unit 71 %; VJP 47, 28
// and 85 %).
// Four meshes of 256^3 with 128^3 particles each: 0.47 ms, VJP 0.56 ms, where
// force meshes written and gathered from took 0.31 + 0.50 and 0.63 ms.
template <bool VJP, int V, bool FAR>
__global__ void __launch_bounds__(512) k_pm_gather(const float4* __restrict__ rec,
                                                   const unsigned int* __restrict__ part,
                                                   const float4* __restrict__ grec, int n, Tiles ts,
                                                   const unsigned int* __restrict__ start,
                                                   const float* __restrict__ phi, const float* __restrict__ F,
                                                   const float* __restrict__ rhob, float* __restrict__ out) {
  constexpr int NT = 512, FX = TX + 2, FY = TY + 2, FZ = TZ + 2;  // cells with a force
  constexpr int PX = TX + 8, PY = TY + 6, PZ = TZ + 6;            // of phi: x from -4, y and z from -3
  // lanes of the stencil loop go along x quads, then z: rows of phi are 64 bytes
  // apart modulo the banks, and an odd plane of fs puts its quads in different ones
  constexpr int FS = FY * FX + 1;
  static_assert(PY * PX * 4 % 256 == 64 && FS % 2 == 1, "conflict-free strides");
  __shared__ float4 fs[FZ * FS];
  __shared__ __align__(16) float ps[PZ * PY * PX];
  __shared__ unsigned beg[TY * TZ], pre[TY * TZ + 1];
  const Tile t = tile_of(ts, n);
  if (t.b < 0) return;
  const int rows = t.w[1] * t.w[2], nseg = (n + TX - 1) / TX;
  const int64_t n2 = (int64_t)n * n, n3 = n2 * n;
  // the tile's part of phi is on its way while the rows are scanned
  constexpr int NL = PZ * PY * (PX / V), NI = (NL + NT - 1) / NT;
  Vec<V> in[NI];
  if (phi) {
    const float* pb = phi + t.b * n3;
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      const int q = min(k * NT + (int)threadIdx.x, NL - 1);
      const int row = q / (PX / V), x = (q - row * (PX / V)) * V, pz = row / PY, py = row - pz * PY;
      // (rows and columns of a ragged tile that no cell needs repeat the last one)
      const int z = wrap1(t.o[2] + min(pz, t.w[2] + 5) - 3, n), y = wrap1(t.o[1] + min(py, t.w[1] + 5) - 3, n),
                gx = wrap1(min(t.o[0] + x - 4, V == 4 ? n : n + 2), n);
      in[k] = at_cell<V, FAR>(pb, ((uint32_t)z * n + y) * n + gx);
    }
  }
  if (threadIdx.x < 64) {  // at most 64 rows: the first wavefront's lanes
    unsigned l = 0;
    if ((int)threadIdx.x < rows) {
      const int lz = threadIdx.x / t.w[1], ly = threadIdx.x - lz * t.w[1];
      const unsigned int* s =
          start + ((((int64_t)t.b * n + t.o[2] + lz) * n + t.o[1] + ly) * nseg + t.tx) * kBins;
      beg[threadIdx.x] = s[0];
      l = s[kBins] - s[0];
    }
    unsigned e = l;
    for (int o = 1; o < 64; o <<= 1) {
      const unsigned u = __shfl_up(e, o, 64);
      if ((int)threadIdx.x >= o) e += u;
    }
    pre[threadIdx.x] = e - l;
    if (threadIdx.x == 63) pre[64] = e;
  }
  const float* rb = VJP ? rhob + t.b * n3 : nullptr;
  if (phi) {
#pragma unroll
    for (int k = 0; k < NI; ++k) {
      const int q = k * NT + (int)threadIdx.x;
      if (q < NL) *reinterpret_cast<Vec<V>*>(&ps[q * V]) = in[k];
    }
  }
  __syncthreads();
  const unsigned total = pre[64];
  if (total == 0) return;
  // a particle's record, on its way before the forces are formed or the taps of the last one are read
  int row = 0;
  float4 v{}, g{};
  auto fetch = [&](unsigned k) {
    row = row_of(pre, rows, k);
    const unsigned q = beg[row] + (k - pre[row]);
    v = rec[q];
    if (VJP) g = grec[q];
    else g.w = __uint_as_float(part[q]);
  };
  if (threadIdx.x < total) fetch(threadIdx.x);
  if (phi) {
    const FDWeights<float> W;
    const float c[4] = {W.w0, W.w1, W.w2, W.w3};
    const int s[4] = {-2, -1, 1, 2};
    // quads of own cells, then the single cells at the two ends
    constexpr int NQ = FZ * FY * (TX / 4);
    for (int q = threadIdx.x; q < NQ; q += NT) {
      const int row = q / (TX / 4), x = (q - row * (TX / 4)) * 4, fy = row / FZ, fz = row - fy * FZ;
      const float* p0 = &ps[((fz + 2) * PY + fy + 2) * PX + x + 4];
      const Vec<4> a = ldv<4>(p0 - 4), m = ldv<4>(p0), h = ldv<4>(p0 + 4);
      const float ex[8] = {a.v[2], a.v[3], m.v[0], m.v[1], m.v[2], m.v[3], h.v[0], h.v[1]};
      float f[3][4];
      for (int k = 0; k < 4; ++k) {
        f[0][k] = fmaf(ex[k + 4], c[3], fmaf(ex[k + 3], c[2], fmaf(ex[k + 1], c[1], ex[k] * c[0])));
        f[1][k] = f[2][k] = 0;
      }
      for (int j = 0; j < 4; ++j) {
        const Vec<4> u = ldv<4>(p0 + s[j] * PX), v = ldv<4>(p0 + s[j] * (PX * PY));
        for (int k = 0; k < 4; ++k) {
          f[1][k] = fmaf(u.v[k], c[j], f[1][k]);
          f[2][k] = fmaf(v.v[k], c[j], f[2][k]);
        }
      }
      Vec<4> r{};
      if (VJP) {
        const uint32_t row0 =
            ((uint32_t)wrap1(t.o[2] + min(fz, t.w[2] + 1) - 1, n) * n + wrap1(t.o[1] + min(fy, t.w[1] + 1) - 1, n)) * n;
        const int gx = t.o[0] + x;
        if (V == 4) {
          r = at_cell<4, FAR>(rb, row0 + wrap1(min(gx, n), n));
        } else {
          for (int k = 0; k < 4; ++k) r.v[k] = at_cell<1, FAR>(rb, row0 + wrap1(min(gx + k, n), n)).v[0];
        }
      }
      float4* dst = &fs[fz * FS + fy * FX + x + 1];
      for (int k = 0; k < 4; ++k) dst[k] = make_float4(f[0][k], f[1][k], f[2][k], r.v[k]);
    }
    // the cell before the tile and the one after it; in a ragged tile the latter
    // is one of the quads' (their cells beyond the row's end wrap as phi does)
    for (int q = threadIdx.x; q < 2 * FZ * FY; q += NT) {
      const int row = q >> 1, x = (q & 1) ? TX : -1, fy = row / FZ, fz = row - fy * FZ;
      const float* p0 = &ps[((fz + 2) * PY + fy + 2) * PX + x + 4];
      float f[3];
      f[0] = fmaf(p0[2], c[3], fmaf(p0[1], c[2], fmaf(p0[-1], c[1], p0[-2] * c[0])));
      f[1] = f[2] = 0;
      for (int j = 0; j < 4; ++j) {
        f[1] = fmaf(p0[s[j] * PX], c[j], f[1]);
        f[2] = fmaf(p0[s[j] * (PX * PY)], c[j], f[2]);
      }
      float r = 0;
      if (VJP)
        r = at_cell<1, FAR>(rb, ((uint32_t)wrap1(t.o[2] + min(fz, t.w[2] + 1) - 1, n) * n +
                                 wrap1(t.o[1] + min(fy, t.w[1] + 1) - 1, n)) * n +
                                    wrap1(min(t.o[0] + x, n), n)).v[0];
      fs[fz * FS + fy * FX + x + 1] = make_float4(f[0], f[1], f[2], r);
    }
  } else {
    const float* Fb = F + t.b * 3 * n3;
    for (int q = threadIdx.x; q < FZ * FY * FX; q += NT) {
      const int row = q / FX, x = q - row * FX, fz = row / FY, fy = row - fz * FY;
      const int64_t m = wrapi(t.o[2] + fz - 1, n) * n2 + (int64_t)wrapi(t.o[1] + fy - 1, n) * n + wrapi(t.o[0] + x - 1, n);
      fs[fz * FS + fy * FX + x] = make_float4(Fb[m], Fb[n3 + m], Fb[2 * n3 + m], VJP ? rb[m] : 0.0f);
    }
  }
  __syncthreads();
  for (unsigned k = threadIdx.x; k < total; k += NT) {
    const int64_t p = __float_as_uint(g.w);
    const int lz = row / t.w[1], ly = row - lz * t.w[1], lx = (int)__float_as_uint(v.w) - t.o[0];
    float w[3][3], dw[3][3], a[3] = {0, 0, 0};
    const float d[3] = {v.x, v.y, v.z}, gx = g.x, gy = g.y, gz = g.z;
    for (int c = 0; c < 3; ++c) {
      tsc_w(d[c], w[c]);
      tsc_dw(d[c], dw[c]);
    }
    const float4* f0 = &fs[lz * FS + ly * FX + lx];
    if (k + NT < total) fetch(k + NT);
#pragma unroll
    for (int k3 = 0; k3 < 3; ++k3)
#pragma unroll
      for (int k2 = 0; k2 < 3; ++k2) {
        const float4 *f = f0 + k3 * FS + k2 * FX, fa = f[0], fb = f[1], fc = f[2];
        if (VJP) {
          const float s0 = fmaf(fa.x, gx, fmaf(fa.y, gy, fmaf(fa.z, gz, fa.w))),
                      s1 = fmaf(fb.x, gx, fmaf(fb.y, gy, fmaf(fb.z, gz, fb.w))),
                      s2 = fmaf(fc.x, gx, fmaf(fc.y, gy, fmaf(fc.z, gz, fc.w)));
          const float sw = fmaf(w[0][2], s2, fmaf(w[0][1], s1, w[0][0] * s0)),
                      sd = fmaf(dw[0][2], s2, fmaf(dw[0][1], s1, dw[0][0] * s0));
          a[0] = fmaf(w[1][k2] * w[2][k3], sd, a[0]);
          a[1] = fmaf(dw[1][k2] * w[2][k3], sw, a[1]);
          a[2] = fmaf(w[1][k2] * dw[2][k3], sw, a[2]);
        } else {
          const float wyz = w[1][k2] * w[2][k3];
          a[0] = fmaf(wyz, fmaf(w[0][2], fc.x, fmaf(w[0][1], fb.x, w[0][0] * fa.x)), a[0]);
          a[1] = fmaf(wyz, fmaf(w[0][2], fc.y, fmaf(w[0][1], fb.y, w[0][0] * fa.y)), a[1]);
          a[2] = fmaf(wyz, fmaf(w[0][2], fc.z, fmaf(w[0][1], fb.z, w[0][0] * fa.z)), a[2]);
        }
      }
    for (int c = 0; c < 3; ++c) out[3 * p + c] = a[c];
  }
}

// CIC density of x*scale on nw^3 (fixed point 2^-31).
__global__ void k_cic_deposit(const float* __restrict__ x, uint32_t np, uint32_t ntot, int nw, float scale, Lattice lt,
                              unsigned long long* __restrict__ acc) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= ntot) return;
  uint32_t b;
  int i[3];
  float f[3], w[3][2];
  cic_point(x, p, np, nw, scale, lt, b, i, f);
  for (int k = 0; k < 3; ++k) cic_w(f[k], w[k]);
  const int64_t n3 = (int64_t)nw * nw * nw;
  unsigned long long* a = acc + (int64_t)b * n3;
  const int xi[2] = {i[0], up1(i[0], nw)}, yi[2] = {i[1], up1(i[1], nw)}, zi[2] = {i[2], up1(i[2], nw)};
  for (int k3 = 0; k3 < 2; ++k3)
    for (int k2 = 0; k2 < 2; ++k2)
      for (int k1 = 0; k1 < 2; ++k1) {
        const float wt = w[0][k1] * w[1][k2] * w[2][k3];  // <= 1: fits a u32 at 2^31
        atomicAdd(&a[((int64_t)zi[k3] * nw + yi[k2]) * nw + xi[k1]],
                  (unsigned long long)__float2uint_rn(wt * 2147483648.0f));
      }
}

__global__ void k_cic_vjp(const float* __restrict__ x, uint32_t np, uint32_t ntot, int nw, float scale, Lattice lt,
                          const float* __restrict__ grho, float* __restrict__ gx) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= ntot) return;
  uint32_t b;
  int i[3];
  float f[3], w[3][2];
  cic_point(x, p, np, nw, scale, lt, b, i, f);
  for (int k = 0; k < 3; ++k) cic_w(f[k], w[k]);
  const int64_t n3 = (int64_t)nw * nw * nw;
  const float dw[2] = {-1.0f, 1.0f};
  const float* gr = grho + (int64_t)b * n3;
  const int xi[2] = {i[0], up1(i[0], nw)}, yi[2] = {i[1], up1(i[1], nw)}, zi[2] = {i[2], up1(i[2], nw)};
  float o[3] = {0, 0, 0};
  for (int k3 = 0; k3 < 2; ++k3)
    for (int k2 = 0; k2 < 2; ++k2)
      for (int k1 = 0; k1 < 2; ++k1) {
        const float v = gr[((int64_t)zi[k3] * nw + yi[k2]) * nw + xi[k1]];
        o[0] = fmaf(dw[k1] * w[1][k2] * w[2][k3], v, o[0]);
        o[1] = fmaf(w[0][k1] * dw[k2] * w[2][k3], v, o[1]);
        o[2] = fmaf(w[0][k1] * w[1][k2] * dw[k3], v, o[2]);
      }
  for (int d = 0; d < 3; ++d) gx[3 * (int64_t)p + d] = o[d] * scale;
}

inline unsigned nblk(int64_t n, int t = 256) { return (unsigned)((n + t - 1) / t); }
// Launches over n cells, a thread each: fn(blocks of 256, first cell, cells), once up to 2^30
// cells and once more for every 2^30 of the largest meshes (three of 1126^3 are more than 2^32,
// as many threads as no launch dimension holds).  Blocks that go on along y or threads
// that go on over the cells hold up all sizes (two meshes of 256^3 to floats 136 and 128 us,
// against 114).
template <class Fn>
inline void over_cells(int64_t n, Fn&& fn) {
  in_pieces(n, (int64_t)1 << 30, [&](int64_t at, int64_t m) { fn(dim3(nblk(m)), at, m); });
}
inline void zero_cells(unsigned long long* a, int64_t n, hipStream_t s) {
  over_cells(n, [&](dim3 grid, int64_t at, int64_t m) {
    hipLaunchKernelGGL(k_zero_u64, grid, dim3(256), 0, s, a + at, m);
  });
}
// Sums to floats (fixed point of `unit`), cleared.
inline void fix_to_float(unsigned long long* acc, int64_t n, double unit, float* out, hipStream_t s) {
  over_cells(n, [&](dim3 grid, int64_t at, int64_t m) {
    hipLaunchKernelGGL(k_fix_to_float, grid, dim3(256), 0, s, acc + at, m, unit, out + at);
  });
}

}  // namespace
}  // namespace cube

using namespace cube;

struct cube_pm_ctx {
  int device = 0;
  cube_pm_config cfg{};
  int64_t n3 = 0;
  FFTCube<float> fc;
  PMBuf<float> G, mesh, Fs, Fbar;
  PMBuf<float2> work;
  PMBuf<unsigned long long> acc;   // B*3*n^3, kept zero between calls
  PMBuf<unsigned long long> accw;  // of the largest CIC density that acc cannot hold, kept zero
  PMBuf<unsigned int> gmax;
  // the particles' order: bin counts (kept zero) and starts, chunk sums, places
  // in the bins, sorted records, particles and cotangents
  PMBuf<unsigned int> bcount, bstart, bsums, rank, part;
  PMBuf<float4> rec, grec;
  Lattice lat;
  std::string err;

  // a captured call's graph holds the addresses of the order's buffers
  void hold_order() {
    for (PMBuf<unsigned int>* b : {&bcount, &bstart, &bsums, &rank, &part}) b->hold();
    rec.hold();
    grec.hold();
  }
  int64_t nbins(int64_t m) const { return cfg.batch * m * m * ceil_div(m, TX) * kBins; }
  static bool capturing(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone;
  }
  // the buffers of an order of ntot particles on meshes of m^3 (fewer than 2^32 cells) are
  // there, or can be made
  bool can_sort(int64_t ntot, int64_t m, size_t have, hipStream_t s) const {
    if (m > 1625 || nbins(m) >= ((int64_t)1 << 31)) return false;
    return ((size_t)nbins(m) <= bcount.n && (size_t)ntot <= rank.n && (size_t)ntot <= rec.n && (size_t)ntot <= have) ||
           !capturing(s);
  }
  // Many particles are sorted first; below these numbers the launches of that form
  // cost more than the global atomics of the other (which also serves meshes
  // beyond 1625 points, and a stream under capture whose order buffers would have
  // to grow).  Measured sorted / not, us, with phi: forces of 17000 particles on
  // 48^3 39 / 50, 128^3 68 / 81, 256^3 302 / 317, 512^3 5480 / 5750; adjoints of 8192
  // on 48^3 46 / 65, 128^3 83 / 114, 256^3 421 / 604, 512^3 6390 / 7700; where F is
  // asked for, which the sorted form's gather does not read, it is up to 16 % slower on
  // meshes of more than some 250 cells a particle (256^3, 25000: 374 / 337) and
  // faster below (100000: 385 / 481).
  static constexpr int64_t kSortFrom = 16384, kSortFromG = 8192;
  // A tile's particles are one workgroup's, so a mesh of a few tiles would wait for as
  // few workgroups: the measure is the largest tile's share of the cells.  Sorted / not,
  // us, 300000 particles: forces on 12^3 (a share of 1/2.3) 2350 / 790, 18^3 (1/5.7) 930 /
  // 530, 22^3 (1/10) 541 / 470, 24^3 (1/14) 427 / 485; adjoints on 18^3 2000 / 1710,
  // 20^3 (1/8) 1474 / 1473, 22^3 1135 / 1653; densities on 16^3 (1/4) 535 / 103, 24^3 174 /
  // 126, 28^3 (1/21) 120 / 119 (130000 particles 61 / 56), 32^3 (1/32) 90 / 108 (47 / 51).
  static constexpr int64_t kShare = 12, kShareG = 8, kShareCIC = 20, kShareCICFew = 32;
  bool shared(int64_t m, int64_t among) const {
    const int64_t largest = std::min<int64_t>(m, TX) * std::min<int64_t>(m, TY) * std::min<int64_t>(m, TZ);
    return cfg.batch * m * m * m >= among * largest;
  }
  bool sorted(int64_t ntot, bool with_g, hipStream_t s) const {
    return ntot >= (with_g ? kSortFromG : kSortFrom) && shared(cfg.n, with_g ? kShareG : kShare) &&
           can_sort(ntot, cfg.n, with_g ? grec.n : part.n, s);
  }
  // CIC densities, eight atomics a particle, of 65536 particles anywhere (sorted / not,
  // us: 32^3 33 / 31, 48^3 25 / 31, 256^3 59 / 68).  Sites of a lattice come in the order of
  // the mesh, which suits the atomics as long as particles have moved little and cells
  // hold several (rms of 0.6 and 2 spacings): 98304 particles on 8 cells each 23 / 22
  // and 26 / 42, 110592 on one 28 / 18 and 35 / 29, 131072 on 3.4 24 / 22 and 28 / 41, 221184 on
  // one 28 / 33 and 40 / 65, 65536 on 64 29 / 33 and 31 / 40.
  bool cic_sorted(int64_t ntot, int64_t nw, hipStream_t s) const {
    const int64_t cells = cfg.batch * nw * nw * nw;
    int64_t from = lat.L == 0 ? 65536 : 60000 + 120000 * ntot / cells;
    if (!shared(nw, kShareCICFew)) from = std::max<int64_t>(from, 262144);
    // meshes below 8 points are all halo
    return nw >= 8 && nw <= 1024 && shared(nw, kShareCIC) && ntot >= from && can_sort(ntot, nw, SIZE_MAX, s);
  }
  // bin counts, starts and places of x on meshes of m^3 (and gmax cleared)
  template <bool CIC>
  void bin(const float* x, int64_t np, int m, float scale, hipStream_t s) {
    const int64_t ntot = np * cfg.batch, nb = nbins(m);
    const bool few = nb <= 1 << 20;
    const unsigned nch = (unsigned)ceil_div(nb, few ? 1024 : 8192);
    bsums.ensure((size_t)ceil_div(nb, 1024));
    bstart.ensure((size_t)nb + 1);
    rank.ensure((size_t)ntot);
    rec.ensure((size_t)ntot);
    if ((size_t)nb > bcount.n)
      hipLaunchKernelGGL(k_zero_u32, dim3(nblk(nb)), dim3(256), 0, s, bcount.ensure((size_t)nb), nb);
    const uint32_t untot = (uint32_t)ntot;
    hipLaunchKernelGGL(k_pm_count<CIC>, dim3(nblk(ntot)), dim3(256), 0, s, x, (uint32_t)np, untot, m, scale, lat,
                       bcount.p, rank.p);
    if (few) {
      hipLaunchKernelGGL(k_pm_sums<128>, dim3(nch), dim3(128), 0, s, bcount.p, nb, bsums.p);
      hipLaunchKernelGGL(k_pm_scan<128>, dim3(nch), dim3(128), 0, s, bcount.p, nb, bsums.p, bstart.p, untot, gmax.p);
    } else {
      hipLaunchKernelGGL(k_pm_sums<1024>, dim3(nch), dim3(1024), 0, s, bcount.p, nb, bsums.p);
      hipLaunchKernelGGL(k_pm_scan<1024>, dim3(nch), dim3(1024), 0, s, bcount.p, nb, bsums.p, bstart.p, untot, gmax.p);
    }
  }
  template <Sort M>
  void place(const float* x, const float* g, int64_t np, int m, float scale, hipStream_t s) {
    const int64_t ntot = np * cfg.batch;
    hipLaunchKernelGGL(k_pm_sort<M>, dim3(nblk(ntot)), dim3(256), 0, s, x, g, (uint32_t)np, (uint32_t)ntot, m, scale,
                       lat, bstart.p, rank.p, rec.p, part.p, grec.p, gmax.p);
    CUBE_HIP(hipGetLastError());
    if (capturing(s)) hold_order();
  }
  // the order of x, with the cotangents g and the slots of their maximum (g may be null)
  void sort(const float* x, const float* g, int64_t np, hipStream_t s) {
    bin<false>(x, np, cfg.n, 1.0f, s);
    if (g) {
      grec.ensure((size_t)(np * cfg.batch));
      place<Sort::kCotangent>(x, g, np, cfg.n, 1.0f, s);
    } else {
      part.ensure((size_t)(np * cfg.batch));
      place<Sort::kPart>(x, g, np, cfg.n, 1.0f, s);
    }
  }
  // Launches of the forms for few particles, fn(blocks, first particle): one, but for more
  // particles than fit the threads of a launch dimension.
  template <class Fn>
  static void over_few(int64_t ntot, Fn&& fn) {
    in_pieces(ntot, ((int64_t)1 << 25) * (kFew / 3),
              [&](int64_t p0, int64_t m) { fn(dim3((unsigned)ceil_div(m, kFew / 3)), (uint32_t)p0); });
  }

  void check_np(int64_t np) const {
    if (np <= 0) throw Error(CUBE_ERR_ARG, "np must be positive");
    if (lat.L > 0 && np != (int64_t)lat.L * lat.L * lat.L)
      throw Error(CUBE_ERR_ARG, "with lattice displacements np must be lattice^3");
    if (np * cfg.batch > 0xffffff00ll) throw Error(CUBE_ERR_ARG, "more particles than threads in a launch");
  }
  // D_d of a mesh, or its transpose
  void fd(bool adjoint, const float* in, float* out, hipStream_t s) {
    const int n = cfg.n, v = quads(n, in, out) ? 4 : 1;
    const int64_t nthr = (int64_t)cfg.batch * n3 / v;
    if (nthr > 0xffffff00ll) throw Error(CUBE_ERR_ARG, "more cells than threads in a launch");
    const dim3 grid(nblk(nthr));
    if (!adjoint && v == 4) hipLaunchKernelGGL(k_fd_force<4>, grid, dim3(256), 0, s, in, n, (uint32_t)nthr, out);
    else if (!adjoint) hipLaunchKernelGGL(k_fd_force<1>, grid, dim3(256), 0, s, in, n, (uint32_t)nthr, out);
    else if (v == 4) hipLaunchKernelGGL(k_fd_adjoint<4>, grid, dim3(256), 0, s, in, n, (uint32_t)nthr, out);
    else hipLaunchKernelGGL(k_fd_adjoint<1>, grid, dim3(256), 0, s, in, n, (uint32_t)nthr, out);
    CUBE_HIP(hipGetLastError());
  }
  static bool quads(int n, const void* a, const void* b) {
    return n % 4 == 0 && (((uintptr_t)a | (uintptr_t)b) & 15) == 0;
  }
  // the gather of the order's particles, from quads of phi where it may
  template <bool VJP>
  void gather(bool quad, const float* phi, const float* F, const float* rhob, float* out, hipStream_t s) {
    auto* const k = cfg.n <= 1024 ? (quad ? k_pm_gather<VJP, 4, false> : k_pm_gather<VJP, 1, false>)
                                  : (quad ? k_pm_gather<VJP, 4, true> : k_pm_gather<VJP, 1, true>);
    const Tiles tiles(cfg.n, cfg.batch);
    hipLaunchKernelGGL(k, dim3(tiles.blocks()), dim3(512), 0, s, rec.p, part.p, grec.p, cfg.n, tiles, bstart.p, phi, F,
                       rhob, out);
  }
  // rho -> phi (B*n^3) at positions x; srt: through the sorted order (with g's)
  void potential(const float* x, const float* g, int64_t np, float* phi, bool srt, hipStream_t s) {
    const int n = cfg.n, B = cfg.batch;
    const int64_t ntot = np * B;
    const Tiles tiles(n, B);
    if (srt) {
      sort(x, g, np, s);
      hipLaunchKernelGGL((k_pm_deposit<1, false>), dim3(tiles.blocks()), dim3(256), 0, s, rec.p, nullptr, n, tiles,
                         bstart.p, nullptr, phi);
    } else {
      over_few(ntot, [&](dim3 grid, uint32_t p0) {
        hipLaunchKernelGGL(k_tsc_deposit<1>, grid, dim3(64), 0, s, x, nullptr, p0, (uint32_t)np, (uint32_t)ntot, n, lat,
                           nullptr, acc.p);
      });
      fix_to_float(acc.p, B * n3, 1.0 / kFix, phi, s);
    }
    fft_convolve<float>(fc, phi, work.p, G.p, B, (float)n3, 0.0f, s);
  }
  // acc at positions x; F and phi (null: scratch) are outputs
  void force(const float* x, int64_t np, float* F, float* phi, float* out, hipStream_t s) {
    const int n = cfg.n;
    const int64_t ntot = np * cfg.batch;
    const bool srt = sorted(ntot, false, s);
    float* const to = phi;
    if (!phi || ((uintptr_t)phi & 15) != 0) phi = mesh.p;  // the transform moves pairs of floats
    potential(x, nullptr, np, phi, srt, s);
    if (!F && !srt) F = Fs.p;
    if (F) fd(false, phi, F, s);
    if (!srt)
      over_few(ntot, [&](dim3 grid, uint32_t p0) {
        hipLaunchKernelGGL(k_tsc_interp, grid, dim3(64), 0, s, x, p0, (uint32_t)np, (uint32_t)ntot, n, lat, F, out);
      });
    else
      gather<false>(quads(n, phi, nullptr), phi, nullptr, nullptr, out, s);
    if (to && to != phi)
      CUBE_HIP(hipMemcpyAsync(to, phi, sizeof(float) * (size_t)(cfg.batch * n3), hipMemcpyDeviceToDevice, s));
    CUBE_HIP(hipGetLastError());
  }
  // its adjoint, with the F or the phi of the same x, or neither
  void vjp(const float* x, int64_t np, const float* F, const float* phi, const float* g, float* gx, hipStream_t s) {
    const int n = cfg.n, B = cfg.batch;
    const int64_t ntot = np * B;
    const Tiles tiles(n, B);
    const bool srt = sorted(ntot, true, s);
    if (!F && !phi) {  // the potential of x again (checkpoint-and-recompute callers); sorts x when it does
      float* again = srt ? Fs.p : mesh.p;
      potential(x, g, np, again, srt, s);
      phi = again;
    } else if (srt) {
      sort(x, g, np, s);
    }
    if (srt) {
      hipLaunchKernelGGL((k_pm_deposit<3, false>), dim3(tiles.blocks()), dim3(256), 0, s, rec.p, grec.p, n, tiles, bstart.p, gmax.p,
                         Fbar.p);
    } else {
      if (!F) {
        fd(false, phi, Fs.p, s);
        F = Fs.p;
      }
      hipLaunchKernelGGL(k_absmax, dim3((unsigned)std::min<int64_t>(ceil_div(3 * ntot, 4096), kSlots)), dim3(1024), 0,
                         s, g, 3 * ntot, gmax.p);
      over_few(ntot, [&](dim3 grid, uint32_t p0) {
        hipLaunchKernelGGL(k_tsc_deposit<3>, grid, dim3(64), 0, s, x, g, p0, (uint32_t)np, (uint32_t)ntot, n, lat,
                           gmax.p, acc.p);
      });
      over_cells(3 * B * n3, [&](dim3 grid, int64_t at, int64_t m) {
        hipLaunchKernelGGL(k_sfix_to_float, grid, dim3(256), 0, s, acc.p + at, m, gmax.p, Fbar.p + at);
      });
    }
    fd(true, Fbar.p, mesh.p, s);
    fft_convolve<float>(fc, mesh.p, work.p, G.p, B, (float)n3, 0.0f, s);
    if (!srt)
      over_few(ntot, [&](dim3 grid, uint32_t p0) {
        hipLaunchKernelGGL(k_tsc_vjp, grid, dim3(64), 0, s, x, p0, (uint32_t)np, (uint32_t)ntot, n, lat, F, g, mesh.p, gx);
      });
    else
      gather<true>(quads(n, phi, mesh.p), phi, F, mesh.p, gx, s);
    CUBE_HIP(hipGetLastError());
  }
};

namespace {
template <class Fn>
int pm_guarded(cube_pm_ctx* ctx, Fn&& f) {
  if (!ctx) return CUBE_ERR_ARG;
  try {
    CUBE_HIP(hipSetDevice(ctx->device));
    f();
    ctx->err.clear();
    return CUBE_OK;
  } catch (const Error& e) {
    ctx->err = e.what();
    return e.code;
  } catch (const std::exception& e) {
    ctx->err = e.what();
    return CUBE_ERR_HIP;
  }
}
}  // namespace

extern "C" {

int cube_pm_create(const cube_pm_config* cfg, cube_pm_ctx** out) {
  if (!cfg || !out) return CUBE_ERR_ARG;
  *out = nullptr;
  if (cfg->n < 8 || cfg->batch < 1 || !(cfg->apm_soft > 0) || cfg->lattice < 0 || cfg->lattice > cfg->n)
    return CUBE_ERR_ARG;
  auto* c = new cube_pm_ctx();
  c->cfg = *cfg;
  c->lat.L = cfg->lattice;
  c->lat.step = cfg->lattice > 0 ? (double)cfg->n / (double)cfg->lattice : 0.0;
  const int rc = pm_guarded(c, [&] {
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) throw Error(CUBE_ERR_NO_DEVICE, "no HIP device");
    CUBE_HIP(hipGetDevice(&c->device));
    (void)scratch_address(c->device);  // the allocation-free entry point's scratch, once per device
    const int n = cfg->n, B = cfg->batch;
    c->n3 = (int64_t)n * n * n;
    c->fc.init(n);
    const int64_t nk = (int64_t)n * n * (n / 2 + 1);
    c->G.ensure((size_t)nk);
    green_device(n, cfg->apm_soft, 0.0f, 1.0f, 1.0, c->G.p, nullptr);
    c->mesh.ensure((size_t)(B * c->n3));
    c->Fs.ensure((size_t)(3 * B * c->n3));
    c->Fbar.ensure((size_t)(3 * B * c->n3));
    c->work.ensure((size_t)(B * nk));
    c->acc.ensure((size_t)(3 * B * c->n3));
    c->gmax.ensure(kSlots * kSlotStride);
    zero_cells(c->acc.p, 3 * B * c->n3, nullptr);
    CUBE_HIP(hipGetLastError());
    CUBE_HIP(hipDeviceSynchronize());
  });
  if (rc != CUBE_OK) {
    delete c;
    return rc;
  }
  *out = c;
  return CUBE_OK;
}

int cube_pm_destroy(cube_pm_ctx* ctx) {
  if (!ctx) return CUBE_OK;
  (void)hipSetDevice(ctx->device);
  (void)hipDeviceSynchronize();
  ctx->fc.release();
  delete ctx;
  return CUBE_OK;
}

const char* cube_pm_last_error(const cube_pm_ctx* ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int cube_pm_green(cube_pm_ctx* ctx, float* G_host) {
  return pm_guarded(ctx, [&] {
    if (!G_host) throw Error(CUBE_ERR_ARG, "null output");
    const int n = ctx->cfg.n;
    CUBE_HIP(hipMemcpy(G_host, ctx->G.p, sizeof(float) * (size_t)n * n * (n / 2 + 1), hipMemcpyDeviceToHost));
  });
}

int cube_pm_force(cube_pm_ctx* ctx, const float* x, int64_t np, float* F, float* acc, void* stream) {
  return pm_guarded(ctx, [&] {
    ctx->check_np(np);
    if (!x || !acc) throw Error(CUBE_ERR_ARG, "null pointer");
    ctx->force(x, np, F, nullptr, acc, (hipStream_t)stream);
  });
}

int cube_pm_force_phi(cube_pm_ctx* ctx, const float* x, int64_t np, float* phi, float* acc, void* stream) {
  return pm_guarded(ctx, [&] {
    ctx->check_np(np);
    if (!x || !acc) throw Error(CUBE_ERR_ARG, "null pointer");
    ctx->force(x, np, nullptr, phi, acc, (hipStream_t)stream);
  });
}

int cube_pm_force_vjp(cube_pm_ctx* ctx, const float* x, int64_t np, const float* F, const float* g_acc, float* g_x,
                      void* stream) {
  return pm_guarded(ctx, [&] {
    ctx->check_np(np);
    if (!x || !g_acc || !g_x) throw Error(CUBE_ERR_ARG, "null pointer");
    ctx->vjp(x, np, F, nullptr, g_acc, g_x, (hipStream_t)stream);
  });
}

int cube_pm_force_vjp_phi(cube_pm_ctx* ctx, const float* x, int64_t np, const float* phi, const float* g_acc,
                          float* g_x, void* stream) {
  return pm_guarded(ctx, [&] {
    ctx->check_np(np);
    if (!x || !g_acc || !g_x) throw Error(CUBE_ERR_ARG, "null pointer");
    ctx->vjp(x, np, nullptr, phi, g_acc, g_x, (hipStream_t)stream);
  });
}

int cube_pm_cic(cube_pm_ctx* ctx, const float* x, int64_t np, int32_t nw, float scale, float* rho, void* stream) {
  return pm_guarded(ctx, [&] {
    ctx->check_np(np);
    if (!x || !rho || nw < 2) throw Error(CUBE_ERR_ARG, "bad argument");
    const hipStream_t s = (hipStream_t)stream;
    const int B = ctx->cfg.batch;
    const int64_t ntot = np * B, nw3 = (int64_t)nw * nw * nw;
    const bool srt = ctx->cic_sorted(ntot, nw, s);
    // The accumulator of the form by atomics: that of the forces, or a larger one, which
    // is made in either form: a call recorded later may have more particles than
    // the order's buffers hold, and cannot allocate.
    const size_t cells = (size_t)(B * nw3);
    const bool own = cells > ctx->acc.n, captured = own && ctx->capturing(s);
    if (own && cells > ctx->accw.n && !(captured && srt))
      zero_cells(ctx->accw.ensure(cells), B * nw3, s);
    if (srt) {
      const Tiles tiles(nw, B);
      ctx->bin<true>(x, np, nw, scale, s);
      ctx->place<Sort::kCIC>(x, nullptr, np, nw, scale, s);
      hipLaunchKernelGGL((k_pm_deposit<1, true>), dim3(tiles.blocks()), dim3(256), 0, s, ctx->rec.p, nullptr, nw, tiles,
                         ctx->bstart.p, nullptr, rho);
      CUBE_HIP(hipGetLastError());
      return;
    }
    if (captured) ctx->accw.hold();
    unsigned long long* const acc = own ? ctx->accw.p : ctx->acc.p;
    hipLaunchKernelGGL(k_cic_deposit, dim3(nblk(ntot)), dim3(256), 0, s, x, (uint32_t)np, (uint32_t)ntot, nw, scale, ctx->lat,
                       acc);
    fix_to_float(acc, B * nw3, 1.0 / 2147483648.0, rho, s);
    CUBE_HIP(hipGetLastError());
  });
}

int cube_pm_cic_noalloc(cube_pm_ctx* ctx, const float* x, int64_t np, int32_t nw, float scale, float* rho,
                        void* stream) {
  return pm_guarded(ctx, [&] {
    ctx->check_np(np);
    if (!x || !rho || nw < 2) throw Error(CUBE_ERR_ARG, "bad argument");
    const int B = ctx->cfg.batch;
    const int64_t nw3 = (int64_t)nw * nw * nw;
    if (nw > 4096 || B * nw3 > kScratchCells)
      throw Error(CUBE_ERR_ARG, "cube_pm_cic_noalloc: batch*nw^3 = " + std::to_string(B * nw3) +
                                    " cells exceeds the fixed scratch of " + std::to_string(kScratchCells) +
                                    " cells (64 MiB); use cube_pm_cic");
    unsigned long long* acc = scratch_address(ctx->device);
    const hipStream_t s = (hipStream_t)stream;
    const int64_t ntot = np * B;
    // the array keeps whatever the last call on this GPU left: clear it here
    zero_cells(acc, B * nw3, s);
    hipLaunchKernelGGL(k_cic_deposit, dim3(nblk(ntot)), dim3(256), 0, s, x, (uint32_t)np, (uint32_t)ntot, nw, scale, ctx->lat, acc);
    fix_to_float(acc, B * nw3, 1.0 / 2147483648.0, rho, s);
    CUBE_HIP(hipGetLastError());
  });
}

int cube_pm_cic_vjp(cube_pm_ctx* ctx, const float* x, int64_t np, int32_t nw, float scale, const float* g_rho,
                    float* g_x, void* stream) {
  return pm_guarded(ctx, [&] {
    ctx->check_np(np);
    if (!x || !g_rho || !g_x || nw < 2) throw Error(CUBE_ERR_ARG, "bad argument");
    const hipStream_t s = (hipStream_t)stream;
    const int64_t ntot = np * ctx->cfg.batch;
    hipLaunchKernelGGL(k_cic_vjp, dim3(nblk(ntot)), dim3(256), 0, s, x, (uint32_t)np, (uint32_t)ntot, nw, scale, ctx->lat, g_rho, g_x);
    CUBE_HIP(hipGetLastError());
  });
}

}  // extern "C"
