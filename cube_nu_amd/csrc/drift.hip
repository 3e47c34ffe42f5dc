// drift.hip -- drift.f90 on the GPU, bit-exact.
//
// The reference fixes the order of particles inside a destination cell by
// its plane-colour OpenMP passes (drift.f90:46-49, 96-136): source planes are
// visited in passes ilayer = (k-(1-ncb)) mod nlayer, each plane by one thread
// in (j, i, l) order.  With the colour count nlayer = 2*ceil(dt_mid*vz_max/4)
// + 2, a destination cell receives from at most one plane per pass, so the
// order is the key (pass(k_src), k_src, j_src, i_src, l).
//
// GPU form (no atomics on any order):
//  1. shift pass: destination of every particle, range check, maximum cell
//     shift per axis, per-destination integer counts (atomic adds of
//     integers are order-independent);
//  2. rank pass (one wavefront per run of up to eight source cells along x, one
//     particle per lane): for each destination direction d, the rank of each
//     particle among its cell's earlier particles with the same d (the lanes with
//     the same cell and d are found by one ballot per bit of that key), and
//     the per-(cell, d) count;
//  3. offset pass (one thread per destination cell): walks its neighbouring
//     source cells in key order and turns the (cell, d) counts into offsets;
//  4. scatter pass: out = base(dest) + offset(cell, d) + rank, with the
//     re-encode xp' = xp + nint(dt_mid*v/(x_resolution*ratio_cs)) wrapped to
//     izipx bytes (drift.f90:117).
// The source cells are those of the tile and of `ring` buffer cells around it.
// Where buffers are images of physical particles, velocities included, and no
// particle moves by more than M cells, those beyond M have nothing to send: 192^3
// in 64 tiles of 12^3 cells visits 14^3 of 24^3.
#include "drift.h"
#include "grid.h"

namespace cube {
namespace {

template <int IZ>
using XT = typename XP<IZ>::T;

}  // namespace

namespace {

template <int IZ>
__device__ inline void dest_cell(const DriftParams& P, const XT<IZ>* xp, const float* vp, int64_t ip,
                                 const int ijk[3], int g[3]) {
  for (int d = 0; d < 3; ++d) {
    const double wv = P.dt_mid * (double)vp[3 * ip + d];        // FP64 coefficient
    const double dx = wv * P.inv_rcs;                            // drift.f90:57 (exact: rcs = 2^k)
    const double xq = ((double)ijk[d] - 1.0) + XP<IZ>::off(xp, ip, d);  // drift.f90:59
    g[d] = (int)ceil(xq + dx);                                   // drift.f90:63
  }
}

__device__ inline void cell_of(const DriftParams& P, int64_t cglob, int* T, int ijk[3]) {
  // extended cell counts stay below 2^31 (64 tiles of nte^3 cells)
  const uint32_t nct = (uint32_t)(P.nte * P.nte * P.nte), cg = (uint32_t)cglob;
  *T = (int)(cg / nct);
  const int e = (int)(cg - (uint32_t)*T * nct);
  ijk[0] = e % P.nte + 1 - P.ncb;
  ijk[1] = (e / P.nte) % P.nte + 1 - P.ncb;
  ijk[2] = e / (P.nte * P.nte) + 1 - P.ncb;
}

__device__ inline bool physical(const DriftParams& P, const int g[3]) {
  return g[0] >= 1 && g[0] <= P.nt && g[1] >= 1 && g[1] <= P.nt && g[2] >= 1 && g[2] <= P.nt;
}

__device__ inline int dcode(const DriftParams& P, const int g[3], const int s[3]) {
  return ((g[2] - s[2] + P.M[2]) * P.D[1] + (g[1] - s[1] + P.M[1])) * P.D[0] + (g[0] - s[0] + P.M[0]);
}

__device__ inline int64_t pcell(const DriftParams& P, int T, const int g[3]) {
  return (((int64_t)T * P.nt + (g[2] - 1)) * P.nt + (g[1] - 1)) * P.nt + (g[0] - 1);
}

template <int IZ>
__global__ void k_drift_shift(DriftParams P, const XT<IZ>* __restrict__ xp, const float* __restrict__ vp,
                              const int32_t* __restrict__ rhoc, const int64_t* __restrict__ off, int64_t ncells,
                              int32_t* __restrict__ flags, int32_t* __restrict__ newcount) {
  const int64_t c = ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (c >= ncells) return;
  int T, ijk[3];
  cell_of(P, c, &T, ijk);
  const int cnt = rhoc[c];
  const int64_t base = off[c];
  const int lo = 1 - 2 * P.ncb, hi = P.nt + 2 * P.ncb;
  int err = 0, ms[3] = {0, 0, 0};
  for (int l0 = 0; l0 < cnt; l0 += 64) {
    const int l = l0 + lane;
    int64_t key = -1;
    if (l < cnt) {
      int g[3];
      dest_cell<IZ>(P, xp, vp, base + l, ijk, g);
      for (int d = 0; d < 3; ++d)
        if (g[d] < lo || g[d] > hi) err = 1;
      if (physical(P, g)) {
        for (int d = 0; d < 3; ++d) ms[d] = max(ms[d], abs(g[d] - ijk[d]));
        key = pcell(P, T, g);
      }
    }
    // one integer atomic per distinct destination in the wavefront
    unsigned long long active = __ballot(key >= 0);
    while (active) {
      const int leader = __ffsll((long long)active) - 1;
      const int64_t lk = __shfl(key, leader, 64);
      const unsigned long long peers = __ballot(key == lk);
      if (lane == leader) atomicAdd(&newcount[lk], (int)__popcll(peers));
      active &= ~peers;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    err |= __shfl_down(err, o, 64);
    for (int d = 0; d < 3; ++d) ms[d] = max(ms[d], __shfl_down(ms[d], o, 64));
  }
  if (lane == 0 && cnt > 0) {
    if (err) atomicOr(&flags[0], DRIFT_OUT_OF_RANGE);
    for (int d = 0; d < 3; ++d) atomic_max_int(&flags[1 + d], ms[d]);
  }
}

// The runs of up to eight source cells: a row of na = nt + 2 ring cells is cut into
// `runs` runs of `len`.
struct Runs {
  uint32_t na, sh, runs, len, n;  // sh: cells of the extended row before the first
};
inline Runs make_runs(const DriftParams& P, int64_t tiles) {
  Runs R{};
  R.na = (uint32_t)(P.nt + 2 * P.ring);
  R.sh = (uint32_t)(P.ncb - P.ring);
  R.runs = (R.na + 7) / 8;
  R.len = (R.na + R.runs - 1) / R.runs;
  R.n = (uint32_t)(tiles * R.na * R.na * R.runs);
  return R;
}
// A wavefront's run: its tile (from the batch's first), its first cell's
// coordinates and extended index, its index among the source cells, its cells.
struct Run {
  int T, ijk[3], cells;
  int64_t c, a;
};
__device__ inline Run run_of(const DriftParams& P, const Runs& R, uint32_t w) {
  uint32_t q = w / R.runs, x = (w - q * R.runs) * R.len;
  uint32_t r = q / R.na;
  const uint32_t y = q - r * R.na, T = r / R.na, z = r - T * R.na;
  Run o;
  o.T = (int)T;
  o.ijk[0] = (int)(x + R.sh) + 1 - P.ncb;
  o.ijk[1] = (int)(y + R.sh) + 1 - P.ncb;
  o.ijk[2] = (int)(z + R.sh) + 1 - P.ncb;
  o.cells = x < R.na ? (int)min(R.len, R.na - x) : 0;
  o.c = (((int64_t)T * P.nte + z + R.sh) * P.nte + y + R.sh) * P.nte + x + R.sh;
  o.a = (((int64_t)T * R.na + z) * R.na + y) * R.na + x;
  return o;
}
// First particle of cell k of the run (k <= cells), from the first's; lanes hold
// them (lane k the k-th).
__device__ inline int cell_start(int starts, int k) { return __builtin_amdgcn_readlane(starts, k); }
__device__ inline int cell_at(int starts, int cells, int pos) {
  int ci = 0;
#pragma unroll
  for (int k = 1; k < 8; ++k) ci += (k < cells && pos >= cell_start(starts, k)) ? 1 : 0;
  return ci;
}

// Rank pass.  COUNT = true also does the shift pass's range check and largest
// shift in the same read of the particles (the destination counts come from the
// offset pass), with P.M a bound given by the caller: a particle whose shift
// exceeds it takes no table entry and sets DRIFT_SHIFT_BOUND, after which the
// caller redoes the drift with the measured bound.  P.images: the ring is cut to
// the bound, so every particle that moves as far as it, wherever it goes, sets that
// flag (by a margin beyond the rounding of the positions, which differ between a
// particle and its images; along an axis at rest, M = 0, any that moves does).  The run's counts are kept in LDS up to kLdsDirs
// directions and written once, else in the (cleared) table.  A wave per cell with
// a loop over its directions, their counts in memory and every cell of the
// extended tiles took 0.353 ms at 192^3 (64 tiles of 12^3 cells, 57 million
// particles with the buffers), this with M = 1 0.110 (11 million).
constexpr int kLdsDirs = 343;  // 44 KB a workgroup
template <int IZ, bool COUNT, bool LDS>
__global__ void __launch_bounds__(256) k_drift_rank(DriftParams P, Runs R, const XT<IZ>* __restrict__ xp,
                                                    const float* __restrict__ vp, const int64_t* __restrict__ off,
                                                    int t0, int32_t* __restrict__ rank, int32_t* __restrict__ table,
                                                    int32_t* __restrict__ flags,
                                                    unsigned long long* __restrict__ ranked) {
  extern __shared__ int32_t counts[];
  const uint32_t w = blockIdx.x * 4u + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (w >= R.n) return;
  const Run o = run_of(P, R, w);
  if (o.cells == 0) return;
  const int64_t oc = off[(int64_t)t0 * P.nte * P.nte * P.nte + o.c + min(lane, o.cells)];
  const int64_t base = __shfl(oc, 0, 64);
  const int starts = (int)(oc - base), tot = cell_start(starts, o.cells);
  const int Dt = P.D[0] * P.D[1] * P.D[2];
  const int bits = 32 - __clz(8 * Dt - 1);
  int32_t* tbl = table + o.a * Dt;
  int32_t* mine = counts + (threadIdx.x >> 6) * 8 * Dt;  // of this wavefront alone
  if (LDS)
    for (int k = lane; k < o.cells * Dt; k += 64) mine[k] = 0;
  const int lo = 1 - 2 * P.ncb, hi = P.nt + 2 * P.ncb;
  int err = 0, ms[3] = {0, 0, 0}, mine_ranked = 0;
  for (int p0 = 0; p0 < tot; p0 += 64) {
    const int pos = p0 + lane;
    const int ci = cell_at(starts, o.cells, pos);
    int key = -1;
    if (pos < tot) {
      const int64_t ip = base + pos;
      const int s[3] = {o.ijk[0] + ci, o.ijk[1], o.ijk[2]};
      int g[3];
      dest_cell<IZ>(P, xp, vp, ip, s, g);
      if (COUNT) {
        for (int d = 0; d < 3; ++d)
          if (g[d] < lo || g[d] > hi) err |= DRIFT_OUT_OF_RANGE;
        if (P.images)
          for (int d = 0; d < 3; ++d)
            if (!(fabs(P.dt_mid * (double)vp[3 * ip + d] * P.inv_rcs) <= fmax(P.M[d] - 1e-6, 0.0))) err |= DRIFT_SHIFT_BOUND;
      }
      if (physical(P, g)) {
        bool fits = true;
        if (COUNT) {
          for (int d = 0; d < 3; ++d) {
            const int sd = abs(g[d] - s[d]);
            ms[d] = max(ms[d], sd);
            fits = fits && sd <= P.M[d];
          }
        }
        if (fits) key = ci * Dt + dcode(P, g, s);
        else err |= DRIFT_SHIFT_BOUND;
      }
    }
    unsigned long long peers = __builtin_amdgcn_ballot_w64(key >= 0);
    if (COUNT) mine_ranked += (int)__popcll(peers);
    for (int b = 0; b < bits; ++b) {
      const bool one = (key >> b) & 1;
      const unsigned long long m = __builtin_amdgcn_ballot_w64(one);
      peers &= one ? m : ~m;
    }
    if (key < 0) peers = 1ull << lane;
    const int leader = __ffsll((long long)peers) - 1;
    int before = 0;
    if (key >= 0 && lane == leader) before = atomicAdd(LDS ? &mine[key] : &tbl[key], (int)__popcll(peers));
    before = __shfl(before, leader, 64);
    if (pos < tot) rank[base + pos] = key < 0 ? -1 : before + __popcll(peers & ((1ull << lane) - 1ull));
  }
  if (LDS)
    for (int k = lane; k < o.cells * Dt; k += 64) tbl[k] = mine[k];
  if (COUNT) {
    for (int q = 32; q > 0; q >>= 1) {
      err |= __shfl_down(err, q, 64);
      for (int d = 0; d < 3; ++d) ms[d] = max(ms[d], __shfl_down(ms[d], q, 64));
    }
    if (lane == 0 && tot > 0) {
      if (err) atomicOr(&flags[0], err);
      for (int d = 0; d < 3; ++d) atomic_max_int(&flags[1 + d], ms[d]);
      if (mine_ranked) atomicAdd(&ranked[blockIdx.x % kSumSlots * kRankedStride], (unsigned long long)mine_ranked);
    }
  }
}

// Offsets of the (cell, direction) counts; COUNT: and the destinations' counts, else
// checked against the shift pass's.
template <bool COUNT>
__global__ void k_drift_offsets(DriftParams P, int t0, int t1, int32_t* __restrict__ table,
                                int32_t* __restrict__ newcount, int32_t* __restrict__ flags) {
  const uint32_t nt = (uint32_t)P.nt, nt2 = nt * nt;
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (uint32_t)(t1 - t0) * nt2 * nt) return;
  const uint32_t Tl = t / (nt2 * nt), q = t - Tl * nt2 * nt, qz = q / nt2, qy = (q - qz * nt2) / nt;
  const int T = t0 + (int)Tl;
  const int g[3] = {(int)(q - qz * nt2 - qy * nt) + 1, (int)qy + 1, (int)qz + 1};
  const int lo = 1 - P.ncb, hi = P.nt + P.ncb;
  const int Dt = P.D[0] * P.D[1] * P.D[2];
  // source planes in pass order (pass(k) = (k - (1-ncb)) mod nlayer), then k
  int ks[2 * kMaxShift + 1];
  int nk = 0;
  for (int k = max(lo, g[2] - P.M[2]); k <= min(hi, g[2] + P.M[2]); ++k) ks[nk++] = k;
  for (int a = 1; a < nk; ++a) {
    int v = ks[a], pv = (v - lo) % P.nlayer, b = a - 1;
    while (b >= 0) {
      int pb = (ks[b] - lo) % P.nlayer;
      if (pb > pv || (pb == pv && ks[b] > v)) {
        ks[b + 1] = ks[b];
        --b;
      } else
        break;
    }
    ks[b + 1] = v;
  }
  const int na = P.nt + 2 * P.ring;
  int running = 0;
  constexpr int B = 9;  // entries loaded at once
  const int i0 = max(lo, g[0] - P.M[0]), ni = min(hi, g[0] + P.M[0]) - i0 + 1;
  const int j0 = max(lo, g[1] - P.M[1]), nj = min(hi, g[1] + P.M[1]) - j0 + 1;
  for (int a = 0; a < nk; ++a) {
    const int k = ks[a], nij = ni * nj;
    for (int e0 = 0; e0 < nij; e0 += B) {
      int64_t idx[B];
      int c[B];
      int i = i0 + e0 % ni, j = j0 + e0 / ni;
#pragma unroll
      for (int e = 0; e < B; ++e) {
        const int s[3] = {i, j, k};
        idx[e] = ((((int64_t)Tl * na + k - 1 + P.ring) * na + j - 1 + P.ring) * na + i - 1 + P.ring) * Dt + dcode(P, g, s);
        c[e] = e0 + e < nij ? table[idx[e]] : 0;
        if (++i == i0 + ni) {
          i = i0;
          ++j;
        }
      }
#pragma unroll
      for (int e = 0; e < B; ++e) {
        if (e0 + e < nij) table[idx[e]] = running;
        running += c[e];
      }
    }
  }
  if (COUNT) newcount[pcell(P, T, g)] = running;
  else if (running != newcount[pcell(P, T, g)]) atomicOr(&flags[0], 4);
}

template <int IZ>
__global__ void __launch_bounds__(256) k_drift_scatter(DriftParams P, Runs R, const XT<IZ>* __restrict__ xp,
                                                       const float* __restrict__ vp, const int64_t* __restrict__ pid,
                                                       const int64_t* __restrict__ off, int t0,
                                                       const int32_t* __restrict__ rank,
                                                       const int32_t* __restrict__ table,
                                                       const int64_t* __restrict__ base_out, XT<IZ>* __restrict__ xo,
                                                       float* __restrict__ vo, int64_t* __restrict__ po,
                                                       int32_t* __restrict__ flags) {
  const uint32_t w = blockIdx.x * 4u + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (w >= R.n) return;
  const Run o = run_of(P, R, w);
  if (o.cells == 0) return;
  const int T = t0 + o.T;
  const int64_t oc = off[(int64_t)t0 * P.nte * P.nte * P.nte + o.c + min(lane, o.cells)];
  const int64_t base = __shfl(oc, 0, 64);
  const int starts = (int)(oc - base), tot = cell_start(starts, o.cells);
  const int Dt = P.D[0] * P.D[1] * P.D[2];
  const int32_t* tbl = table + o.a * Dt;
  // 1 / (x_resolution rcs): both powers of two, so wv * shs == wv / (xr rcs)
  const double shs = P.inv_rcs * (double)(1 << XP<IZ>::B);
  for (int p0 = 0; p0 < tot; p0 += 64) {
    const int l = p0 + lane;
    const int ci = cell_at(starts, o.cells, l);
    if (l >= tot) continue;
    const int64_t ip = base + l;
    const int r = rank[ip];
    if (r < 0) continue;
    const int s[3] = {o.ijk[0] + ci, o.ijk[1], o.ijk[2]};
    int g[3];
    dest_cell<IZ>(P, xp, vp, ip, s, g);
    const int64_t pos = base_out[pcell(P, T, g)] + tbl[ci * Dt + dcode(P, g, s)] + r;
    for (int d = 0; d < 3; ++d) {
      const double wv = P.dt_mid * (double)vp[3 * ip + d];
      const double sh = wv * shs;  // drift.f90:117
      const long long dn = (long long)round(sh);  // nint: half away from zero
      const long long nv = (long long)xp[3 * ip + d] + dn;
      if (IZ == 2) xo[3 * pos + d] = (int16_t)(uint16_t)(nv & 0xffff);
      else xo[3 * pos + d] = (int8_t)(uint8_t)(nv & 0xff);
      vo[3 * pos + d] = vp[3 * ip + d];
    }
    const int64_t pv = pid ? pid[ip] : 1;
    if (po) po[pos] = pv;
    if (pv <= 0) atomicOr(&flags[0], DRIFT_PID_ZERO);
  }
}

__global__ void k_drift_rhoc(DriftParams P, int64_t ncells, const int32_t* __restrict__ newcount,
                             int32_t* __restrict__ rhoc) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncells) return;
  int T, ijk[3];
  cell_of(P, c, &T, ijk);
  rhoc[c] = physical(P, ijk) ? newcount[pcell(P, T, ijk)] : 0;
}

__global__ void k_tile_check(const int64_t* __restrict__ off, int64_t nct, int ntiles, int64_t cap,
                             int32_t* __restrict__ flags) {
  for (int T = threadIdx.x; T < ntiles; T += blockDim.x) {
    const int64_t n = off[(int64_t)(T + 1) * nct] - off[(int64_t)T * nct];
    atomic_max_int(&flags[4], (int32_t)(n < (int64_t)INT32_MAX ? n : (int64_t)INT32_MAX));
    if (n > cap) atomicOr(&flags[0], DRIFT_TILE_OVERFLOW);
  }
}

__global__ void k_buffer_rhoc(Geo g, const int32_t* __restrict__ rp, int32_t* __restrict__ re,
                              int32_t* __restrict__ physcount) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= g.ncells_ext) return;
  const int64_t T = c / g.ncell_tile, e = c % g.ncell_tile;
  const int64_t it[3] = {T % g.nnt, (T / g.nnt) % g.nnt, T / (g.nnt * g.nnt)};
  const int64_t ijk[3] = {e % g.nte + 1 - g.ncb, (e / g.nte) % g.nte + 1 - g.ncb, e / (g.nte * g.nte) + 1 - g.ncb};
  int64_t st[3], sc[3];
  for (int d = 0; d < 3; ++d) {
    int64_t gc = it[d] * g.nt + ijk[d] - 1;
    gc = ((gc % g.nc) + g.nc) % g.nc;
    st[d] = gc / g.nt;
    sc[d] = gc % g.nt + 1;
  }
  const int64_t Ts = (st[2] * g.nnt + st[1]) * g.nnt + st[0];
  const int32_t v = rp[rc_index(sc[0], sc[1], sc[2], Ts, g.nte, g.ncb)];
  re[c] = v;
  const bool phys = ijk[0] >= 1 && ijk[0] <= g.nt && ijk[1] >= 1 && ijk[1] <= g.nt && ijk[2] >= 1 && ijk[2] <= g.nt;
  if (phys) physcount[((T * g.nt + ijk[2] - 1) * g.nt + ijk[1] - 1) * g.nt + ijk[0] - 1] = v;
}


}  // namespace

void drift_tile_check(const int64_t* off, int64_t ncell_tile, int ntiles, int64_t np_tile_max, int32_t* flags,
                      hipStream_t s) {
  hipLaunchKernelGGL(k_tile_check, dim3(1), dim3(256), 0, s, off, ncell_tile, ntiles, np_tile_max, flags);
  CUBE_HIP(hipGetLastError());
}

void drift_shift(const DriftParams& P, const void* xp, const float* vp, const int32_t* rhoc, const int64_t* off,
                 int64_t ncells, DriftScratch& S, hipStream_t s) {
  const Blocks b = blocks_xy(ceil_div(ncells, 4));  // a wavefront per cell
  if (P.izipx == 2)
    hipLaunchKernelGGL(k_drift_shift<2>, dim3(b.x, b.y), dim3(256), 0, s, P, (const int16_t*)xp, vp, rhoc, off, ncells,
                       S.flags, S.newcount);
  else
    hipLaunchKernelGGL(k_drift_shift<1>, dim3(b.x, b.y), dim3(256), 0, s, P, (const int8_t*)xp, vp, rhoc, off, ncells,
                       S.flags, S.newcount);
  CUBE_HIP(hipGetLastError());
}

namespace {
template <int IZ, bool COUNT>
void rank_launch(const DriftParams& P, const void* xp, const float* vp, const int64_t* off, int t0, int t1,
                 DriftScratch& S, hipStream_t s) {
  const Runs R = make_runs(P, t1 - t0);
  const dim3 grid((unsigned)ceil_div(R.n, 4));
  const int Dt = P.D[0] * P.D[1] * P.D[2];
  if (Dt <= kLdsDirs) {
    hipLaunchKernelGGL((k_drift_rank<IZ, COUNT, true>), grid, dim3(256), 4 * 8 * Dt * sizeof(int32_t), s, P, R,
                       (const XT<IZ>*)xp, vp, off, t0, S.rank, S.table, S.flags, S.ranked);
  } else {
    zero_async(S.table, sizeof(int32_t) * (size_t)(t1 - t0) * R.na * R.na * R.na * Dt, s);
    hipLaunchKernelGGL((k_drift_rank<IZ, COUNT, false>), grid, dim3(256), 0, s, P, R, (const XT<IZ>*)xp, vp, off, t0,
                       S.rank, S.table, S.flags, S.ranked);
  }
  CUBE_HIP(hipGetLastError());
}
}  // namespace

void drift_rank(const DriftParams& P, const void* xp, const float* vp, const int64_t* off, int t0, int t1,
                DriftScratch& S, hipStream_t s, bool count) {
  if (P.izipx == 2) {
    if (count) rank_launch<2, true>(P, xp, vp, off, t0, t1, S, s);
    else rank_launch<2, false>(P, xp, vp, off, t0, t1, S, s);
  } else {
    if (count) rank_launch<1, true>(P, xp, vp, off, t0, t1, S, s);
    else rank_launch<1, false>(P, xp, vp, off, t0, t1, S, s);
  }
}

void drift_offsets(const DriftParams& P, int t0, int t1, DriftScratch& S, hipStream_t s, bool count) {
  const int64_t n = (int64_t)(t1 - t0) * P.nt * P.nt * P.nt;
  const dim3 grid((unsigned)ceil_div(n, 256));
  if (count)
    hipLaunchKernelGGL(k_drift_offsets<true>, grid, dim3(256), 0, s, P, t0, t1, S.table, S.newcount, S.flags);
  else
    hipLaunchKernelGGL(k_drift_offsets<false>, grid, dim3(256), 0, s, P, t0, t1, S.table, S.newcount, S.flags);
  CUBE_HIP(hipGetLastError());
}

void drift_scatter(const DriftParams& P, const void* xp, const float* vp, const int64_t* pid, const int64_t* off,
                   int t0, int t1, DriftScratch& S, void* xp_out, float* vp_out, int64_t* pid_out, hipStream_t s) {
  const Runs R = make_runs(P, t1 - t0);
  const dim3 grid((unsigned)ceil_div(R.n, 4));
  if (P.izipx == 2)
    hipLaunchKernelGGL(k_drift_scatter<2>, grid, dim3(256), 0, s, P, R, (const int16_t*)xp, vp, pid, off, t0, S.rank,
                       S.table, S.base, (int16_t*)xp_out, vp_out, pid_out, S.flags);
  else
    hipLaunchKernelGGL(k_drift_scatter<1>, grid, dim3(256), 0, s, P, R, (const int8_t*)xp, vp, pid, off, t0, S.rank,
                       S.table, S.base, (int8_t*)xp_out, vp_out, pid_out, S.flags);
  CUBE_HIP(hipGetLastError());
}

void drift_write_rhoc(const DriftParams& P, const DriftScratch& S, int32_t* rhoc_out, hipStream_t s) {
  const int64_t nct = (int64_t)P.nte * P.nte * P.nte;
  const int64_t ncells = (int64_t)P.nnt * P.nnt * P.nnt * nct;
  hipLaunchKernelGGL(k_drift_rhoc, dim3((unsigned)ceil_div(ncells, 256)), dim3(256), 0, s, P, ncells, S.newcount,
                     rhoc_out);
  CUBE_HIP(hipGetLastError());
}

void buffer_rhoc(const Geo& g, const int32_t* rhoc_phys, int32_t* rhoc_ext, int32_t* physcount, hipStream_t s) {
  hipLaunchKernelGGL(k_buffer_rhoc, dim3((unsigned)ceil_div(g.ncells_ext, 256)), dim3(256), 0, s, g, rhoc_phys,
                     rhoc_ext, physcount);
  CUBE_HIP(hipGetLastError());
}

namespace {

// nn=1 buffer copy by rows: an x-row of an extended tile is three runs of
// consecutive cells, each a contiguous run of particles in the source
// layout (cells 1..nt of the tile, the last ncb cells of the periodic left
// neighbour, the first ncb of the right one) and in the extended layout.
// One wavefront per run copies it with coalesced, independent loads (xp as its
// 16- or 8-bit elements, vp as floats, pid as 64-bit words).  Bound by what it
// writes: 192^3 particles in 64 tiles of 12^3 cells become 57 million of 26 bytes,
// in 0.34 ms (4.3 TB/s; 0.35 as three runs in turn by a workgroup).
struct RowRun {
  int64_t e0, p0;  // extended and physical (1 row of nt) cells of its start
  int cells;
  bool self;  // the tile's own cells of a physical row
};
__device__ inline bool row_run(const Geo& g, bool ext_source, RowRun& o) {
  const int nte = (int)g.nte, nt = (int)g.nt, nc = (int)g.nc, nnt = (int)g.nnt, ncb = (int)g.ncb;
  const uint32_t w = blockIdx.x * 4u + (threadIdx.x >> 6), r = w / 3u, seg = w - 3u * r;
  const uint32_t rz = r / (uint32_t)nte;  // (T, ze, ye) with ye fastest
  const int ye = (int)(r - rz * nte), T = (int)(rz / (uint32_t)nte), ze = (int)(rz - (uint32_t)T * nte);
  if (T >= (int)g.ntiles) return false;
  const int it[3] = {T % nnt, (T / nnt) % nnt, T / (nnt * nnt)};
  // source tile and cell (from 0) of an extended cell (from 0) along one axis, periodic
  auto src = [&](int tile, int e, int& t, int& c) {
    int gc = tile * nt + e - ncb;
    gc = gc < 0 ? gc + nc : (gc >= nc ? gc - nc : gc);
    t = gc / nt;
    c = gc - t * nt;
  };
  const int xe0 = seg == 0 ? 0 : (seg == 1 ? ncb : ncb + nt);
  int tx, ty, tz, sx, sy, sz;
  src(it[0], xe0, tx, sx);
  src(it[1], ye, ty, sy);
  src(it[2], ze, tz, sz);
  const int Ts = (tz * nnt + ty) * nnt + tx;
  o.cells = seg == 1 ? nt : ncb;
  o.self = seg == 1 && ye >= ncb && ye < ncb + nt && ze >= ncb && ze < ncb + nt;
  o.e0 = (((int64_t)T * nte + ze) * nte + ye) * nte + xe0;
  o.p0 = ext_source ? (((int64_t)Ts * nte + sz + ncb) * nte + sy + ncb) * nte + sx + ncb
                    : (((int64_t)Ts * nt + sz) * nt + sy) * nt + sx;
  return true;
}
template <typename T>
__device__ inline void copy_run(T* dst, const T* src, int64_t n) {
  int64_t q = threadIdx.x & 63;
  for (; q + 192 < n; q += 256) {
    const T a = src[q], b = src[q + 64], c = src[q + 128], d = src[q + 192];
    dst[q] = a;
    dst[q + 64] = b;
    dst[q + 128] = c;
    dst[q + 192] = d;
  }
  const T a = q < n ? src[q] : T{}, b = q + 64 < n ? src[q + 64] : T{}, c = q + 128 < n ? src[q + 128] : T{};
  if (q < n) dst[q] = a;
  if (q + 64 < n) dst[q + 64] = b;
  if (q + 128 < n) dst[q + 128] = c;
}

template <int IZ>
__global__ void __launch_bounds__(256) k_buffer_rows(Geo g, const int64_t* __restrict__ eoff,
                                                     const int64_t* __restrict__ poff, const XT<IZ>* __restrict__ xp,
                                                     const float* __restrict__ vp, const int64_t* __restrict__ pid,
                                                     XT<IZ>* __restrict__ xo, float* __restrict__ vo,
                                                     int64_t* __restrict__ po) {
  RowRun r;
  if (!row_run(g, false, r)) return;
  const int64_t src = poff[r.p0], n = poff[r.p0 + r.cells] - src, dst = eoff[r.e0];
  copy_run(vo + 3 * dst, vp + 3 * src, 3 * n);
  copy_run(xo + 3 * dst, xp + 3 * src, 3 * n);
  if (pid) copy_run(po + dst, pid + src, n);
}

// buffer_v at nn=1 (buffer_particle.f90:11-27, buffer_xvp(.false., .true.)):
// in the extended layout, the velocities (and IDs) of every buffer cell are
// overwritten by those of the physical cell it is the periodic image of.  The
// same three runs per (tile, z, y) row as k_buffer_rows, read from the
// physical cells of the extended array itself: sources are physical cells and
// destinations buffer cells, so no run is both.  A run copies the smaller of
// its source and destination counts (equal in a layout made by the buffer
// step), so every access stays inside both runs.
template <bool PID>
__global__ void __launch_bounds__(256) k_buffer_v_rows(Geo g, const int64_t* __restrict__ eoff, float* vp,
                                                       int64_t* pid) {
  RowRun r;
  if (!row_run(g, true, r) || r.self) return;  // a row's physical cells are their own source
  const int64_t src = eoff[r.p0], nsrc = eoff[r.p0 + r.cells] - src;
  const int64_t dst = eoff[r.e0], ndst = eoff[r.e0 + r.cells] - dst;
  const int64_t n = nsrc < ndst ? nsrc : ndst;
  copy_run(vp + 3 * dst, vp + 3 * src, 3 * n);
  if (PID) copy_run(pid + dst, pid + src, n);
}

}  // namespace

void buffer_v(const Geo& g, const int64_t* ext_off, float* vp, int64_t* pid, hipStream_t s) {
  const int64_t rows = g.ntiles * g.nte * g.nte;
  if (pid)
    hipLaunchKernelGGL(k_buffer_v_rows<true>, dim3((unsigned)ceil_div(3 * rows, 4)), dim3(256), 0, s, g, ext_off, vp, pid);
  else
    hipLaunchKernelGGL(k_buffer_v_rows<false>, dim3((unsigned)ceil_div(3 * rows, 4)), dim3(256), 0, s, g, ext_off, vp, pid);
  CUBE_HIP(hipGetLastError());
}

void buffer_copy(const Geo& g, const int32_t* rhoc_ext, const int64_t* ext_off, const int64_t* phys_off,
                 const void* xp, const float* vp, const int64_t* pid, void* xp_out, float* vp_out, int64_t* pid_out,
                 hipStream_t s) {
  (void)rhoc_ext;
  const int64_t rows = g.ntiles * g.nte * g.nte;
  if (g.izipx == 2)
    hipLaunchKernelGGL(k_buffer_rows<2>, dim3((unsigned)ceil_div(3 * rows, 4)), dim3(256), 0, s, g, ext_off, phys_off,
                       (const int16_t*)xp, vp, pid, (int16_t*)xp_out, vp_out, pid_out);
  else
    hipLaunchKernelGGL(k_buffer_rows<1>, dim3((unsigned)ceil_div(3 * rows, 4)), dim3(256), 0, s, g, ext_off, phys_off,
                       (const int8_t*)xp, vp, pid, (int8_t*)xp_out, vp_out, pid_out);
  CUBE_HIP(hipGetLastError());
}

}  // namespace cube
