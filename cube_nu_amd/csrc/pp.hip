// pp.hip -- PP_Force (kick.f90:376-588) on the GPU.
//
// Binning: every PP cell (1/ratio_sf of a coarse cell) is nested in exactly
// one coarse cell, so one wavefront per (sub-tile, coarse cell) owns the PP
// cells it fills: counts and in-cell order are deterministic without
// atomics, and the in-cell order is the reference's (coarse-cell particle
// order).
//
// Force: a persistent kernel whose workgroups claim bricks of 4^3 physical PP
// cells from a work queue; each pair of lanes owns a target particle and sums
// the pair force from the 27 neighbouring PP cells in a fixed order.  Both
// members of a physical pair evaluate the pair, so no cross-thread
// accumulation is needed and the result is deterministic.
// The in-range test uses the reference's FP32 operations on exact FP32
// positions, so the set of interacting pairs is the reference's.
#include "pm.h"
#include "pp.h"

namespace cube {
namespace {

template <int IZ>
using XT = typename XP<IZ>::T;

// PP cell of a particle, kick.f90:420-431 in FP32, and its x sub-bin: the
// PP cell idx covers xv in [idx-1, idx), and sub-bin q = floor(kSX * frac(xv))
// (exact: xv - floor(xv) and the power-of-two product are exact in FP32).
template <int IZ>
__device__ inline bool pp_cell(const PPLevel& L, const PPBox& B, int ci, int cj, int ck, const XT<IZ>* xp, int64_t ip,
                               float xf[3], int idx[3], int& q) {
  const int ijk[3] = {ci, cj, ck};
  bool in = true;
  for (int d = 0; d < 3; ++d) {
    // (ijk - 1) + (u + 1/2) 2^-B, rounded once: as an integer of 2^-(B+1) (tiles are far below 2^14 cells)
    const int v = (ijk[d] - 1) * (2 << XP<IZ>::B) + 2 * (int)XP<IZ>::raw(xp, ip, d) + 1;
    const float xvec = (float)v * (1.0f / (float)(2 << XP<IZ>::B));
    xf[d] = xvec * (float)L.rcs;
    float xv = (float)L.sf * (xvec - (float)(B.ifs[d] * L.ntt));
    const float fl = floorf(xv);
    idx[d] = (int)fl + 1;
    if (d == 0) q = min((int)((xv - fl) * (float)kSX), kSX - 1);
    in = in && idx[d] >= 0 && idx[d] <= L.npgrid + 1;
  }
  return in;
}

// One wavefront per (box, coarse cell of the sub-tile + 1-cell ring), one
// particle per lane.  A PP cell lies inside one coarse cell (idx =
// floor(sf*(xvec - ifs*ntt)) + 1 with xvec < c), so the wavefront owns the
// counts of the nsb = sf^3 * kSX sub-bins of its coarse cell and keeps them in
// LDS (dynamic, nsb ints per wavefront).  The lanes holding the same sub-bin
// key are found with one ballot per key bit; a lane's rank among them is a
// population count, so within a sub-bin the order is the coarse-cell particle
// order, and the lowest such lane advances the sub-bin's LDS counter (one
// writer per key).  FILL=0 writes the counts, FILL=1 the entries at
// start + rank.  Sub-bins are numbered ((z*m + y)*m + x)*kSX + q: each (y, z)
// row of the PP grid is one contiguous, x-ordered run of the CSR.  The count pass
// needs no order: LDS adds take the ballots' place, and it writes every sub-bin, so
// that none is cleared first.  Bound by a chain of loads per wavefront (the texture
// data unit is busy 99 % of the cycles, the vector pipe 53 and 47 % of its issue
// slots): 512^3 2.0 + 2.9 ms (2.5 + 2.9 with ballots in both; 3 GB of entries).
template <int IZ, int FILL>
__global__ void __launch_bounds__(256) k_pp_bin(PPLevel L, const PPBox* __restrict__ boxes, int nbox,
                                                const XT<IZ>* __restrict__ xp, const int32_t* __restrict__ rhoc,
                                                const int64_t* __restrict__ off, int32_t* __restrict__ count,
                                                const uint32_t* __restrict__ start, float4* __restrict__ ent) {
  extern __shared__ int lcnt[];
  const int nr = L.ntt + 2;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (FILL && blockIdx.x == 0 && threadIdx.x < kPPPad) {
    // the padding behind the last entry is read (and weighted with zero): finite
    const int64_t m1 = L.npgrid + 2;
    ent[start[nbox * m1 * m1 * m1 * kSX] + threadIdx.x] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
  // 32-bit: a 64-bit division is ~100 instructions, and an image has far fewer than 2^32 coarse cells
  const uint32_t wv = blockIdx.x * 4u + (uint32_t)wave;
  if (wv >= (uint32_t)nbox * nr * nr * nr) return;
  const int ib = (int)(wv / (uint32_t)(nr * nr * nr));
  const int qc = (int)(wv % (uint32_t)(nr * nr * nr));
  const PPBox B = boxes[ib];
  const int c[3] = {B.ifs[0] * L.ntt + (qc % nr), B.ifs[1] * L.ntt + (qc / nr) % nr,
                    B.ifs[2] * L.ntt + qc / (nr * nr)};  // nc1-1 + offset (Fortran nc1 = ifs*ntt+1)
  const int64_t cell = rc_index(c[0], c[1], c[2], B.T, L.nte, L.ncb);
  const int cnt = rhoc[cell];
  const int64_t base = off[cell], tile = off[(int64_t)B.T * L.nte * L.nte * L.nte];
  const int m = L.npgrid + 2;
  const int sf = L.sf, nsb = sf * sf * sf * kSX;
  const int kbits = 32 - __clz(nsb - 1);  // bits of a sub-bin key
  int lo[3];  // PP index of the coarse cell's first PP cell per axis
  for (int d = 0; d < 3; ++d) lo[d] = sf * (c[d] - 1 - B.ifs[d] * L.ntt) + 1;
  int* lc = lcnt + wave * nsb;
  for (int t = lane; t < nsb; t += 64) lc[t] = 0;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int64_t cbase = (int64_t)ib * m * m * m;
  const unsigned long long lt = (1ull << lane) - 1ull;
  for (int l0 = 0; l0 < cnt; l0 += 64) {
    const int l = l0 + lane;
    float xf[3] = {0, 0, 0};
    int idx[3] = {0, 0, 0};
    int q = 0;
    bool in = false;
    if (l < cnt) in = pp_cell<IZ>(L, B, c[0], c[1], c[2], xp, base + l, xf, idx, q);
    const int key = in ? (((idx[2] - lo[2]) * sf + (idx[1] - lo[1])) * sf + (idx[0] - lo[0])) * kSX + q : 0;
    if (!FILL) {  // counts need no order
      if (in) atomicAdd(&lc[key], 1);
      continue;
    }
    unsigned long long eq = __ballot(in);
    for (int bt = 0; bt < kbits; ++bt) {
      const unsigned long long mb = __ballot((key >> bt) & 1);
      eq &= ((key >> bt) & 1) ? mb : ~mb;
    }
    const int prev = in ? lc[key] : 0;
    if (in) {
      const int rank = (int)__popcll(eq & lt);
      const int64_t pc = cbase + ((int64_t)idx[2] * m + idx[1]) * m + idx[0];
      bool ghost = false;
      for (int d = 0; d < 3; ++d) ghost = ghost || idx[d] == 0 || idx[d] == L.npgrid + 1;
      // particle index within its tile, ghosts of the sub-tile marked by the sign
      ent[start[pc * kSX + q] + prev + rank] = make_float4(
          xf[0], xf[1], xf[2], __uint_as_float((unsigned)(base + l - tile) | (ghost ? 0x80000000u : 0u)));
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (in && (eq & lt) == 0) lc[key] = prev + (int)__popcll(eq);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  if (!FILL) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int t = lane; t < nsb; t += 64) {
      // every sub-bin of the grid belongs to one coarse cell (the ghost ones hang over its edge)
      const int pc = t / kSX;
      const int ix = lo[0] + pc % sf, iy = lo[1] + (pc / sf) % sf, iz = lo[2] + pc / (sf * sf);
      if ((unsigned)ix < (unsigned)m && (unsigned)iy < (unsigned)m && (unsigned)iz < (unsigned)m)
        count[(cbase + ((int64_t)iz * m + iy) * m + ix) * kSX + t % kSX] = lc[t];
    }
  }
}

// Physical PP cells per brick per dim.
constexpr int kPB = 4;
// Lanes per target in the FP32 force kernel: a target's candidates are dealt
// to kPPGroup lanes in turn and their partial sums combined at the end (pairs
// of lanes read consecutive entries).
constexpr int kPPGroup = 2;

// FP32 pair law.  F(r, app) - F(r, r_pp) = 1/r^2 - c Q(ep) for r > app, with
// ep = 2r/r_pp < 2 and Q the two polynomials of F_ra (kick.f90:360-374; Q =
// 12/ep^2 + po(ep) above ep = 1).  Q comes from a cubic Hermite table over kQSeg
// segments of [0, 2] kept in LDS: ep = 1 is a segment edge and Q is C^1 there; its
// error is below 2e-5 on |Q| <= 104 (h^4 max|Q^(4)| / 384 with h = 1/32), below
// 1e-6 of 1/r_pp^2 in the pair force, at the level of FP32 rounding.  (A table in
// r^2 saves two operations of a pair and 6 % of the time, but its rounding moves
// the largest force, and with it the time step and the coordinates' last bits.)
constexpr int kQSeg = 64;

__device__ inline void q_branch(double e, bool outer, double& q, double& dq) {
  if (outer) {
    q = 12.0 / (e * e) + (((((7.0 * e - 48.0) * e + 70.0) * e + 224.0) * e - 840.0) * e + 896.0) * e - 224.0;
    dq = -24.0 / (e * e * e) + ((((42.0 * e - 240.0) * e + 280.0) * e + 672.0) * e - 1680.0) * e + 896.0;
  } else {
    q = e * (224.0 + e * e * (-224.0 + e * (70.0 + e * (48.0 - 21.0 * e))));
    dq = 224.0 + e * e * (-672.0 + e * (280.0 + e * (240.0 - 126.0 * e)));
  }
}

// Segment s of the table: Q(s h + f h) = ((c.w f + c.z) f + c.y) f + c.x; entry
// kQSeg holds the last one's value at f = 1 (an r just below r_pp may round to it).
__device__ inline void fill_qtab(float4* tab) {
  for (int sg = threadIdx.x; sg <= kQSeg; sg += blockDim.x) {
    const double h = 2.0 / kQSeg;
    const int i = min(sg, kQSeg - 1);
    const bool outer = i >= kQSeg / 2;
    double y0, d0, y1, d1;
    q_branch(i * h, outer, y0, d0);
    q_branch((i + 1) * h, outer, y1, d1);
    d0 *= h;
    d1 *= h;
    const float4 c = make_float4((float)y0, (float)d0, (float)(3.0 * (y1 - y0) - 2.0 * d0 - d1),
                                 (float)(2.0 * (y0 - y1) + d0 + d1));
    tab[sg] = sg < kQSeg ? c : make_float4(((c.w + c.z) + c.y) + c.x, 0.0f, 0.0f, 0.0f);
  }
}

// Q(2r/r_pp) at t = r kQSeg / r_pp (beyond the range: its end value).
__device__ inline float q_range(const float4* tab, float t) {
  t = fminf(t, (float)kQSeg);
  const float4 c = tab[(int)t];
  const float f = __builtin_amdgcn_fractf(t);
  return fmaf(fmaf(fmaf(c.w, f, c.z), f, c.y), f, c.x);
}

// F(r, app) in full for the rare r <= app (ep <= 2).
__device__ inline float f_app(const PPLevel& L, float r) {
  const float ea = (2.0f * r) * L.inv_app;
  const float a2 = ea * ea;
  return ea > 1.0f
             ? L.c_app * (12.0f * __builtin_amdgcn_rcpf(a2) +
                          fmaf(ea, fmaf(ea, fmaf(ea, fmaf(ea, fmaf(ea, fmaf(ea, 7.0f, -48.0f), 70.0f), 224.0f),
                                                 -840.0f),
                                        896.0f),
                               -224.0f))
             : L.c_app * ea * fmaf(a2, fmaf(ea, fmaf(ea, fmaf(ea, -21.0f, 48.0f), 70.0f), -224.0f), 224.0f);
}

// FP64 form: the reference's operations (kick.f90:523-530, 554-560) in FP64:
// f1 += (x2-x1)/r * (F(r,app) - F(r,r_pp)).
__device__ inline void pair_force64(const PPLevel& L, const float4 me, const float4 o, double f1[3]) {
  const double rv0 = (double)o.x - me.x, rv1 = (double)o.y - me.y, rv2 = (double)o.z - me.z;
  const double r2 = (rv0 * rv0 + rv1 * rv1) + rv2 * rv2;
  const double r = sqrt(r2);
  const double fr = f_ra<double>(r, (double)L.app, f_ra_coef<double>((double)L.app)) -
                    f_ra<double>(r, (double)L.pp_range, f_ra_coef<double>((double)L.pp_range));
  f1[0] = f1[0] + (rv0 / r) * fr;
  f1[1] = f1[1] + (rv1 / r) * fr;
  f1[2] = f1[2] + (rv2 / r) * fr;
}

// Bricks of kPB^3 physical PP cells are claimed by persistent workgroups from
// kPPClaimCounters counters (workgroup i uses counter i % 8) until none remain.
// With at least 64 sub-tiles a counter hands out the bricks of sub-tiles ctr,
// ctr + 8, ... (the host's densest-first order, kick.f90:132-138), one sub-tile's
// bricks in turn, so that they run on one XCD and share its L2; with fewer, it
// hands out bricks 8 k + ctr, so that every counter has work.  A claim is one of
// `parts` shares of a brick's targets: with few bricks a launch would end on
// the densest one's workgroup (64^3 particles, 4096 bricks: 365 us with whole
// bricks, 309 in shares, 202 with the counters and the output slots on cache
// lines of their own; 128^3, 32768 bricks: 0.48 ms against 1.25 at the start).
// A workgroup's first claim is its own place in the queue; the counters, each
// on a cache line of its own, hand out the rest.
__device__ inline int64_t claim_brick(unsigned* claim, bool first, int64_t nbricks, int64_t nbps, bool xcd_local) {
  const int ctr = blockIdx.x % kPPClaimCounters;
  const int64_t k = first ? (int64_t)(blockIdx.x / kPPClaimCounters)
                          : (int64_t)atomicAdd(&claim[ctr * kPPClaimStride], 1u) +
                                (gridDim.x - ctr + kPPClaimCounters - 1) / kPPClaimCounters;
  if (!xcd_local) return min(k * kPPClaimCounters + ctr, nbricks);
  const int64_t box = (k / nbps) * kPPClaimCounters + ctr;
  return box < nbricks / nbps ? box * nbps + k % nbps : nbricks;
}

// A brick's tables: rs, the starts of the x sub-bins of its (kPB+2)^2 rows
// (cells c0-1 .. c0+kPB along x; rows outside the PP grid are empty, sub-bins
// past a row's end read the end), and pre, the prefix sums of its cells' counts.
constexpr int kNB = kPB + 2, kRW = kSX * kNB + 1;
struct Brick {
  int ib, c0[3];
};
__device__ inline Brick brick_tables(const PPLevel& L, int64_t brick, int nbr, const uint32_t* __restrict__ start,
                                     int* rs, int* pre) {
  Brick K;
  const uint32_t b = (uint32_t)brick, n = (uint32_t)nbr;  // nbox nbr^3 < 2^32
  K.c0[0] = 1 + (int)(b % n) * kPB;
  K.c0[1] = 1 + (int)((b / n) % n) * kPB;
  K.c0[2] = 1 + (int)((b / (n * n)) % n) * kPB;
  K.ib = (int)(b / (n * n * n));
  const int m = L.npgrid + 2, mS = m * kSX;
  const int64_t cbase = (int64_t)K.ib * m * m * m;
  for (int q = threadIdx.x; q < kNB * kNB * kRW; q += blockDim.x) {
    const int row = q / kRW, xs = q - row * kRW, y = K.c0[1] - 1 + row % kNB, z = K.c0[2] - 1 + row / kNB;
    int st = 0;
    if (y <= L.npgrid + 1 && z <= L.npgrid + 1)
      st = (int)start[(cbase + ((int64_t)z * m + y) * m) * kSX + min(kSX * (K.c0[0] - 1) + xs, mS)];
    rs[q] = st;
  }
  __syncthreads();
  if (threadIdx.x < kPB * kPB * kPB) {  // one wavefront: cell counts and their prefix sums
    const int q = threadIdx.x, lx = q % kPB, ly = (q / kPB) % kPB, lz = q / (kPB * kPB);
    const int row = ((lz + 1) * kNB + ly + 1) * kRW;
    const bool in = K.c0[0] + lx <= L.npgrid && K.c0[1] + ly <= L.npgrid && K.c0[2] + lz <= L.npgrid;
    int s = in ? rs[row + kSX * (lx + 2)] - rs[row + kSX * (lx + 1)] : 0;
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(s, o, 64);
      if (q >= o) s += v;
    }
    pre[q + 1] = s;
    if (q == 0) pre[0] = 0;
  }
  __syncthreads();
  return K;
}
static_assert(kPB * kPB * kPB == 64, "a brick's cells are one wavefront");

// Cell of a brick's target t: the largest c with pre[c] <= t.
__device__ inline int target_cell(const int* pre, int t) {
  int lo = 0;
#pragma unroll
  for (int s = kPB * kPB * kPB / 2; s > 0; s >>= 1)
    if (pre[lo + s] <= t) lo += s;
  return lo;
}

// The x window of the (dy, dz) column of PP cells around a target: a partner
// at y/z distance >= (ey, ez) is in range only within x +- sqrt(r_pp^2 - ey^2 -
// ez^2), a contiguous run of the x-ordered row, found from two sub-bin starts.
// fr: the target's offset in its PP cell; u: its x in sub-bins of the staged
// rows; lx: its cell.  The cut carries a margin of 1e-3 cell, far above the
// rounding here, so every pair the reference tests in range is in a window.
__device__ inline void column_run(const PPLevel& L, const int* rs, int rowt, int lx, float u, const float fr[3],
                                  int dy, int dz, int& beg, int& n) {
  const float ey = dy < 0 ? fr[1] : (dy > 0 ? 1.0f - fr[1] : 0.0f);
  const float ez = dz < 0 ? fr[2] : (dz > 0 ? 1.0f - fr[2] : 0.0f);
  const float e2 = ey * ey + ez * ez;
  const float hw = (float)kSX * __builtin_amdgcn_sqrtf(fmaxf(L.rcut2 - e2, 0.0f));
  const int wlo = max((int)floorf(u - hw), kSX * lx);
  const int whi = min((int)floorf(u + hw), kSX * (lx + 3) - 1);
  const int row = rowt + (dz * kNB + dy) * kRW;
  beg = rs[row + wlo];
  n = e2 < L.rcut2 ? rs[row + whi + 1] - beg : 0;
}

// Maxima and pair counts of a workgroup into its slot (one wavefront's atomics).
__device__ inline void pp_reduce(PPOut* __restrict__ out, float f2, const float vm[3], unsigned long long npp,
                                 unsigned long long npg) {
  __shared__ float rm[4][4];
  __shared__ unsigned long long rc[4][2];
  float v[4] = {f2, vm[0], vm[1], vm[2]};
  for (int o = 32; o > 0; o >>= 1)
    for (int k = 0; k < 4; ++k) v[k] = fmaxf(v[k], __shfl_xor(v[k], o, 64));
  for (int o = 32; o > 0; o >>= 1) {
    npp += __shfl_xor(npp, o, 64);
    npg += __shfl_xor(npg, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    const int w = threadIdx.x >> 6;
    for (int k = 0; k < 4; ++k) rm[w][k] = v[k];
    rc[w][0] = npp;
    rc[w][1] = npg;
  }
  __syncthreads();
  PPOut::Slot& sl = out->slot[blockIdx.x % kSumSlots];
  if (threadIdx.x < 4) {
    const int k = threadIdx.x;
    const float m = fmaxf(fmaxf(rm[0][k], rm[1][k]), fmaxf(rm[2][k], rm[3][k]));
    atomic_max_nonneg(k == 0 ? &sl.f2max : &sl.vmax[k - 1], m);
  } else if (threadIdx.x < 6) {
    const int k = threadIdx.x - 4;
    const unsigned long long c = rc[0][k] + rc[1][k] + rc[2][k] + rc[3][k];
    if (c) atomicAdd(k == 0 ? &sl.pairs_pp : &sl.pairs_pg, c);
  }
}

// v += f mass_scale a_mid dt/6/pi (kick.f90:576-582): g = fl32(f mass_scale) as
// the reference forms it, times the FP64 coefficient, added in FP64.
__device__ inline void pp_kick(const PPLevel& L, double vsc, const float f[3], float* __restrict__ vp, int64_t ip,
                               float& f2, float vm[3]) {
  float g[3];
  for (int d = 0; d < 3; ++d) g[d] = f[d] * L.mass_scale;
  f2 = fmaxf(f2, (g[0] * g[0] + g[1] * g[1]) + g[2] * g[2]);
  for (int d = 0; d < 3; ++d) {
    const float v = (float)((double)vp[3 * ip + d] + (double)g[d] * vsc);
    vp[3 * ip + d] = v;
    vm[d] = fmaxf(vm[d], fabsf(v));
  }
}

// FP32 force.  Two lanes per target particle; a wavefront's 32 targets first
// write their windows in the nine (dy, dz) columns to LDS (each lane every
// other column; empty ones dropped), then each pair of lanes walks its own
// list of runs, 2 U entries at a time, lane j taking entries j, j + 2, ... .  So a
// wavefront runs as long as its longest target, not the sum over columns of
// its longest column.  Entries are read U at a time straight from L1/L2 (the
// array is padded, so the reads need no clamp) and tested with the reference's
// FP32 operations on exact positions: the interacting set is the reference's.
// Both members of a physical pair evaluate it, and a target's partial sums are
// added in a fixed order (its columns in turn, each dealt to the two lanes), so the
// result is deterministic.
//
// U reads in flight per lane against wavefronts per SIMD: 3 with eight (64
// VGPRs) is the fastest on long lists of short runs, whose reads miss L1 (512^3
// at z = 2: 23.2 ms; 4 with eight 23.6, 6 with five 27), 6 with five (96
// VGPRs) on the long runs of clustered input (192^3 at z = 0.5: 3.0 ms against
// 3.5), 4 with seven between them (64^3); the engine's autotuner picks.  At 512^3
// (2.85e9 pairs) 23.2 ms are 4.9 TFLOP/s at 40 flops a pair (25.4 ms with the
// columns walked in step and a branch per pair); TA is busy 80% and VALU 68% of
// the cycles.  Slower, on the form with columns in step: candidates staged in
// LDS (50 KB a workgroup leave three wavefronts per SIMD), 8-byte exact-integer
// entries (half the load traffic, 30% more VALU), a two-pass form with in-range
// masks, PP cells split along y as well, one or four lanes per target.
constexpr int pp_workgroups(int u) { return u == 3 ? 8 : (u == 4 ? 7 : 5); }
template <int U>
__global__ void __launch_bounds__(256, pp_workgroups(U)) k_pp_force(PPLevel L, const PPBox* __restrict__ boxes, int64_t nbricks,
                                                     const uint32_t* __restrict__ start,
                                                     const float4* __restrict__ ent, const int64_t* __restrict__ off,
                                                     float* __restrict__ vp, PPOut* __restrict__ out,
                                                     unsigned* __restrict__ claim, bool xcd_local, int parts) {
  constexpr int G = kPPGroup;
  static_assert(G == 2, "two lanes per target");
  __shared__ int rs[kNB * kNB * kRW];
  __shared__ int pre[kPB * kPB * kPB + 1];
  __shared__ float4 qtab[kQSeg + 1];
  __shared__ int2 cols[4][32][9];
  __shared__ int64_t s_brick;
  fill_qtab(qtab);
  const float tscale = L.two_inv_range * (0.5f * kQSeg);
  const double vsc = L.vdev ? *L.vdev : L.v_scale;
  const int nbr = (L.npgrid + kPB - 1) / kPB;
  const int lane = threadIdx.x & 63, gj = lane & 1;
  int2* run = cols[threadIdx.x >> 6][lane >> 1];
  float f2 = 0, vm[3] = {0, 0, 0};
  unsigned long long npp = 0, npg = 0;
  for (bool first = true;; first = false) {
    __syncthreads();  // the previous brick's tables are no longer read
    if (threadIdx.x == 0)
      s_brick = claim_brick(claim, first, nbricks * parts, (int64_t)nbr * nbr * nbr * parts,
                            xcd_local);
    __syncthreads();
    if (s_brick >= nbricks * parts) break;
    const int part = (int)(s_brick % parts);
    const Brick K = brick_tables(L, s_brick / parts, nbr, start, rs, pre);
    const PPBox B = boxes[K.ib];
    const int64_t tile = off[(int64_t)B.T * L.nte * L.nte * L.nte];
    const int nall_t = pre[kPB * kPB * kPB], ntg = (int)((int64_t)nall_t * (part + 1) / parts);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int t0 = (int)((int64_t)nall_t * part / parts) + wave * 32; t0 < ntg; t0 += 128) {
      const int t = t0 + (lane >> 1);
      const bool ok = t < ntg;
      float4 me = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      int ncol = 0;
      if (ok) {
        const int c = target_cell(pre, t);
        const int lc[3] = {c % kPB, (c / kPB) % kPB, c / (kPB * kPB)};
        const int rowt = ((lc[2] + 1) * kNB + lc[1] + 1) * kRW;
        me = ent[rs[rowt + kSX * (lc[0] + 1)] + (t - pre[c])];
        // PP coordinates of the target, the binning's xv = sf (xvec - ifs ntt)
        // (xvec = xf / rcs exactly for a power-of-two rcs)
        const float xme[3] = {me.x, me.y, me.z};
        float fr[3];
        for (int d = 0; d < 3; ++d) {
          const float xv = (float)L.sf * (xme[d] * L.inv_rcs - (float)(B.ifs[d] * L.ntt));
          fr[d] = xv - (float)(K.c0[d] - 1 + lc[d]);
        }
        const float u = (fr[0] + (float)(lc[0] + 1)) * (float)kSX;
        int beg[5], n[5], mine = 0;  // columns that hold any, as bits
#pragma unroll
        for (int i = 0; i < 5; ++i) {
          const int q = 2 * i + gj;  // column (dy, dz) = (q % 3 - 1, q / 3 - 1)
          n[i] = 0;
          beg[i] = 0;
          if (q < 9) column_run(L, rs, rowt, lc[0], u, fr, q % 3 - 1, q / 3 - 1, beg[i], n[i]);
          mine |= (n[i] > 0) << q;
        }
        const int all = mine | __shfl_xor(mine, 1, 64);
        ncol = __popc(all);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
          const int q = 2 * i + gj;
          if (n[i] > 0) run[__popc(all & ((1 << q) - 1))] = make_int2(beg[i], n[i]);
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      float f1[3] = {0, 0, 0};
      int k = 0, p = gj;
      int2 e = ncol > 0 ? run[0] : make_int2(0, 0);
      int npair = 0, nghost = 0;
      while (k < ncol) {
        const float4* src = ent + (e.x + p);
        const int rem = e.y - p;
        float4 o[U];
#pragma unroll
        for (int i = 0; i < U; ++i) o[i] = src[i * G];
        p += U * G;
        if (p >= e.y) {  // the next run
          ++k;
          p = gj;
          e = k < ncol ? run[k] : make_int2(0, 0);
        }
        // U pairs side by side, without a branch: of 64 lanes one is nearly
        // always in range
        float rv[U][3], r2[U], sc[U];
        bool in[U], near = false;
#pragma unroll
        for (int i = 0; i < U; ++i) {
          rv[i][0] = o[i].x - me.x;
          rv[i][1] = o[i].y - me.y;
          rv[i][2] = o[i].z - me.z;
          r2[i] = (rv[i][0] * rv[i][0] + rv[i][1] * rv[i][1]) + rv[i][2] * rv[i][2];
          in[i] = i * G < rem && 0.0f < r2[i] && r2[i] < L.pp_range2;  // exact-input FP32 test (kick.f90:525, 556)
          near = near || (in[i] && r2[i] <= L.app2);
          const float rinv = __builtin_amdgcn_rsqf(r2[i]);
          sc[i] = rinv * fmaf(-L.c_range, q_range(qtab, (r2[i] * rinv) * tscale), rinv * rinv);
        }
        if (__any(near)) {  // ep(r, app) <= 2: F(r, app) in full
#pragma unroll
          for (int i = 0; i < U; ++i) {
            const float rinv = __builtin_amdgcn_rsqf(r2[i]);
            const float r = r2[i] * rinv;
            if (in[i] && r2[i] <= L.app2)
              sc[i] = rinv * fmaf(-L.c_range, q_range(qtab, r * tscale), f_app(L, r));
          }
        }
#pragma unroll
        for (int i = 0; i < U; ++i) {
          const float g = in[i] ? sc[i] : 0.0f;
          f1[0] = fmaf(rv[i][0], g, f1[0]);
          f1[1] = fmaf(rv[i][1], g, f1[1]);
          f1[2] = fmaf(rv[i][2], g, f1[2]);
          npair += in[i];
          nghost += in[i] && __float_as_int(o[i].w) < 0;
        }
      }
      // the two lanes' sums: each step adds the same two operands on both
      for (int d = 0; d < 3; ++d) f1[d] += __shfl_xor(f1[d], 1, 64);
      npp += (unsigned)(npair - nghost);
      npg += (unsigned)nghost;
      if (ok && gj == 0) pp_kick(L, vsc, f1, vp, tile + (int64_t)(__float_as_uint(me.w) & 0x7fffffffu), f2, vm);
    }
  }  // claimed bricks
  pp_reduce(out, f2, vm, npp, npg);
}

// FP64 form: one lane per target, the pair law in FP64 with the reference's
// operations, the same bricks, windows and in-range test.
__global__ void __launch_bounds__(256) k_pp_force64(PPLevel L, const PPBox* __restrict__ boxes, int64_t nbricks,
                                                    const uint32_t* __restrict__ start,
                                                    const float4* __restrict__ ent, const int64_t* __restrict__ off,
                                                    float* __restrict__ vp, PPOut* __restrict__ out,
                                                    unsigned* __restrict__ claim, bool xcd_local, int parts) {
  constexpr int U = 6;
  static_assert(U <= kPPPad, "reads past a run stay inside the entry padding");
  __shared__ int rs[kNB * kNB * kRW];
  __shared__ int pre[kPB * kPB * kPB + 1];
  __shared__ int64_t s_brick;
  const double vsc = L.vdev ? *L.vdev : L.v_scale;
  const int nbr = (L.npgrid + kPB - 1) / kPB;
  float f2 = 0, vm[3] = {0, 0, 0};
  unsigned long long npp = 0, npg = 0;
  for (bool first = true;; first = false) {
    __syncthreads();
    if (threadIdx.x == 0)
      s_brick = claim_brick(claim, first, nbricks * parts, (int64_t)nbr * nbr * nbr * parts,
                            xcd_local);
    __syncthreads();
    if (s_brick >= nbricks * parts) break;
    const int part = (int)(s_brick % parts);
    const Brick K = brick_tables(L, s_brick / parts, nbr, start, rs, pre);
    const PPBox B = boxes[K.ib];
    const int64_t tile = off[(int64_t)B.T * L.nte * L.nte * L.nte];
    const int nall_t = pre[kPB * kPB * kPB], ntg = (int)((int64_t)nall_t * (part + 1) / parts);
    for (int t = (int)((int64_t)nall_t * part / parts) + threadIdx.x; t < ntg; t += 256) {
      const int c = target_cell(pre, t);
      const int lc[3] = {c % kPB, (c / kPB) % kPB, c / (kPB * kPB)};
      const int rowt = ((lc[2] + 1) * kNB + lc[1] + 1) * kRW;
      const float4 me = ent[rs[rowt + kSX * (lc[0] + 1)] + (t - pre[c])];
      const float xme[3] = {me.x, me.y, me.z};
      float fr[3];
      for (int d = 0; d < 3; ++d) {
        const float xv = (float)L.sf * (xme[d] * L.inv_rcs - (float)(B.ifs[d] * L.ntt));
        fr[d] = xv - (float)(K.c0[d] - 1 + lc[d]);
      }
      const float u = (fr[0] + (float)(lc[0] + 1)) * (float)kSX;
      double f1[3] = {0, 0, 0};
      int npair = 0, nghost = 0;
      for (int dz = -1; dz <= 1; ++dz)
        for (int dy = -1; dy <= 1; ++dy) {
          int beg, nn;
          column_run(L, rs, rowt, lc[0], u, fr, dy, dz, beg, nn);
          const float4* run = ent + beg;
          for (int p = 0; p < nn; p += U) {
            float4 o[U];
#pragma unroll
            for (int k = 0; k < U; ++k) o[k] = run[p + k];
#pragma unroll
            for (int k = 0; k < U; ++k) {
              const float rv0 = o[k].x - me.x, rv1 = o[k].y - me.y, rv2 = o[k].z - me.z;
              const float r2 = (rv0 * rv0 + rv1 * rv1) + rv2 * rv2;
              if (p + k < nn && 0.0f < r2 && r2 < L.pp_range2) {
                pair_force64(L, me, o[k], f1);
                ++npair;
                nghost += __float_as_int(o[k].w) < 0;
              }
            }
          }
        }
      npg += (unsigned)nghost;
      npp += (unsigned)(npair - nghost);
      const float f[3] = {(float)f1[0], (float)f1[1], (float)f1[2]};
      pp_kick(L, vsc, f, vp, tile + (int64_t)(__float_as_uint(me.w) & 0x7fffffffu), f2, vm);
    }
  }
  pp_reduce(out, f2, vm, npp, npg);
}

}  // namespace

int64_t pp_bin_count(int izipx, const PPLevel& L, const PPBox* boxes, int nbox, const void* xp, const int32_t* rhoc,
                     const int64_t* off, PPScratch& S, hipStream_t s) {
  const int m = L.npgrid + 2;
  const int64_t ncell = (int64_t)nbox * m * m * m * kSX;
  const int nr = L.ntt + 2;
  const int64_t nthr = (int64_t)nbox * nr * nr * nr * 64;
  const size_t lds = sizeof(int) * 4 * L.sf * L.sf * L.sf * kSX;
  if (izipx == 2)
    hipLaunchKernelGGL((k_pp_bin<2, 0>), dim3((unsigned)ceil_div(nthr, 256)), dim3(256), lds, s, L, boxes, nbox,
                       (const int16_t*)xp, rhoc, off, S.count, nullptr, nullptr);
  else
    hipLaunchKernelGGL((k_pp_bin<1, 0>), dim3((unsigned)ceil_div(nthr, 256)), dim3(256), lds, s, L, boxes, nbox,
                       (const int8_t*)xp, rhoc, off, S.count, nullptr, nullptr);
  CUBE_HIP(hipGetLastError());
  const int64_t* sum = scan_counts32(S.count, S.start, ncell, S.scan_tmp, S.scan_tmp_bytes, s);
  int64_t total = 0;
  ReadBack rb(*S.page);
  rb.get(&total, sum, sizeof(total), s);
  rb.wait();
  return total;
}

void pp_bin_fill(int izipx, const PPLevel& L, const PPBox* boxes, int nbox, const void* xp, const int32_t* rhoc,
                 const int64_t* off, PPScratch& S, hipStream_t s) {
  const int nr = L.ntt + 2;
  const int64_t nthr = (int64_t)nbox * nr * nr * nr * 64;
  const size_t lds = sizeof(int) * 4 * L.sf * L.sf * L.sf * kSX;
  if (izipx == 2)
    hipLaunchKernelGGL((k_pp_bin<2, 1>), dim3((unsigned)ceil_div(nthr, 256)), dim3(256), lds, s, L, boxes, nbox,
                       (const int16_t*)xp, rhoc, off, S.count, S.start, S.entries);
  else
    hipLaunchKernelGGL((k_pp_bin<1, 1>), dim3((unsigned)ceil_div(nthr, 256)), dim3(256), lds, s, L, boxes, nbox,
                       (const int8_t*)xp, rhoc, off, S.count, S.start, S.entries);
  CUBE_HIP(hipGetLastError());
}

template <int U>
static void launch_pp_f32(dim3 grid, hipStream_t s, const PPLevel& L, const PPBox* boxes, int64_t nbricks,
                          PPScratch& S, const int64_t* off, float* vp, PPOut* out, bool xcd_local, int parts) {
  static_assert(U * kPPGroup <= kPPPad, "reads past a run stay inside the entry padding");
  hipLaunchKernelGGL((k_pp_force<U>), grid, dim3(256), 0, s, L, boxes, nbricks, S.start, S.entries, off, vp, out,
                     S.claim, xcd_local, parts);
}

void pp_force(const PPLevel& L, int precision, const PPBox* boxes, int nbox, const int64_t* off, float* vp,
              PPScratch& S, PPOut* out, hipStream_t s, int unroll) {
  const int64_t nbr = (L.npgrid + kPB - 1) / kPB;
  const int64_t nbricks = nbr * nbr * nbr * nbox;
  static int n_cu = 0;
  if (n_cu == 0) {
    int dev = 0;
    CUBE_HIP(hipGetDevice(&dev));
    CUBE_HIP(hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev));
  }
  zero_async(S.claim, sizeof(unsigned) * kPPClaimCounters * kPPClaimStride, s);
  // as many workgroups as fit on the chip at once (the launch bound's
  // occupancy in the FP32 form, four in the FP64 form), each then claims bricks
  // until none remain
  const int per_cu = precision == 64 ? 4 : pp_workgroups(unroll);
  const int64_t resident = (int64_t)n_cu * per_cu;
  // shares of a brick: enough claims that the last ones are short
  const int parts = (int)std::max<int64_t>(1, std::min<int64_t>(8, ceil_div(8 * resident, std::max<int64_t>(nbricks, 1))));
  const dim3 grid((unsigned)std::min<int64_t>(nbricks * parts, resident));
  const bool xcd_local = nbox >= 64;  // whole sub-tiles per counter only when there are enough of them
  if (precision == 64)
    hipLaunchKernelGGL(k_pp_force64, grid, dim3(256), 0, s, L, boxes, nbricks, S.start, S.entries, off, vp, out,
                       S.claim, xcd_local, parts);
  else if (unroll == 4)
    launch_pp_f32<4>(grid, s, L, boxes, nbricks, S, off, vp, out, xcd_local, parts);
  else if (unroll == 6)
    launch_pp_f32<6>(grid, s, L, boxes, nbricks, S, off, vp, out, xcd_local, parts);
  else
    launch_pp_f32<3>(grid, s, L, boxes, nbricks, S, off, vp, out, xcd_local, parts);
  CUBE_HIP(hipGetLastError());
}

}  // namespace cube
