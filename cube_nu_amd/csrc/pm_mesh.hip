// pm_mesh.hip -- tile and sub-tile densities from one deposit per mesh
// resolution.
//
// The windows of the tile (PM2) and sub-tile (PM3) meshes overlap by their
// buffers: depositing per window repeats every particle 1.95 times at 512^3,
// 8 at 128^3 and 27 at 64^3.  The buffer cells are periodic images of the
// physical ones, and the deposit sums integers, so a window's density is, bit
// for bit, a cut from the periodic mesh of the whole image at that resolution
// -- but for the window's outermost layer of cells, which lacks the taps of
// the particles outside the window.  So every physical particle is deposited
// once into the image's mesh (k_mesh_deposit), the six faces of every window
// are summed on their own from the window's boundary coarse cells
// (k_mesh_faces: a quarter of their particles at w = 8, nine taps each), and
// k_mesh_window cuts the windows out.
#include <algorithm>

#include "grid.h"
#include "pm_dev.h"
#include "pm_mesh.h"

namespace cube {
namespace {

// The three encoded coordinates of particle ip, in two loads.
template <int IZ>
__device__ inline void load_xp(const XT<IZ>* __restrict__ xp, int64_t ip, uint32_t u[3]) {
  const XT<IZ>* p = xp + 3 * ip;
  if constexpr (IZ == 2) {
    uint32_t xy;
    __builtin_memcpy(&xy, p, 4);
    u[0] = xy & 0xffffu;
    u[1] = xy >> 16;
    u[2] = (uint16_t)p[2];
  } else {
    uint16_t xy;
    __builtin_memcpy(&xy, p, 2);
    u[0] = xy & 0xffu;
    u[1] = xy >> 8;
    u[2] = (uint8_t)p[2];
  }
}

// Mesh of the whole image: cell a covers [a, a+1) mesh units; a particle with
// floor f deposits into f-1, f, f+1 with the weights of particle_mesh.f90:56-62.
//
// Workgroup = BD^3 cells [BD b - 1, BD b + BD - 2] per axis: with this offset
// the contributors are the block's own coarse cells and one lower layer,
// (BD/w + 1)^3 cells; of a lower cell's particles those in the last two mesh
// layers along each lower axis reach the block.  The cells' particles form one
// list (LDS prefix sum of the counts) that the wavefronts share in 8 segments
// each; lane l reads particle l/8, l/8 + 8, ... of segment l%8, so that the 64
// lanes of a deposit come from 8 places of the block: particles of one coarse
// cell share few mesh cells, and their atomics would serialise (a
// microbenchmark of 64-bit LDS adds: 18.5 CU cycles per wavefront from one
// 4^3-cell coarse cell, 13.2 from several).  Hits (1.42 per particle at BD =
// 16) queue per wavefront and are deposited 64 at a time into 2^-32
// fixed-point sums; rows are padded to BD + 1 cells, so that the 27 addresses
// are one base and constant offsets and neighbouring rows start in other banks.
// 512^3 particles: 2.6 ms at w = 4 (512^3 mesh), 4.5 at w = 8 (1024^3 mesh, 4.3
// GB written); the deposit per window took 8.9 and 6.4 + 5.8 for its lists.
template <int IZ, int BD>
__global__ void __launch_bounds__(256) k_mesh_deposit(MeshGeo M, const XT<IZ>* __restrict__ xp,
                                                      const int32_t* __restrict__ rhoc,
                                                      const int64_t* __restrict__ off, float* __restrict__ mesh,
                                                      float mass) {
  constexpr int MAXC = (BD / 4 + 1) * (BD / 4 + 1) * (BD / 4 + 1);
  constexpr int NS = 32;  // list segments of a workgroup
  constexpr int SY = BD + 1, SZ = BD * SY;
  __shared__ unsigned long long acc[BD * SZ];
  __shared__ unsigned long long queue[4][128];
  __shared__ int cnt[MAXC], pre[MAXC + 1], wsum[4];
  __shared__ uint32_t gof[MAXC];        // first particle of a cell (the caller holds np < 2^32)
  __shared__ unsigned short key[MAXC];  // cell coordinates l (3 bits each), bit 9 + d: l_d == 0
  const int nb = M.n / BD, g = BD / M.w, gc = g + 1;
  const int b = (int)xcd_block(blockIdx.x, gridDim.x);
  const int bi[3] = {b % nb, (b / nb) % nb, b / (nb * nb)};
  const int nC = gc * gc * gc;
  for (int t = threadIdx.x; t < nC; t += 256) {
    const int l[3] = {t % gc, (t / gc) % gc, t / (gc * gc)};
    int T = 0, c[3], k = 0;
    for (int d = 2; d >= 0; --d) {
      int cc = bi[d] * g - 1 + l[d];
      cc = cc < 0 ? cc + M.nc : cc;
      const int it = cc / M.nt;
      c[d] = cc - it * M.nt + 1;
      T = T * M.nnt + it;
      k |= (l[d] << (3 * d)) | (l[d] == 0 ? 512 << d : 0);
    }
    const int64_t cell = rc_index(c[0], c[1], c[2], T, M.nte, M.ncb);
    cnt[t] = rhoc[cell];
    gof[t] = (uint32_t)off[cell];
    key[t] = (unsigned short)k;
  }
  for (int t = threadIdx.x; t < BD * SZ; t += 256) acc[t] = 0;
  __syncthreads();
  block_scan(cnt, pre, nC, wsum);
  const int total = pre[nC];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int sh = M.sh, w = M.w;
  const float rsh = 1.0f / (float)(1u << sh);
  const uint32_t fmask = (1u << sh) - 1u, low = (uint32_t)(w - 2) << sh;  // a lower cell's last two layers
  unsigned long long* q = queue[wave];
  auto process = [&](int nq) {
    wave_sync_lds();
    if (lane < nq) {
      const unsigned long long e = q[lane];
      const int k = (int)(e >> 48);
      int f[3];
      float wt[3][3];
      bool ok[3][3];
      for (int d = 0; d < 3; ++d) {
        const uint32_t u = (uint32_t)(e >> (16 * d)) & 0xffffu;
        f[d] = w * (((k >> (3 * d)) & 7) - 1) + (int)(u >> sh);  // floor relative to BD b
        tsc_weights_frac<float>(((float)(u & fmask) + 0.5f) * rsh, wt[d]);
        for (int i = 0; i < 3; ++i) ok[d][i] = (unsigned)(f[d] + i) < (unsigned)BD;
      }
      for (int i = 0; i < 3; ++i) wt[2][i] *= kFixF;  // exact: a power of two
      unsigned long long* a = acc + (f[2] * SZ + f[1] * SY + f[0]);
#pragma unroll
      for (int i3 = 0; i3 < 3; ++i3)
#pragma unroll
        for (int i2 = 0; i2 < 3; ++i2)
#pragma unroll
          for (int i1 = 0; i1 < 3; ++i1)
            if (ok[2][i3] && ok[1][i2] && ok[0][i1])
              atomicAdd(&a[i3 * SZ + i2 * SY + i1],
                        (unsigned long long)__float2uint_rn((wt[0][i1] * wt[1][i2]) * wt[2][i3]));
    }
    wave_sync_lds();
  };
  const int seg = wave * 8 + (lane & 7);
  const int i1 = (int)((int64_t)total * (seg + 1) / NS);
  int i = (int)((int64_t)total * seg / NS) + (lane >> 3);
  int c = i < i1 ? find_cell(pre, nC, i) : 0;
  int qn = 0;
  constexpr int U = 4;
  while (__any(i < i1)) {
    uint32_t u[U][3];
    int kc[U];
    bool val[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      val[k] = i < i1;
      kc[k] = 0;
      u[k][0] = u[k][1] = u[k][2] = 0;
      if (val[k]) {
        while (i >= pre[c + 1]) ++c;
        kc[k] = key[c];
        load_xp<IZ>(xp, (int64_t)gof[c] + (i - pre[c]), u[k]);
      }
      i += 8;
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const bool hit = val[k] && u[k][0] >= ((kc[k] & 512) ? low : 0u) && u[k][1] >= ((kc[k] & 1024) ? low : 0u) &&
                       u[k][2] >= ((kc[k] & 2048) ? low : 0u);
      const unsigned long long m = __ballot(hit);
      if (hit)
        q[qn + (int)__popcll(m & ((1ull << lane) - 1ull))] =
            ((unsigned long long)kc[k] << 48) | ((unsigned long long)u[k][2] << 32) |
            (unsigned long long)((u[k][1] << 16) | u[k][0]);
      qn += (int)__popcll(m);
      if (qn >= 64) {
        process(64);
        const unsigned long long mv = (lane < qn - 64) ? q[64 + lane] : 0ull;
        wave_sync_lds();
        if (lane < qn - 64) q[lane] = mv;
        qn -= 64;
      }
    }
  }
  if (qn > 0) process(qn);
  __syncthreads();
  for (int t = threadIdx.x; t < BD * BD * BD; t += 256) {
    const int l[3] = {t % BD, (t / BD) % BD, t / (BD * BD)};
    const unsigned long long v = acc[l[2] * SZ + l[1] * SY + l[0]];
    int a[3];
    for (int d = 0; d < 3; ++d) {
      a[d] = bi[d] * BD - 1 + l[d];
      a[d] = a[d] < 0 ? a[d] + M.n : a[d];
    }
    mesh[((int64_t)a[2] * M.n + a[1]) * M.n + a[0]] = (float)((double)v * (1.0 / (double)kFixF)) * mass;
  }
}

// Faces of the windows: face 2 axis + side of box b at faces[(6 b + face) n^2],
// [v][u] with u, v the lower and the higher of the other two axes.  One
// workgroup per strip of `rows` v-rows of a face sums the taps of the
// particles of the boundary layer of coarse cells whose floor is the face's
// layer (middle tap) or the next one inside (outer tap).  Cells' counts and starts
// come to LDS at once, each wavefront reads its quarter of the list four
// particles a lane at a time, and the quarter to half that lie in the two layers
// queue to be deposited 64 at a time, as in k_mesh_deposit.  4096 windows of 80^3
// and 64 of 160^3 1.5 ms, 4096 of 40^3 0.22 (2.25 and 0.36 with a cell per
// wavefront, its count, start and particles read in turn, and a quarter of the
// lanes at work).
template <int IZ>
__global__ void __launch_bounds__(256) k_mesh_faces(MeshGeo M, PMLevel L, const PMBox* __restrict__ boxes, int rows,
                                                    int maxc, const XT<IZ>* __restrict__ xp,
                                                    const int32_t* __restrict__ rhoc, const int64_t* __restrict__ off,
                                                    float* __restrict__ faces, float mass) {
  extern __shared__ unsigned long long facc[];  // [rows][n], then the cell tables
  __shared__ unsigned long long queue[4][128];
  __shared__ int wsum[4];
  const int n = L.n, nr = n / M.w, nstrip = (n + rows - 1) / rows;
  int* cnt = reinterpret_cast<int*>(facc + rows * n);
  int* pre = cnt + maxc;
  uint32_t* gof = reinterpret_cast<uint32_t*>(pre + maxc + 1);  // (the caller holds np < 2^32)
  unsigned short* key = reinterpret_cast<unsigned short*>(gof + maxc);
  const int strip = (int)(blockIdx.x % (unsigned)nstrip), face = (int)((blockIdx.x / (unsigned)nstrip) % 6);
  const int64_t box = blockIdx.x / ((unsigned)nstrip * 6);
  const int ax = face >> 1, side = face & 1, au = ax == 0 ? 1 : 0, av = ax == 2 ? 1 : 2;
  const PMBox B = boxes[box];
  const int v0 = strip * rows, v1 = min(n, v0 + rows);  // rows [v0, v1)
  const int sh = M.sh, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // coarse cells (window-local 0..nr-1) that reach the strip: floors v0-1 .. v1
  const int cv0 = max(0, v0 - 1) / M.w, cv1 = min(n - 1, v1) / M.w;
  const int ncell = nr * (cv1 - cv0 + 1);
  const int cax = side ? nr - 1 : 0;
  for (int t = threadIdx.x; t < ncell; t += 256) {
    const int cu = t % nr, cv = cv0 + t / nr;
    const int c0 = ax == 0 ? cax : cu, c1 = ax == 1 ? cax : (ax == 0 ? cu : cv), c2 = ax == 2 ? cax : cv;
    const int64_t cell = rc_index(B.nc1[0] - L.nloop + c0, B.nc1[1] - L.nloop + c1, B.nc1[2] - L.nloop + c2, B.T,
                                  M.nte, M.ncb);
    cnt[t] = rhoc[cell];
    gof[t] = (uint32_t)off[cell];
    key[t] = (unsigned short)(cu | (cv << 8));
  }
  for (int t = threadIdx.x; t < (v1 - v0) * n; t += 256) facc[t] = 0;
  __syncthreads();
  block_scan(cnt, pre, ncell, wsum);
  const int total = pre[ncell];
  const float rsh = 1.0f / (float)(1u << sh);
  const uint32_t fmask = (1u << sh) - 1u;
  // the coordinate across the face of its two layers
  const uint32_t ulo = side ? (uint32_t)(M.w - 2) << sh : 0u, uhi = side ? ~0u : (2u << sh) - 1u;
  unsigned long long* q = queue[wave];
  auto process = [&](int nq) {
    wave_sync_lds();
    if (lane < nq) {
      const unsigned long long e = q[lane];
      const uint32_t ua = (uint32_t)e & 0xffffu, uu = (uint32_t)(e >> 16) & 0xffffu, uv = (uint32_t)(e >> 32) & 0xffffu;
      const int k = (int)(e >> 48);
      const int fa = M.w * cax + (int)(ua >> sh), in = side ? n - 1 - fa : fa;  // layers inside the face
      const int fu = M.w * (k & 255) + (int)(uu >> sh), fv = M.w * (k >> 8) + (int)(uv >> sh);
      float wa[3], wu[3], wv[3];
      tsc_weights_frac<float>(((float)(ua & fmask) + 0.5f) * rsh, wa);
      tsc_weights_frac<float>(((float)(uu & fmask) + 0.5f) * rsh, wu);
      tsc_weights_frac<float>(((float)(uv & fmask) + 0.5f) * rsh, wv);
      // the tap that falls on the face, with the 2^32 of the fixed point (exact)
      const float w1 = (in == 0 ? wa[1] : (side ? wa[2] : wa[0])) * kFixF;
#pragma unroll
      for (int jv = 0; jv < 3; ++jv) {
        const int mv = fv - 1 + jv;
        if (mv < v0 || mv >= v1) continue;
#pragma unroll
        for (int ju = 0; ju < 3; ++ju) {
          const int mu = fu - 1 + ju;
          if (mu < 0 || mu >= n) continue;
          // (wx wy) wz, as every deposit forms it
          const float cw = ax == 2 ? (wu[ju] * wv[jv]) * w1 : (w1 * wu[ju]) * wv[jv];
          atomicAdd(&facc[(mv - v0) * n + mu], (unsigned long long)__float2uint_rn(cw));
        }
      }
    }
    wave_sync_lds();
  };
  // each wavefront takes a quarter of the list, four particles a lane at a time
  const int i1 = (int)((int64_t)total * (wave + 1) / 4);
  int i = (int)((int64_t)total * wave / 4) + lane;
  int c = i < i1 ? find_cell(pre, ncell, i) : 0;
  int qn = 0;
  constexpr int U = 4;
  while (__any(i < i1)) {
    uint32_t u[U][3];
    int kc[U];
    bool val[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      val[k] = i < i1;
      kc[k] = 0;
      u[k][0] = u[k][1] = u[k][2] = 0;
      if (val[k]) {
        while (i >= pre[c + 1]) ++c;
        kc[k] = key[c];
        load_xp<IZ>(xp, (int64_t)gof[c] + (i - pre[c]), u[k]);
      }
      i += 64;
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const uint32_t ua = ax == 0 ? u[k][0] : (ax == 1 ? u[k][1] : u[k][2]);
      const uint32_t uu = au == 0 ? u[k][0] : u[k][1], uv = av == 1 ? u[k][1] : u[k][2];
      const bool hit = val[k] && ua >= ulo && ua <= uhi;
      const unsigned long long m = __ballot(hit);
      if (hit)
        q[qn + (int)__popcll(m & ((1ull << lane) - 1ull))] =
            ((unsigned long long)kc[k] << 48) | ((unsigned long long)uv << 32) | (unsigned long long)((uu << 16) | ua);
      qn += (int)__popcll(m);
      if (qn >= 64) {
        process(64);
        const unsigned long long mv = (lane < qn - 64) ? q[64 + lane] : 0ull;
        wave_sync_lds();
        if (lane < qn - 64) q[lane] = mv;
        qn -= 64;
      }
    }
  }
  if (qn > 0) process(qn);
  __syncthreads();
  float* out = faces + ((6 * box + face) * n + v0) * n;
  for (int t = threadIdx.x; t < (v1 - v0) * n; t += 256)
    out[t] = (float)((double)facc[t] * (1.0 / (double)kFixF)) * mass;
}

// The windows as cubes: one thread per four cells of a row (n is a multiple of
// w >= 4; a row starts at a multiple of w of the image mesh, so four cells
// never straddle its end), one workgroup row of the grid per z-plane.
__global__ void __launch_bounds__(256) k_mesh_window(MeshGeo M, int n, const int4* __restrict__ org,
                                                     const float* __restrict__ mesh, const float* __restrict__ faces,
                                                     float* __restrict__ out) {
  const int nq = n / 4, t = blockIdx.y * 256 + threadIdx.x;
  const int y = t / nq, x = (t - y * nq) * 4;
  if (y >= n) return;
  const int64_t box = blockIdx.x / (unsigned)n;
  const int z = (int)(blockIdx.x % (unsigned)n);
  const float* fb = faces + 6 * box * n * n;
  float4 v;
  if (z == 0 || z == n - 1) v = *(const float4*)(fb + ((int64_t)(z == 0 ? 4 : 5) * n + y) * n + x);
  else if (y == 0 || y == n - 1) v = *(const float4*)(fb + ((int64_t)(y == 0 ? 2 : 3) * n + z) * n + x);
  else {
    const int4 o = org[box];
    const int p[3] = {o.x + x, o.y + y, o.z + z};
    int a[3];
    for (int d = 0; d < 3; ++d) a[d] = p[d] >= M.n ? p[d] - M.n : p[d];
    v = *(const float4*)(mesh + ((int64_t)a[2] * M.n + a[1]) * M.n + a[0]);
    if (x == 0) v.x = fb[(int64_t)z * n + y];
    if (x == n - 4) v.w = fb[((int64_t)n + z) * n + y];
  }
  *(float4*)(out + ((box * n + z) * n + y) * n + x) = v;
}

// Buffer cells as periodic images of the physical ones (counts and encoded
// coordinates, particle by particle): one wavefront per extended cell.
template <int IZ>
__global__ void __launch_bounds__(256) k_mesh_images(Geo g, const XT<IZ>* __restrict__ xp,
                                                     const int32_t* __restrict__ rhoc,
                                                     const int64_t* __restrict__ off, int32_t* __restrict__ bad) {
  const int64_t c = ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (c >= g.ncells_ext) return;
  const int64_t T = c / g.ncell_tile, e = c % g.ncell_tile;
  const int64_t it[3] = {T % g.nnt, (T / g.nnt) % g.nnt, T / (g.nnt * g.nnt)};
  const int64_t ijk[3] = {e % g.nte + 1 - g.ncb, (e / g.nte) % g.nte + 1 - g.ncb, e / (g.nte * g.nte) + 1 - g.ncb};
  int64_t st[3], sc[3];
  bool phys = true;
  for (int d = 0; d < 3; ++d) {
    phys = phys && ijk[d] >= 1 && ijk[d] <= g.nt;
    int64_t gc = (it[d] * g.nt + ijk[d] - 1) % g.nc;
    gc = gc < 0 ? gc + g.nc : gc;
    st[d] = gc / g.nt;
    sc[d] = gc % g.nt + 1;
  }
  if (phys) return;
  const int64_t src = rc_index(sc[0], sc[1], sc[2], (st[2] * g.nnt + st[1]) * g.nnt + st[0], g.nte, g.ncb);
  const int n = rhoc[c];
  bool diff = n != rhoc[src];
  if (!diff)
    for (int l = lane; l < 3 * n; l += 64) diff = diff || xp[3 * off[c] + l] != xp[3 * off[src] + l];
  if (__any(diff) && lane == 0) *bad = 1;
}

}  // namespace

MeshGeo mesh_geo(const Geo& g, int w, int bits) {
  MeshGeo M;
  M.w = w;
  M.n = (int)g.nc * w;
  M.sh = bits - (31 - __builtin_clz((unsigned)w));
  M.nc = (int)g.nc;
  M.nt = (int)g.nt;
  M.nnt = (int)g.nnt;
  M.nte = (int)g.nte;
  M.ncb = (int)g.ncb;
  return M;
}

bool pm_mesh_applies(const Geo& g, const PMLevel& L) {
  return !L.periodic && !L.xdiv && (L.w == 4 || L.w == 8) && L.nforce % L.w == 0 && L.win_lo == 1 - L.nloop * L.w &&
         L.win_hi == L.nforce + L.nloop * L.w && L.n == L.nforce + 2 * L.nloop * L.w && (g.nc * L.w) % 8 == 0 && L.n <= g.nc * L.w &&
         L.nloop <= g.ncb && L.n / L.w <= 256;  // (cell tables of a face's strip: 8 bits an axis, 1024 cells)
}

void pm_mesh_deposit(int izipx, const MeshGeo& M, const void* xp, const int32_t* rhoc, const int64_t* off,
                     float* mesh, float mass, hipStream_t s) {
  // 16^3 blocks have half the repeated contributors of 8^3 ones, but fill the chip only from 2048 of them
  const int bd = M.n % 16 == 0 && (int64_t)M.n * M.n * M.n / 4096 >= 2048 ? 16 : 8;
  const int64_t nb = M.n / bd;
  const dim3 grid((unsigned)(nb * nb * nb));
  if (izipx == 2 && bd == 16)
    hipLaunchKernelGGL((k_mesh_deposit<2, 16>), grid, dim3(256), 0, s, M, (const int16_t*)xp, rhoc, off, mesh, mass);
  else if (izipx == 2)
    hipLaunchKernelGGL((k_mesh_deposit<2, 8>), grid, dim3(256), 0, s, M, (const int16_t*)xp, rhoc, off, mesh, mass);
  else if (bd == 16)
    hipLaunchKernelGGL((k_mesh_deposit<1, 16>), grid, dim3(256), 0, s, M, (const int8_t*)xp, rhoc, off, mesh, mass);
  else
    hipLaunchKernelGGL((k_mesh_deposit<1, 8>), grid, dim3(256), 0, s, M, (const int8_t*)xp, rhoc, off, mesh, mass);
  CUBE_HIP(hipGetLastError());
}

void pm_mesh_faces(int izipx, const MeshGeo& M, const PMLevel& L, const PMBox* boxes, int nbox, const void* xp,
                   const int32_t* rhoc, const int64_t* off, float* faces, float mass, hipStream_t s) {
  // strips of at most 32 KB
  const int rows = std::min(L.n, std::max(1, 32768 / (8 * L.n)));
  const int nstrip = (L.n + rows - 1) / rows;
  const int nr = L.n / M.w, maxc = nr * std::min(nr, (rows + 1) / M.w + 2);  // cells that reach a strip
  const size_t lds = (size_t)rows * L.n * 8 + (size_t)maxc * 14 + 8;
  const dim3 grid((unsigned)((int64_t)nbox * 6 * nstrip));
  if (izipx == 2)
    hipLaunchKernelGGL(k_mesh_faces<2>, grid, dim3(256), lds, s, M, L, boxes, rows, maxc, (const int16_t*)xp, rhoc, off,
                       faces, mass);
  else
    hipLaunchKernelGGL(k_mesh_faces<1>, grid, dim3(256), lds, s, M, L, boxes, rows, maxc, (const int8_t*)xp, rhoc, off,
                       faces, mass);
  CUBE_HIP(hipGetLastError());
}

int4 mesh_origin(const MeshGeo& M, const PMLevel& L, const PMBox& B) {
  const int it[3] = {B.T % M.nnt, (B.T / M.nnt) % M.nnt, B.T / (M.nnt * M.nnt)};
  int a[3];
  for (int d = 0; d < 3; ++d) a[d] = (((it[d] * M.nt + B.nc1[d] - 1 - L.nloop) * M.w) % M.n + M.n) % M.n;
  return make_int4(a[0], a[1], a[2], 0);
}

void pm_mesh_window(const MeshGeo& M, int n, const int4* org, int nbox, const float* mesh, const float* faces,
                    float* out, hipStream_t s) {
  hipLaunchKernelGGL(k_mesh_window, dim3((unsigned)(nbox * n), (unsigned)ceil_div(n * (n / 4), 256)), dim3(256), 0, s,
                     M, n, org, mesh, faces, out);
  CUBE_HIP(hipGetLastError());
}

void mesh_check_images(int izipx, const Geo& g, const void* xp, const int32_t* rhoc, const int64_t* off, int32_t* bad,
                       hipStream_t s) {
  zero_async(bad, sizeof(int32_t), s);
  const Blocks b = blocks_xy(ceil_div(g.ncells_ext, 4));
  const dim3 grid(b.x, b.y);
  if (izipx == 2)
    hipLaunchKernelGGL(k_mesh_images<2>, grid, dim3(256), 0, s, g, (const int16_t*)xp, rhoc, off, bad);
  else
    hipLaunchKernelGGL(k_mesh_images<1>, grid, dim3(256), 0, s, g, (const int8_t*)xp, rhoc, off, bad);
  CUBE_HIP(hipGetLastError());
}

}  // namespace cube
