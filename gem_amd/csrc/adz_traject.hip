// Departure-point trajectories on gfx950: adz_set (tables), adz_prepareWinds,
// adz_traject and adz_interp_traj of GEM's gemdyn (src/gemdyn/src/base/).
//
// The fixed-point iteration of adz_traject.F90:66-107 is independent per arrival point
// (each point reads the static wind field at its own current position), so one lane owns
// one arrival point for all iterations and keeps the iterate in registers; only the final
// iterate is stored.  The storage type S of the derived winds and positions is the
// reference's `real` (S = float, bit-exact with its trajectories) or FP64 (S = double).
// Arithmetic is FP64 everywhere, evaluated in the source's left-to-right order with no FMA
// contraction (built with -ffp-contract=off).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "adz_common.h"
#include "adz_qv.h"
#include "adz_tile.h"

using namespace adz;

namespace adz {

// Scalars and device tables a trajectory kernel needs (by value).
struct TrajParams {
  int ni, nj, nk, i0g, j0g;
  int lminx, lminy, nit, njt, nij;
  int i0, in, j0, jn, i0u, inu, j0v, jnv, i0b, inb, j0b, jnb, k0, k0t, k0m;
  int k00;   // first level of the iteration, adz_traject.F90:63-64
  int k00i;  // first level of the pb set, adz_interp_traj.F90:38-39
  double iminposx, imaxposx, iminposy, imaxposy;
  double sig, ovdzm, ovdzt, zmin, zmax, vw5, vw6, inv_hx, inv_hy, inv_rayt;
  double ww_star, wp_nk, wm_nk;  // Ver_wmstar_8(nk), wp, wm of adz_interp_traj.F90:42-44
  int pnz_m, pnz_t;
  const double* zm;      // 0..nk+1
  const double* zt;      // 0..nk+1
  const double* odelz_m; // 0..nk
  const double* odelz_t;
  const int* search_m;
  const int* search_t;
  const double* cy;      // index j - lminy
  const double* vw;      // 8 rows of nk+1: vw1m vw2m vw3m vw4m vw1t vw2t vw3t vw4t
};

__device__ __forceinline__ int d_level_search(const double* z, const int* tab, int pnz, double ovdz, double sig, int nk,
                                              double pos) {
  // adz_traject.F90:85-89; the two clamps on table indices never bind for positions
  // inside [zmin, zmax] and only keep a corrupted input from reading out of bounds
  int kk1 = (int)((pos - z[0]) * ovdz + 1.0);
  kk1 = min(max(1, kk1), pnz);
  kk1 = tab[kk1 - 1];
  if (sig * pos > sig * z[min(kk1 + 1, nk + 1)]) kk1 = kk1 + 1;
  if (sig * pos < sig * z[min(max(kk1, 0), nk + 1)]) kk1 = kk1 - 1;
  return kk1;
}

// zindx, adz_interp_traj.F90:189-204
__device__ __forceinline__ double d_zindx(const TrajParams& P, double posz) {
  posz = fmin(fmax(posz, P.zmin), P.zmax);
  int kk1 = d_level_search(P.zt, P.search_t, P.pnz_t, P.ovdzt, P.sig, P.nk, posz);
  kk1 = min(P.nk + 1, max(0, kk1));
  int nb = max(min(kk1, P.nk - 1), 1);
  return (posz - P.zt[nb]) * P.odelz_t[nb] + (double)nb;
}

__device__ __forceinline__ double clampd(double v, double lo, double hi) { return fmin(fmax(v, lo), hi); }

__device__ __forceinline__ long ext_idx(const TrajParams& P, int i, int j, int k) {
  return (long)(i - P.lminx) + (long)P.nit * ((j - P.lminy) + (long)P.njt * (k - 1));
}
__device__ __forceinline__ long wp_idx(const TrajParams& P, int i, int j, int k, int c) {
  return (long)(i + 1) + (long)(P.ni + 4) * ((j + 1) + (long)(P.nj + 4) * ((k - 1) + (long)P.nk * (c - 1)));
}
__device__ __forceinline__ long p3_idx(const TrajParams& P, int i, int j, int k) {  // (3, ni, nj, k0m:nk)
  return 3 * ((long)(i - 1) + (long)P.ni * ((j - 1) + (long)P.nj * (k - P.k0m)));
}
__device__ __forceinline__ long box_idx(int i0, int in, int j0, int jn, int k0, int i, int j, int k) {
  return 3 * ((long)(i - i0) + (long)(in - i0 + 1) * ((j - j0) + (long)(jn - j0 + 1) * (k - k0)));
}

// ---------------------------------------------------------------- adz_prepareWinds
// One level of the tile per row of the grid (no division by a level's points).
constexpr int kMaxGridY = 65535;

// adz_prepareWinds.F90:37-47 and :62-101 on the extended domain.
template <class S>
__global__ void k_prep_uvwd(S* __restrict__ uvw_d, const float* __restrict__ uu, const float* __restrict__ vv,
                            const float* __restrict__ ww, TrajParams P) {
  const unsigned h = blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= (unsigned)P.nij) return;
  const int j = (int)(h / (unsigned)P.nit) + P.lminy;
  for (int k = (int)blockIdx.y + 1; k <= P.nk; k += (int)gridDim.y) {
    const long q = h + (long)P.nij * (k - 1);
    const double ir = P.inv_rayt;
    uvw_d[3 * q + 0] = (S)(ir * (double)uu[q] * P.cy[j - P.lminy]);
    uvw_d[3 * q + 1] = (S)(ir * (double)vv[q]);
    double w;
    const int nk = P.nk;
    if (k == 1) w = P.vw5 * (double)ww[q];
    else if (k == nk) w = P.vw6 * (double)ww[q - P.nij];
    else {
      const double* vw = P.vw;
      double wx = (k >= 3) ? vw[k] : 0.0;
      int km2 = max(1, k - 2);
      long base = q - (long)(k - 1) * P.nij;
      w = wx * (double)ww[base + (long)(km2 - 1) * P.nij] + vw[(nk + 1) + k] * (double)ww[q - P.nij] +
          vw[2 * (nk + 1) + k] * (double)ww[q] + vw[3 * (nk + 1) + k] * (double)ww[q + P.nij];
    }
    uvw_d[3 * q + 2] = (S)w;
  }
}

// adz_prepareWinds.F90:48-61 and :69-86 on the interior: arrival winds.
template <class S>
__global__ void k_prep_arr(S* __restrict__ uarr, S* __restrict__ varr, S* __restrict__ warr,
                           const float* __restrict__ ut0, const float* __restrict__ vt0, const float* __restrict__ zdt0,
                           TrajParams P) {
  const unsigned h = blockIdx.x * blockDim.x + threadIdx.x, nxy = (unsigned)P.ni * (unsigned)P.nj;
  if (h >= nxy) return;
  const unsigned jq = h / (unsigned)P.ni;
  const int j = (int)jq + 1, i = (int)(h - jq * (unsigned)P.ni) + 1;
  for (int k = (int)blockIdx.y + 1; k <= P.nk; k += (int)gridDim.y) {
    const long a = h + (long)nxy * (k - 1);
    const double alpha1 = -1.0 / 16.0, alpha2 = 9.0 / 16.0, ir = P.inv_rayt;
    S u1 = (S)ut0[ext_idx(P, i - 2, j, k)] + (S)ut0[ext_idx(P, i + 1, j, k)];
    S u2 = (S)ut0[ext_idx(P, i, j, k)] + (S)ut0[ext_idx(P, i - 1, j, k)];
    uarr[a] = (S)((((double)u1 * alpha1 + (double)u2 * alpha2) * ir) * P.cy[j - P.lminy]);
    S v1 = (S)vt0[ext_idx(P, i, j - 2, k)] + (S)vt0[ext_idx(P, i, j + 1, k)];
    S v2 = (S)vt0[ext_idx(P, i, j, k)] + (S)vt0[ext_idx(P, i, j - 1, k)];
    varr[a] = (S)(((double)v1 * alpha1 + (double)v2 * alpha2) * ir);
    const int nk = P.nk;
    double w;
    if (k == 1) w = P.vw5 * (double)zdt0[ext_idx(P, i, j, 1)];
    else if (k == nk) w = P.vw6 * (double)zdt0[ext_idx(P, i, j, nk - 1)];
    else {
      const double* vw = P.vw;
      double wx = (k >= 3) ? vw[k] : 0.0;
      int km2 = max(1, k - 2);
      w = wx * (double)zdt0[ext_idx(P, i, j, km2)] + vw[(nk + 1) + k] * (double)zdt0[ext_idx(P, i, j, k - 1)] +
          vw[2 * (nk + 1) + k] * (double)zdt0[ext_idx(P, i, j, k)] +
          vw[3 * (nk + 1) + k] * (double)zdt0[ext_idx(P, i, j, k + 1)];
    }
    warr[a] = (S)w;
  }
}

// ---------------------------------------------------------------- adz_traject
// adz_traject.F90:66-104: niter fixed-point updates of one arrival point (i,j,k) per lane.
//
// A block takes a tile of tw x tr points, at most 256, on kTrajLevels levels (four waves per
// level; 64 x 4 on wide grids, see traj_tile) and copies the box of the derived winds (three
// interleaved components) that its points read into LDS; every iteration reduces the box it needs
// over the block and stages a new one only where that leaves the one in LDS, which has a margin of
// one element on every side where that fits.  The stencil of a point is 192 values, of which the lanes of a tile read few that
// differ; as per-lane loads they were 48 16-byte loads per lane and iteration.
// Rows of the box begin kWindPitch elements apart (a row is one 1 KB DMA instruction of a
// wave, two in FP64): lanes are three words apart, free of bank conflicts, and rows a multiple
// of the banks.  A tile whose box does not fit reads per lane, in the same arithmetic and order.
// FLAT (tw = 0): blocks of 256 points in the order of the arrays, which fill their lanes in rows
// of any length, and every lane reads for itself.
//
// What bounds it: FP64 arithmetic.  1024 x 512 x 84 points, three iterations: 4.5 ms as
// per-lane loads with 70 % of the cycles issuing vector instructions (880 per iteration, 192
// of them selects and copies for the first row's missing sum, 192 conversions); 3.6 ms now
// (780 of them, 76 %), where 2.3 ms would be arithmetic alone.  Held to 128 registers, without
// spills (which cost more than the boxes gain), for two blocks per CU; in FP64 one block fits.
constexpr int kTrajLevels = 2, kTrajWaves = 4 * kTrajLevels, kTrajRows = 78;
constexpr int kWindPitch = 256;  // elements

// tricub3_ref (its operations and their order): columns 0 and 1 of the stencil, then 2 and 3,
// and of each a row of a plane (6 values) at a time with the next one on its way; read(h, r, z,
// v) gives the values of columns 2h and 2h + 1, row r, plane z.  More values at a time would
// cost the registers that keep four waves on a SIMD.
template <class S, class Read>
__device__ __forceinline__ void tricub3_steps(Read read, const double* c, double* out) {
  S v[2][6];
  double dst[6], za[6];
  auto load = [&](int q) { read(q / 16, q / 4 % 4, q % 4, v[q & 1]); };
  load(0);
#pragma unroll
  for (int q = 0; q < 32; q++) {
    if (q < 31) load(q + 1);
#pragma unroll
    for (int e = 0; e < 6; e++) {
      const double x = to_f64(v[q & 1][e]);
      za[e] = q % 4 == 0 ? x * c[8] : fma(x, c[8 + q % 4], za[e]);
    }
    // the sums are formed here, and the values of step q + 2 are not read before
    asm volatile("" : "+v"(za[0]), "+v"(za[1]), "+v"(za[2]), "+v"(za[3]), "+v"(za[4]), "+v"(za[5]) : : "memory");
    if (q % 4 == 3) {
      const int r = q / 4 % 4;
#pragma unroll
      for (int e = 0; e < 6; e++) dst[e] = r == 0 ? za[e] * c[4] : fma(za[e], c[4 + r], dst[e]);
      asm volatile("" : "+v"(dst[0]), "+v"(dst[1]), "+v"(dst[2]), "+v"(dst[3]), "+v"(dst[4]), "+v"(dst[5]));
    }
    if (q % 16 == 15) {
#pragma unroll
      for (int e = 0; e < 3; e++)
        out[e] = q == 15 ? fma(dst[e + 3], c[1], dst[e] * c[0]) : fma(dst[e + 3], c[3], fma(dst[e], c[2], out[e]));
    }
  }
}

template <class S, bool FLAT>
__global__ __launch_bounds__(FLAT ? 256 : 64 * kTrajWaves, FLAT ? 1 : sizeof(S) == 4 ? 4 : 2) void k_traject(
    S* __restrict__ pxyzm, double* __restrict__ wpxyz, S* __restrict__ uvw_dep, S* __restrict__ pm,
    const S* __restrict__ uvw_d, const S* __restrict__ uarr, const S* __restrict__ varr, const S* __restrict__ warr, ZtabDev lv, TrajParams P,
    int niter, double dtA, double dtD, double dtzA, double dtzD, unsigned tw, unsigned tr) {
  __shared__ __attribute__((aligned(16))) S box[FLAT ? 4 : kTrajRows * kWindPitch];
  __shared__ int red[18], moved[3];
  const unsigned lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int i, j, k;
  bool valid;
  if constexpr (FLAT) {
    const unsigned a = blockIdx.x * 256 + threadIdx.x, nxy = (unsigned)P.ni * (unsigned)P.nj;
    const unsigned kq = a / nxy, rem = a - kq * nxy, jq = rem / (unsigned)P.ni;
    i = (int)(rem - jq * (unsigned)P.ni) + 1; j = (int)jq + 1; k = (int)kq + P.k00;
    valid = k <= P.nk;
  } else {
    if (threadIdx.x < 18) red[threadIdx.x] = kFar;
    if (threadIdx.x < 3) moved[threadIdx.x] = 0;
    __syncthreads();
    const unsigned nbi = (P.ni + tw - 1) / tw, nbj = (P.nj + tr - 1) / tr;
    const unsigned nbk = (P.nk - P.k00 + kTrajLevels) / kTrajLevels;
    const long ntiles = (long)nbi * nbj * nbk, t = tile_of_block(ntiles, 1);
    if (t >= ntiles) return;  // the whole block leaves: no barrier is reached
    const unsigned tk = (unsigned)(t / ((long)nbi * nbj)), tij = (unsigned)(t - (long)tk * nbi * nbj);
    const unsigned tj = tij / nbi, ti = tij - tj * nbi;
    const unsigned l = threadIdx.x & 255, lj = l / tw, li = l - lj * tw;
    i = (int)(tw * ti + li) + 1; j = (int)(tr * tj + lj) + 1; k = (int)(kTrajLevels * tk + wv / 4) + P.k00;
    valid = lj < tr && i <= P.ni && j <= P.nj && k <= P.nk;
  }
  S px = (S)0, py = (S)0, pz = (S)0;
  S ua = (S)0, va = (S)0, wa = (S)0;
  if (valid) {
    const long p = p3_idx(P, i, j, k);
    const long aw = (long)(i - 1) + (long)P.ni * ((j - 1) + (long)P.nj * (k - 1));
    px = pxyzm[p]; py = pxyzm[p + 1]; pz = pxyzm[p + 2];
    ua = uarr[aw]; va = varr[aw]; wa = warr[aw];
  }
  const S* f3 = uvw_d + 3L * ((long)(1 - P.lminx) + (long)P.nit * (1 - P.lminy));
  // box in LDS: local columns [bx0, bx1], rows [by0, by1], planes [bz0, bz1]; empty at first
  unsigned boxes = 0;
  int bx0 = kFar, bx1 = -kFar, by0 = kFar, by1 = -kFar, bz0 = kFar, bz1 = -kFar;
  for (int it = 0; it < niter; it++) {
    Index x;
    const bool ok = valid && index_step((double)px, (double)py, (double)pz, lv, &x);
    const int pz1 = x.pz + (x.zlinear ? 1 : 3);
    bool staged = !FLAT;
    if constexpr (!FLAT) {
      const bool out = ok && (x.ix - 1 < bx0 || x.ix + 2 > bx1 || x.iy - 1 < by0 || x.iy + 2 > by1 || x.pz < bz0 || pz1 > bz1);
      // does any lane of the block need a new box?  (Word it % 3 tells; the barrier also says
      // that every wave is done with the old one.)
      if (__ballot(out) != 0 && lane == 0) moved[it % 3] = 1;
      if (threadIdx.x == 0) moved[(it + 1) % 3] = 0;
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(moved[it % 3])) {
        int ext[6] = {ok ? x.ix - 1 : kFar, ok ? -(x.ix + 2) : kFar, ok ? x.iy - 1 : kFar, ok ? -(x.iy + 2) : kFar,
                      ok ? x.pz : kFar, ok ? -pz1 : kFar};
        tile_min6(ext, red, boxes++);
        const int x0 = ext[0], x1 = -ext[1], y0 = ext[2], y1 = -ext[3], z0 = ext[4], z1 = -ext[5];
        const int mx0 = max(x0 - 1, lv.ilo), mx1 = min(x1 + 1, lv.ihi), my0 = max(y0 - 1, lv.jlo),
                  my1 = min(y1 + 1, lv.jhi), mz0 = max(z0 - 1, 0), mz1 = min(z1 + 1, lv.nk - 1);
        const int cols = kWindPitch / 3;
        const bool roomy = (my1 - my0 + 1) * (mz1 - mz0 + 1) <= kTrajRows && mx1 - mx0 + 1 <= cols;
        if (roomy) { bx0 = mx0; bx1 = mx1; by0 = my0; by1 = my1; bz0 = mz0; bz1 = mz1; }
        else { bx0 = x0; bx1 = x1; by0 = y0; by1 = y1; bz0 = z0; bz1 = z1; }
        const int nyb = by1 - by0 + 1, nzb = bz1 - bz0 + 1;
        const long n3 = 3L * lv.ni * (long)sizeof(S), nij3 = 3L * lv.nij * (long)sizeof(S);  // bytes of a row, of a plane
        staged = bx1 - bx0 < cols && (long)nyb * nzb <= kTrajRows && n3 * nyb + nij3 * nzb < 0x7fff0000L;
        if (staged) {
          const char* b0 = (const char*)(f3 + 3 * ((bx0 - 1) + (long)(by0 - 1) * lv.ni + (long)bz0 * lv.nij));
          const long left = (const char*)(uvw_d + 3L * P.nij * P.nk) + 16 - b0;  // (the array ends in 16 spare bytes)
          const __amdgpu_buffer_rsrc_t rs = field_rsrc(b0, (unsigned)min(left, 0x7fff0000L));
          const int quads = (3 * (bx1 - bx0 + 1) * (int)sizeof(S) + 15) / 16;
          constexpr int kI = kWindPitch * (int)sizeof(S) / 1024;  // DMA instructions per row
          for (int r = wv; r < nyb * nzb; r += kTrajWaves) {
            const int zz = r / nyb, yy = r - zz * nyb;
            const int off = yy * (int)n3 + zz * (int)nij3;
  #pragma unroll
            for (int h = 0; h < kI; h++) {
              const int q = 64 * h + (int)lane;
              __builtin_amdgcn_raw_ptr_buffer_load_lds(
                  rs, (__attribute__((address_space(3))) void*)(box + r * kWindPitch + h * (1024 / (int)sizeof(S))), 16,
                  q < quads ? off + 16 * q : 0x7fff0000, 0, 0, 0);
            }
          }
          __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
          __syncthreads();
        } else {
          bx0 = kFar;  // nothing in LDS
        }
      }
    }
    double w3[3] = {__builtin_nan(""), __builtin_nan(""), __builtin_nan("")};
    if (ok) {
      double c[20];
      weights_ref(x, lv, c);
      if constexpr (FLAT) {
        tricub3_ref<S>(f3 + 3 * x.off, c, 3L * lv.ni, 3L * lv.nij, x.zlinear, w3);
      } else if (staged) {
        const int nyb = by1 - by0 + 1;
        const int b = ((x.iy - 1 - by0) + nyb * (x.pz - bz0)) * kWindPitch + 3 * (x.ix - 1 - bx0);
        const int o1 = x.zlinear ? 0 : nyb * kWindPitch, o2 = o1 + nyb * kWindPitch, o3 = o2 + o1;
        tricub3_steps<S>([&](int h, int r, int z, S* v) {
          int e = b + r * kWindPitch + (z == 0 ? 0 : z == 1 ? o1 : z == 2 ? o2 : o3);
          asm("" : "+v"(e));  // one address, the six values at immediate offsets
#pragma unroll
          for (int q = 0; q < 6; q++) v[q] = box[e + 6 * h + q];
        }, c, w3);
      } else {
        const long o1 = x.zlinear ? 0 : 3L * lv.nij, o2 = o1 + 3L * lv.nij, o3 = o2 + o1;
        tricub3_steps<S>([&](int h, int r, int z, S* v) {
          const S* s = f3 + 3 * x.off + 3L * r * lv.ni + (z == 0 ? 0 : z == 1 ? o1 : z == 2 ? o2 : o3) + 6 * h;
#pragma unroll
          for (int q = 0; q < 6; q++) v[q] = s[q];
        }, c, w3);
      }
    }
    if (valid) {
      // (opaque in the loop: what follows from them is formed here rather than held through it)
      int i1 = i, j1 = j;
      asm volatile("" : "+v"(i1), "+v"(j1), "+v"(ua), "+v"(va), "+v"(wa));
      const long p = p3_idx(P, i1, j1, k);
      const S ud = (S)w3[0], vd = (S)w3[1], wd = (S)w3[2];
      const double xm = (double)(i1 + P.i0g - 1) - (dtD * (double)ud + dtA * (double)ua) * P.inv_hx;
      const double ym = (double)(j1 + P.j0g - 1) - (dtD * (double)vd + dtA * (double)va) * P.inv_hy;
      double pos = P.zm[k] - dtzD * (double)wd - dtzA * (double)wa;
      double zmv = fmin(fmax(pos, P.zmin), P.zmax);
      int kk = d_level_search(P.zm, P.search_m, P.pnz_m, P.ovdzm, P.sig, P.nk, zmv);
      int kk1 = min(P.nk + 1, max(0, kk));
      int nb = max(min(kk1, P.nk - 1), 1);
      const double pzm = (zmv - P.zm[nb]) * P.odelz_m[nb] + (double)nb;
      px = (S)clampd(xm, P.iminposx, P.imaxposx);
      py = (S)clampd(ym, P.iminposy, P.imaxposy);
      pz = (S)pzm;
      if (it == niter - 1) {
        pxyzm[p] = px; pxyzm[p + 1] = py; pxyzm[p + 2] = pz;
        uvw_dep[p] = ud; uvw_dep[p + 1] = vd; uvw_dep[p + 2] = wd;
        if (i1 >= P.i0 && i1 <= P.in && j1 >= P.j0 && j1 <= P.jn && k >= P.k0) {  // Adz_pm, adz_traject.F90:112-116
          const long m = box_idx(P.i0, P.in, P.j0, P.jn, P.k0, i1, j1, k);
          pm[m] = px; pm[m + 1] = py; pm[m + 2] = pz;
        }
        wpxyz[wp_idx(P, i1, j1, k, 1)] = xm;
        wpxyz[wp_idx(P, i1, j1, k, 2)] = ym;
        wpxyz[wp_idx(P, i1, j1, k, 3)] = pzm;
      }
    }
  }
}

// adz_inittraj.F90:25-37
template <class S>
__global__ void k_inittraj(S* __restrict__ pxyzm, double* __restrict__ wpxyz, TrajParams P) {
  long a = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long nxy = (long)P.ni * P.nj;
  if (a >= nxy * (P.nk - P.k0m + 1)) return;
  int k = (int)(a / nxy) + P.k0m;
  int j = (int)((a % nxy) / P.ni) + 1;
  int i = (int)(a % P.ni) + 1;
  long p = p3_idx(P, i, j, k);
  pxyzm[p] = (S)(i + P.i0g - 1);
  pxyzm[p + 1] = (S)(j + P.j0g - 1);
  pxyzm[p + 2] = (S)k;
  wpxyz[wp_idx(P, i, j, k, 1)] = (double)pxyzm[p];
  wpxyz[wp_idx(P, i, j, k, 2)] = (double)pxyzm[p + 1];
  wpxyz[wp_idx(P, i, j, k, 3)] = (double)pxyzm[p + 2];
}

// ---------------------------------------------------------------- adz_interp_traj
// Positions of the u and v grids (Adz_pmu, Adz_pmv: adz_interp_traj.F90:45-78) and of the
// thermodynamic levels (Adz_pb: :80-174, and its part Adz_pt: :176-181) from the FP64 history
// W, in one pass over it.  A lane takes kc consecutive levels of one column, the four levels of
// the vertical stencil passing through its registers; a block's 64 columns by 4 rows (fewer columns
// by more rows where rows are short) share the horizontal stencils in the first-level cache.
//
// What bounds it: memory, 88 bytes of history, winds and positions per point at 2.8 TB/s, in
// nine streams.  1024 x 512 x 84: 1.22 ms in one kernel (1.26 with an eighth of the tiles per
// XCD; 4 or 16 levels per lane 1.24 and 1.35); as five (pmu, pmv, pb and the copies into pt
// and into pm, now stored by k_traject), each reading the history again, 1.91 ms.
template <class S>
__global__ __launch_bounds__(256) void k_sets(S* __restrict__ pmu, S* __restrict__ pmv, S* __restrict__ pb,
                                              S* __restrict__ pt, const double* __restrict__ W,
                                              const S* __restrict__ uvw_dep, const float* __restrict__ zdt0,
                                              TrajParams P, double dtzD, double dtzA, int kc, int ltw) {
  const unsigned tw = 1u << ltw, tr = 256u >> ltw;  // columns and rows of a tile
  const unsigned nbi = (P.ni + tw - 1) >> ltw, nbj = (P.nj + tr - 1) / tr, nbk = (P.nk + kc - 1) / kc;
  const long ntiles = (long)nbi * nbj * nbk, t = tile_of_block(ntiles, 0);
  if (t >= ntiles) return;
  const unsigned tk = (unsigned)(t / ((long)nbi * nbj)), tij = (unsigned)(t - (long)tk * nbi * nbj), tj = tij / nbi;
  const int i = (int)(tw * (tij - tj * nbi) + (threadIdx.x & (tw - 1))) + 1, j = (int)(tr * tj + (threadIdx.x >> ltw)) + 1;
  if (i > P.ni || j > P.nj) return;
  const int nk = P.nk, k1 = (int)tk * kc + 1, k2 = min(nk, k1 + kc - 1), kstart = max(P.k00i, 2);
  const bool onu = i >= P.i0u && i <= P.inu && j >= P.j0 && j <= P.jn;
  const bool onv = i >= P.i0 && i <= P.in && j >= P.j0v && j <= P.jnv;
  const bool onb = i >= P.i0b && i <= P.inb && j >= P.j0b && j <= P.jnb;
  const bool ont = i >= P.i0 && i <= P.in && j >= P.j0 && j <= P.jn;
  const double aa = -0.0625, bb = 0.5625, half = 0.5;
  const double* vw = P.vw;
  // x, y and vertical wind of levels k-1, k, k+1 and k+2 (levels outside [k0m, nk] are not used)
  double x[4], y[4], d[4];
  auto level = [&](int q, int k) {
    k = min(max(k, P.k0m), nk);
    x[q] = W[wp_idx(P, i, j, k, 1)];
    y[q] = W[wp_idx(P, i, j, k, 2)];
    d[q] = (double)uvw_dep[p3_idx(P, i, j, k) + 2];
  };
  level(1, k1 - 1); level(2, k1); level(3, k1 + 1);
  for (int k = k1; k <= k2; k++) {
#pragma unroll
    for (int q = 0; q < 3; q++) { x[q] = x[q + 1]; y[q] = y[q + 1]; d[q] = d[q + 1]; }
    level(3, k + 2);
    const double z0 = W[wp_idx(P, i, j, k, 3)];
    auto between = [&](double w0, int c, int di, int dj) {  // half a point back, along i or j
      const double wm1 = W[wp_idx(P, i - di, j - dj, k, c)], w1 = W[wp_idx(P, i + di, j + dj, k, c)];
      const double w2 = W[wp_idx(P, i + 2 * di, j + 2 * dj, k, c)];
      return aa * (wm1 + w2) + bb * (w0 + w1);
    };
    auto put = [&](S* out, long q, double r0, double r1, double r2) {
      out[q] = (S)clampd(r0, P.iminposx, P.imaxposx);
      out[q + 1] = (S)clampd(r1, P.iminposy, P.imaxposy);
      out[q + 2] = (S)clampd(r2, 0.0, (double)(nk + 1));
    };
    if (onu && k >= P.k0)
      put(pmu, box_idx(P.i0u, P.inu, P.j0, P.jn, P.k0, i, j, k), between(x[1], 1, 1, 0) - 0.5, between(y[1], 2, 1, 0),
          between(z0, 3, 1, 0));
    if (onv && k >= P.k0)
      put(pmv, box_idx(P.i0, P.in, P.j0v, P.jnv, P.k0, i, j, k), between(x[1], 1, 0, 1), between(y[1], 2, 0, 1) - 0.5,
          between(z0, 3, 0, 1));
    if (!onb || (k == 1 ? P.k00i != 1 : k < kstart)) continue;
    double xt, yt, zt;
    if (k >= 2 && k <= nk - 2) {
      double v1 = vw[4 * (nk + 1) + k], v2 = vw[5 * (nk + 1) + k], v3 = vw[6 * (nk + 1) + k], v4 = vw[7 * (nk + 1) + k];
      xt = v1 * x[0] + v2 * x[1] + v3 * x[2] + v4 * x[3];
      yt = v1 * y[0] + v2 * y[1] + v3 * y[2] + v4 * y[3];
      double wdt = v1 * d[0] + v2 * d[1] + v3 * d[2] + v4 * d[3];
      zt = P.zt[k] - dtzD * wdt - dtzA * (double)zdt0[ext_idx(P, i, j, k)];
    } else if (k < nk) {  // 1 and nk - 1
      xt = (x[1] + x[2]) * half;
      yt = (y[1] + y[2]) * half;
      double wdt = (d[1] + d[2]) * half;
      zt = P.zt[k] - dtzD * wdt - dtzA * (double)zdt0[ext_idx(P, i, j, k)];
    } else {
      xt = P.wp_nk * x[1] + P.wm_nk * x[0];
      yt = P.wp_nk * y[1] + P.wm_nk * y[0];
      double wdt = (d[0] + d[1]) * half;
      zt = P.zt[k] - P.ww_star * (dtzD * wdt + dtzA * (double)zdt0[ext_idx(P, i, j, k - 1)]);
    }
    const S sx = (S)clampd(xt, P.iminposx, P.imaxposx), sy = (S)clampd(yt, P.iminposy, P.imaxposy);
    const S sz = (S)d_zindx(P, zt);
    const long q = box_idx(P.i0b, P.inb, P.j0b, P.jnb, 1, i, j, k);
    pb[q] = sx; pb[q + 1] = sy; pb[q + 2] = sz;
    if (ont && k >= P.k0t) {
      const long m = box_idx(P.i0, P.in, P.j0, P.jn, P.k0t, i, j, k);
      pt[m] = sx; pt[m + 1] = sy; pt[m + 2] = sz;
    }
  }
}

}  // namespace adz

// ====================================================================== host side
struct adz_ctx {
  int pos_dtype, itraj, niter;
  TrajParams P;
  // host copies of the derived tables
  std::vector<double> zm, zt, zx, delz_m, delz_t, odelz_m, odelz_t, cy, vw;
  std::vector<int> search_m, search_t;
  adz_ztab* zq = nullptr;
  adz_ztab* zth = nullptr;
  void* tables = nullptr;  // device copy of the tables
  void* qvtab = nullptr;   // delz_t and the cubic / quintic denominators (BICHQV)
  void* amtab = nullptr;   // Ver_dz_8%t(k), Ver_idz_8%t(k), k = 0..nk (air mass)
  // device state
  void* uvw_d = nullptr; void* warr = nullptr; void* uvw_dep = nullptr; void* pxyzm = nullptr;
  double* wpxyz = nullptr;
  void* pm = nullptr; void* pmu = nullptr; void* pmv = nullptr; void* pt = nullptr; void* pb = nullptr;
  long n_uvw_d, n_arr, n_p3, n_wp, n_pm, n_pmu, n_pmv, n_pt, n_pb;
};

namespace {

// Level-search table: adz_set.F90:193-215 (REAL128 smallest_dz and bin starts as written)
void search_table(const std::vector<double>& z, const std::vector<double>& delz, int nk, double sig, double* ovdz,
                  std::vector<int>* tab) {
  __float128 smallest = (__float128)(sig * delz[1]);
  for (int k = 2; k <= nk; k++) {
    __float128 v = (__float128)(sig * delz[k]);
    if (v < smallest) smallest = v;
  }
  double o = (double)((__float128)1.0 / smallest);
  double pn = (double)1.0f + sig * (z[nk + 1] - z[0]) * o;
  int pnz = (int)std::lround(pn);
  *ovdz = (double)((__float128)sig / smallest);
  tab->assign(pnz, 0);
  int k0 = 0;
  for (int k = 1; k <= pnz; k++) {
    __float128 posz = (__float128)(sig * z[0]) + (__float128)(double)(k - 1) * smallest;
    if (posz > (__float128)(sig * z[k0 + 1])) k0 = std::min(nk + 1, k0 + 1);
    (*tab)[k - 1] = k0;
  }
}

double lag3(double zz, double z1, double z2, double z3, double z4) {
  return (((zz - z2) * (zz - z3) * (zz - z4)) / ((z1 - z2) * (z1 - z3) * (z1 - z4)));
}

unsigned nb(long n) { return (unsigned)((n + 255) / 256); }

void free_ctx(adz_ctx* c) {
  void* bufs[] = {c->tables, c->qvtab, c->amtab, c->uvw_d, c->warr, c->uvw_dep, c->pxyzm, c->wpxyz,
                  c->pm, c->pmu, c->pmv, c->pt, c->pb};
  for (void* b : bufs)
    if (b) (void)hipFree(b);
  if (c->zq) adz_vsearch_free(c->zq);
  if (c->zth) adz_vsearch_free(c->zth);
  delete c;
}

// Tile of k_traject: of the widths that split the rows into equal parts of 32 to 64 points, with
// as many rows as 256 lanes hold (at most 8, for the box), the one that leaves the fewest lanes
// without a point.  (65 x 103 x 49, cold: 109 us per lane, 176 with tiles of 64 x 4 and a
// whole tile for the last column, 112 with 33 x 7; 200 x 150 x 60, cold: 466 and 425.)
// Rows of fewer than kFlatRow points would leave a quarter of the lanes and more without one, and
// are taken flat.  The whole call, flat (in tiles), us: 8 x 800 x 60 115 (177), 16 x 800 x 60 159
// (192), 20 x 600 x 60 143 (158), 24 x 600 x 60 164 (161); in FP64 170 (241), 244 (258), 219 (238),
// 240 (243).
constexpr int kFlatRow = 24;
void traj_tile(int ni, int nj, unsigned* tw, unsigned* tr) {
  *tw = *tr = 0;
  if (ni < kFlatRow) return;
  long best = -1;
  for (int nt = (ni + 63) / 64; nt == (ni + 63) / 64 || (ni + nt - 1) / nt >= 32; nt++) {
    const int w = (ni + nt - 1) / nt, r = std::min(8, 256 / w);
    const long blocks = (long)((ni + w - 1) / w) * ((nj + r - 1) / r);
    if (best < 0 || blocks < best) { best = blocks; *tw = w; *tr = r; }
  }
}

template <class S>
int run_traject(adz_ctx* c, double dt, int advec, double bA_m, double bA, const float* uu, const float* vv,
                const float* ww, const float* ut0, const float* vt0, const float* zdt0, hipStream_t st) {
  TrajParams& P = c->P;
  double dtA = 0, dtzA = 0;
  if (advec == 1) { dtA = dt * 0.5; dtzA = dt * 0.5; }
  if (advec == 2) { dtA = dt * bA_m; dtzA = dt * bA; }
  if (advec == 3) { dtA = (1.0 - bA_m) * dt; dtzA = (1.0 - bA) * dt; }
  double dtD = dt - dtA, dtzD = dt - dtzA;
  if (advec == 0) dtA = dtD = dtzA = dtzD = 0.0;
  long nint = (long)P.ni * P.nj * P.nk;
  hipLaunchKernelGGL(k_prep_uvwd<S>, dim3(nb(P.nij), std::min(P.nk, kMaxGridY)), dim3(256), 0, st, (S*)c->uvw_d, uu, vv, ww, P);
  S* arr = (S*)c->warr;
  hipLaunchKernelGGL(k_prep_arr<S>, dim3(nb((long)P.ni * P.nj), std::min(P.nk, kMaxGridY)), dim3(256), 0, st, arr, arr + nint, arr + 2 * nint, ut0, vt0, zdt0, P);
  unsigned tw, tr;
  traj_tile(P.ni, P.nj, &tw, &tr);
  const long points = (long)P.ni * P.nj * (P.nk - P.k00 + 1);
  const long tiles =
      tw ? (long)((P.ni + tw - 1) / tw) * ((P.nj + tr - 1) / tr) * ((P.nk - P.k00 + kTrajLevels) / kTrajLevels) : 0;
  hipLaunchKernelGGL((tw ? k_traject<S, false> : k_traject<S, true>), tw ? tile_grid(tiles) : dim3(nb(points)),
                     dim3(tw ? 64 * kTrajWaves : 256), 0, st, (S*)c->pxyzm, c->wpxyz, (S*)c->uvw_dep, (S*)c->pm,
                     (const S*)c->uvw_d, arr, arr + nint, arr + 2 * nint, c->zq->dev, P, c->niter, dtA, dtD, dtzA, dtzD, tw,
                     tr);
  c->niter = c->itraj;  // adz_traject.F90:120
  // levels per lane: as many as leave eight waves for every SIMD, at most 8
  // columns of a tile of k_sets: 64; in rows of up to 32 points as many as there are, rounded up (the
  // call on 8 x 800 x 60 points 115 -> 80 us, 16 x 800 x 60 159 -> 138)
  int ltw = 6;
  while (ltw > 3 && P.ni <= (1 << (ltw - 1))) ltw--;
  const long cols = (long)((P.ni + (1 << ltw) - 1) >> ltw) * ((P.nj + (256 >> ltw) - 1) / (256 >> ltw));
  const int kc = (int)std::min(8L, std::max(1L, cols * 4 * P.nk / (8 * 1024)));
  hipLaunchKernelGGL(k_sets<S>, tile_grid(cols * ((P.nk + kc - 1) / kc)), dim3(256), 0, st, (S*)c->pmu, (S*)c->pmv,
                     (S*)c->pb, (S*)c->pt, c->wpxyz, (const S*)c->uvw_dep, zdt0, P, dtzD, dtzA, kc, ltw);
  ADZ_HIP_CHECK(hipGetLastError());
  return ADZ_OK;
}

}  // namespace

extern "C" {

int adz_set(const adz_grid* g, int pos_dtype, int itraj, adz_ctx** out) {
  if (!g || !out || !g->zm || !g->zt || !g->zx || !g->lat) return fail(ADZ_EINVAL, "adz_set: null argument");
  if (pos_dtype != ADZ_F32 && pos_dtype != ADZ_F64) return fail(ADZ_EINVAL, "adz_set: pos_dtype must be F32 or F64");
  if (g->nk < 4 || g->ni < 8 || g->nj < 8 || g->halox < 2 || g->haloy < 2 || itraj < 1)
    return fail(ADZ_EINVAL, "adz_set: need nk>=4, ni,nj>=8, halo>=2, itraj>=1");
  if ((long)g->ni * g->nj * (g->nk + 1) >= (1L << 31))
    return fail(ADZ_EINVAL, "adz_set: a tile of 2^31 points or more (split the domain)");
  adz_ctx* c = new adz_ctx();
  c->pos_dtype = pos_dtype; c->itraj = itraj; c->niter = itraj;
  TrajParams& P = c->P;
  std::memset(&P, 0, sizeof(P));
  const int ni = g->ni, nj = g->nj, nk = g->nk;
  P.ni = ni; P.nj = nj; P.nk = nk; P.i0g = g->i0g; P.j0g = g->j0g;
  // adz_set.F90:65-172
  int lmaxx = ni + g->halox, lmaxy = nj + g->haloy;
  P.lminx = 1 - g->halox; P.lminy = 1 - g->haloy;
  P.nit = lmaxx - P.lminx + 1; P.njt = lmaxy - P.lminy + 1; P.nij = P.nit * P.njt;
  const int ext = 1;
  int pil_w = g->west ? g->pil_w : 0, pil_e = g->east ? g->pil_e : 0;
  int pil_s = g->south ? g->pil_s : 0, pil_n = g->north ? g->pil_n : 0;
  P.i0 = 1 + pil_w - (ext + 1) * g->west; P.in = ni - pil_e + ext * g->east;
  P.j0 = 1 + pil_s - (ext + 1) * g->south; P.jn = nj - pil_n + ext * g->north;
  P.i0u = 1 + pil_w; P.j0v = 1 + pil_s; P.inu = g->niu - pil_e; P.jnv = g->njv - pil_n;
  P.k0 = g->gbpil_t + 1; P.k0t = std::max(1, g->gbpil_t); P.k0m = std::max(P.k0t - 2, 1);
  if (g->bc_lam_flux != 0) P.k0m = 1;
  P.k00 = (P.k0 > 1) ? 1 : P.k0m;  // adz_traject.F90:63-64
  P.k00i = std::max(P.k0t - 1, 1);  // adz_interp_traj.F90:38-39
  if (g->bc_lam_flux != 0 && P.k0 > 1) P.k00i = 1;
  const double EPS_8 = 2.0e-5;
  const int BCS = 4;
  P.iminposx = g->i0g + P.lminx + EPS_8; P.imaxposx = g->i0g + lmaxx - 2 - EPS_8;
  P.iminposy = g->j0g + P.lminy + EPS_8; P.imaxposy = g->j0g + lmaxy - 2 - EPS_8;
  if (g->west) P.iminposx = g->i0g + BCS + EPS_8;
  if (g->east) P.imaxposx = g->i0g + ni - BCS - 1 - EPS_8;
  if (g->south) P.iminposy = g->j0g + BCS + EPS_8;
  if (g->north) P.imaxposy = g->j0g + nj - BCS - 1 - EPS_8;
  P.i0b = 1 + BCS * g->west; P.inb = ni - BCS * g->east; P.j0b = 1 + BCS * g->south; P.jnb = nj - BCS * g->north;
  if (P.i0 < 1 || P.in > ni || P.j0 < 1 || P.jn > nj || P.i0 < P.i0b || P.in > P.inb || P.j0 < P.j0b || P.jn > P.jnb) {
    delete c;
    return fail(ADZ_EINVAL, "adz_set: pilot widths too small for the interpolation boxes (need pil >= 6 on edges)");
  }
  if (P.in < P.i0 || P.jn < P.j0 || P.inu < P.i0u || P.jnv < P.j0v || P.inb < P.i0b || P.jnb < P.j0b ||
      P.k0 > nk || P.k0t > nk) {
    delete c;
    return fail(ADZ_EINVAL, "adz_set: tile too small for its pilot zones (an interpolation box is empty)");
  }
  c->zm.assign(g->zm, g->zm + nk + 2); c->zt.assign(g->zt, g->zt + nk + 2); c->zx.assign(g->zx, g->zx + nk + 1);
  const auto& zm = c->zm; const auto& zt = c->zt; const auto& zx = c->zx;
  P.sig = (zm[nk] - zm[1]) / std::fabs(zm[nk] - zm[1]);
  c->delz_m.assign(nk + 1, (double)9.e33f); c->delz_t.assign(nk + 1, (double)9.e33f);
  c->odelz_m.assign(nk + 1, 0.0); c->odelz_t.assign(nk + 1, 0.0);
  const float verysmall = 1.17549435e-38f * 1.e5f;
  for (int k = 0; k <= nk; k++) {
    if (std::fabs(zm[k + 1] - zm[k]) > (double)verysmall) c->delz_m[k] = zm[k + 1] - zm[k];
    if (std::fabs(zt[k + 1] - zt[k]) > (double)verysmall) c->delz_t[k] = zt[k + 1] - zt[k];
    c->odelz_m[k] = 1.0 / c->delz_m[k];
    c->odelz_t[k] = 1.0 / c->delz_t[k];
  }
  search_table(zm, c->delz_m, nk, P.sig, &P.ovdzm, &c->search_m);
  search_table(zt, c->delz_t, nk, P.sig, &P.ovdzt, &c->search_t);
  P.pnz_m = (int)c->search_m.size(); P.pnz_t = (int)c->search_t.size();
  c->cy.resize(P.njt);
  for (int j = 0; j < P.njt; j++) c->cy[j] = 1.0 / std::cos(g->lat[j]);
  c->vw.assign(8 * (nk + 1), 0.0);
  double* vw = c->vw.data();
  for (int k = 2; k <= nk - 1; k++) {
    double rx = zm[k], ra = zx[k - 2], rb = zx[k - 1], rc = zx[k], rd = zx[k + 1];
    vw[k] = lag3(rx, ra, rb, rc, rd);
    vw[(nk + 1) + k] = lag3(rx, rb, ra, rc, rd);
    vw[2 * (nk + 1) + k] = lag3(rx, rc, ra, rb, rd);
    vw[3 * (nk + 1) + k] = lag3(rx, rd, ra, rb, rc);
  }
  for (int k = 2; k <= nk - 2; k++) {
    double rx = zt[k], ra = zm[k - 1], rb = zm[k], rc = zm[k + 1], rd = zm[k + 2];
    vw[4 * (nk + 1) + k] = lag3(rx, ra, rb, rc, rd);
    vw[5 * (nk + 1) + k] = lag3(rx, rb, ra, rc, rd);
    vw[6 * (nk + 1) + k] = lag3(rx, rc, ra, rb, rd);
    vw[7 * (nk + 1) + k] = lag3(rx, rd, ra, rb, rc);
  }
  P.vw5 = (zx[0] - zm[1]) / (zx[0] - zx[1]);
  P.vw6 = (zm[nk] - zx[nk]) / (zx[nk - 1] - zx[nk]);
  P.zmin = g->zmin; P.zmax = g->zmax; P.inv_hx = g->inv_hx; P.inv_hy = g->inv_hy; P.inv_rayt = g->inv_rayt;
  P.ww_star = g->wmstar_nk;
  P.wp_nk = (zt[nk] - zm[nk - 1]) * g->idz_t_nkm1;
  P.wm_nk = 1.0 - P.wp_nk;

  // device tables
  size_t nd = (size_t)(nk + 2) * 2 + (size_t)(nk + 1) * 2 + P.njt + 8 * (nk + 1);
  size_t bytes = nd * 8 + (c->search_m.size() + c->search_t.size()) * 4;
  if (hipMalloc(&c->tables, bytes) != hipSuccess) { free_ctx(c); return fail(ADZ_ENOMEM, "adz_set: tables"); }
  std::vector<char> h(bytes);
  char* p = h.data();
  auto put = [&](const void* src, size_t b) { std::memcpy(p, src, b); p += b; };
  put(zm.data(), 8 * (nk + 2)); put(zt.data(), 8 * (nk + 2)); put(c->odelz_m.data(), 8 * (nk + 1));
  put(c->odelz_t.data(), 8 * (nk + 1)); put(c->cy.data(), 8 * P.njt); put(vw, 8 * 8 * (nk + 1));
  put(c->search_m.data(), 4 * c->search_m.size()); put(c->search_t.data(), 4 * c->search_t.size());
  if (hipMemcpy(c->tables, h.data(), bytes, hipMemcpyHostToDevice) != hipSuccess) {
    free_ctx(c);
    return fail(ADZ_EHIP, "adz_set: table upload");
  }
  char* d = (char*)c->tables;
  P.zm = (const double*)d; d += 8 * (nk + 2);
  P.zt = (const double*)d; d += 8 * (nk + 2);
  P.odelz_m = (const double*)d; d += 8 * (nk + 1);
  P.odelz_t = (const double*)d; d += 8 * (nk + 1);
  P.cy = (const double*)d; d += 8 * P.njt;
  P.vw = (const double*)d; d += 8 * 8 * (nk + 1);
  P.search_m = (const int*)d; d += 4 * c->search_m.size();
  P.search_t = (const int*)d;

  // BICHQV tables (adz_set.F90:286-307): delz_t, then the inverse cubic and quintic
  // Lagrange denominators of the thermodynamic levels, each indexed by k
  {
    std::vector<double> q(11 * (size_t)(nk + 1), 0.0);
    std::memcpy(q.data(), c->delz_t.data(), 8 * (nk + 1));
    double* c4 = q.data() + (nk + 1);
    double* c6 = c4 + 4 * (nk + 1);
    auto tri = [](double za, double zb, double zc, double zd) { return ((za - zb) * (za - zc) * (za - zd)); };
    auto qui = [](double zx, double za, double zb, double zc, double zd, double ze) {
      return ((zx - za) * (zx - zb) * (zx - zc) * (zx - zd) * (zx - ze));
    };
    for (int k = 2; k <= nk - 2; k++) {
      double ra = zt[k - 1], rb = zt[k], rc = zt[k + 1], rd = zt[k + 2];
      c4[k] = 1.0 / tri(ra, rb, rc, rd);
      c4[(nk + 1) + k] = 1.0 / tri(rb, ra, rc, rd);
      c4[2 * (nk + 1) + k] = 1.0 / tri(rc, ra, rb, rd);
      c4[3 * (nk + 1) + k] = 1.0 / tri(rd, ra, rb, rc);
    }
    for (int k = 3; k <= nk - 3; k++) {
      double rx = zt[k - 2], ra = zt[k - 1], rb = zt[k], rc = zt[k + 1], rd = zt[k + 2], re = zt[k + 3];
      c6[k] = 1.0 / qui(rx, ra, rb, rc, rd, re);
      c6[(nk + 1) + k] = 1.0 / qui(ra, rx, rb, rc, rd, re);
      c6[2 * (nk + 1) + k] = 1.0 / qui(rb, rx, ra, rc, rd, re);
      c6[3 * (nk + 1) + k] = 1.0 / qui(rc, rx, ra, rb, rd, re);
      c6[4 * (nk + 1) + k] = 1.0 / qui(rd, rx, ra, rb, rc, re);
      c6[5 * (nk + 1) + k] = 1.0 / qui(re, rx, ra, rb, rc, rd);
    }
    if (hipMalloc(&c->qvtab, 8 * q.size()) != hipSuccess) { free_ctx(c); return fail(ADZ_ENOMEM, "adz_set: tables"); }
    if (hipMemcpy(c->qvtab, q.data(), 8 * q.size(), hipMemcpyHostToDevice) != hipSuccess) {
      free_ctx(c);
      return fail(ADZ_EHIP, "adz_set: table upload");
    }
  }

  // layer thicknesses of the air mass (set_zeta.F90:271-275): Ver_dz_8%t(k) =
  // Ver_z_8%m(k+1) - Ver_z_8%m(k) and its inverse, k = 1..nk (entry 0 unused)
  {
    std::vector<double> a(2 * (size_t)(nk + 1), 0.0);
    for (int k = 1; k <= nk; k++) {
      a[k] = zm[k + 1] - zm[k];
      a[(nk + 1) + k] = 1.0 / a[k];
    }
    if (hipMalloc(&c->amtab, 8 * a.size()) != hipSuccess) { free_ctx(c); return fail(ADZ_ENOMEM, "adz_set: tables"); }
    if (hipMemcpy(c->amtab, a.data(), 8 * a.size(), hipMemcpyHostToDevice) != hipSuccess) {
      free_ctx(c);
      return fail(ADZ_EHIP, "adz_set: table upload");
    }
  }

  // vertical descriptors (adz_set.F90:128-131) over the extended arrays
  int st = adz_vsearch_setup_plus(&zm[1], nk, P.nit, P.njt, 1 - g->i0g, 1 - g->j0g, &c->zq);
  if (st == ADZ_OK) st = adz_vsearch_setup_plus(&zt[1], nk, P.nit, P.njt, 1 - g->i0g, 1 - g->j0g, &c->zth);
  if (st != ADZ_OK) { free_ctx(c); return st; }
  adz_vsearch_set_bounds(c->zq, P.lminx, lmaxx, P.lminy, lmaxy);
  adz_vsearch_set_bounds(c->zth, P.lminx, lmaxx, P.lminy, lmaxy);

  // device state (adz_set.F90:313-341, 346-360)
  const size_t sz = pos_dtype == ADZ_F32 ? 4 : 8;
  long nxy = (long)ni * nj;
  c->n_uvw_d = 3L * P.nij * nk; c->n_arr = 3 * nxy * nk; c->n_p3 = 3 * nxy * (nk - P.k0m + 1);
  c->n_wp = (long)(ni + 4) * (nj + 4) * nk * 3;
  c->n_pm = 3L * (P.in - P.i0 + 1) * (P.jn - P.j0 + 1) * (nk - P.k0 + 1);
  c->n_pmu = 3L * (P.inu - P.i0u + 1) * (P.jn - P.j0 + 1) * (nk - P.k0 + 1);
  c->n_pmv = 3L * (P.in - P.i0 + 1) * (P.jnv - P.j0v + 1) * (nk - P.k0 + 1);
  c->n_pt = 3L * (P.in - P.i0 + 1) * (P.jn - P.j0 + 1) * (nk - P.k0t + 1);
  c->n_pb = 3L * (P.inb - P.i0b + 1) * (P.jnb - P.j0b + 1) * nk;
  struct { void** p; size_t b; } al[] = {
      {&c->uvw_d, c->n_uvw_d * sz + 16}, {&c->warr, c->n_arr * sz}, {&c->uvw_dep, c->n_p3 * sz},
      {&c->pxyzm, c->n_p3 * sz},    {(void**)&c->wpxyz, (size_t)c->n_wp * 8}, {&c->pm, c->n_pm * sz},
      {&c->pmu, c->n_pmu * sz},     {&c->pmv, c->n_pmv * sz}, {&c->pt, c->n_pt * sz}, {&c->pb, c->n_pb * sz}};
  for (auto& a : al) {
    if (hipMalloc(a.p, a.b) != hipSuccess) { free_ctx(c); return fail(ADZ_ENOMEM, "adz_set: state allocation"); }
    if (hipMemset(*a.p, 0, a.b) != hipSuccess) { free_ctx(c); return fail(ADZ_EHIP, "adz_set: state clear"); }
  }
  *out = c;
  return ADZ_OK;
}

int adz_ctx_free(adz_ctx* c) {
  if (c) free_ctx(c);
  return ADZ_OK;
}

int adz_ctx_info(const adz_ctx* c, int* iv, double* dv) {
  if (!c || !iv || !dv) return fail(ADZ_EINVAL, "adz_ctx_info: null argument");
  const TrajParams& P = c->P;
  int a[] = {P.lminx, P.ni + (P.nit - P.ni) / 2, P.lminy, P.nj + (P.njt - P.nj) / 2, P.nit, P.njt, P.nij,
             P.i0, P.in, P.j0, P.jn, P.i0u, P.inu, P.j0v, P.jnv, P.i0b, P.inb, P.j0b, P.jnb, P.k0, P.k0t, P.k0m,
             P.pnz_m, P.pnz_t};
  std::memcpy(iv, a, sizeof(a));
  double b[] = {P.iminposx, P.imaxposx, P.iminposy, P.imaxposy, P.sig, P.ovdzm, P.ovdzt, P.vw5, P.vw6};
  std::memcpy(dv, b, sizeof(b));
  return ADZ_OK;
}

int adz_ctx_table(const adz_ctx* c, int which, void* out) {
  if (!c || !out || which < 0 || which > 12) return fail(ADZ_EINVAL, "adz_ctx_table: bad argument");
  int nk = c->P.nk;
  if (which == 0) std::memcpy(out, c->search_m.data(), 4 * c->search_m.size());
  else if (which == 1) std::memcpy(out, c->search_t.data(), 4 * c->search_t.size());
  else if (which <= 9) std::memcpy(out, c->vw.data() + (which - 2) * (nk + 1), 8 * (nk + 1));
  else if (which == 10) std::memcpy(out, c->cy.data(), 8 * c->cy.size());
  else if (which == 11) std::memcpy(out, c->odelz_m.data(), 8 * (nk + 1));
  else std::memcpy(out, c->odelz_t.data(), 8 * (nk + 1));
  return ADZ_OK;
}

int adz_ctx_array(adz_ctx* c, int which, void** dptr, long* nelem) {
  if (!c || !dptr) return fail(ADZ_EINVAL, "adz_ctx_array: null argument");
  void* p[] = {c->pxyzm, c->wpxyz, c->uvw_dep, c->pm, c->pmu, c->pmv, c->pt, c->pb, c->uvw_d, c->warr};
  long n[] = {c->n_p3, c->n_wp, c->n_p3, c->n_pm, c->n_pmu, c->n_pmv, c->n_pt, c->n_pb, c->n_uvw_d, c->n_arr};
  if (which < 0 || which > 9) return fail(ADZ_EINVAL, "adz_ctx_array: unknown array");
  *dptr = p[which];
  if (nelem) *nelem = n[which];
  return ADZ_OK;
}

const adz_ztab* adz_ctx_ztab(const adz_ctx* c, int thermo) { return c ? (thermo ? c->zth : c->zq) : nullptr; }

}  // extern "C"

bool adz::ctx_qv(const adz_ctx* c, QvDev* q) {
  if (!c || !c->qvtab) return false;
  const int nk = c->P.nk;
  q->posz = c->P.zt;
  q->odz = c->P.odelz_t;
  q->dz = (const double*)c->qvtab;
  q->c4 = q->dz + (nk + 1);
  q->c6 = q->c4 + 4 * (nk + 1);
  q->nk = nk;
  q->offi = 1 - c->P.i0g;
  q->offj = 1 - c->P.j0g;
  q->lminx = c->P.lminx; q->lmaxx = c->P.lminx + c->P.nit - 1;
  q->lminy = c->P.lminy; q->lmaxy = c->P.lminy + c->P.njt - 1;
  q->pos_dtype = c->pos_dtype;
  return true;
}

bool adz::ctx_airmass(const adz_ctx* c, AirmassTables* t) {
  if (!c || !c->amtab) return false;
  const int nk = c->P.nk;
  t->dz = (const double*)c->amtab;
  t->idz = t->dz + (nk + 1);
  t->nk = nk; t->ni = c->P.ni; t->nj = c->P.nj; t->k0t = c->P.k0t;
  return true;
}

extern "C" {

// ---------------------------------------------------------------- restart of the SL state
// What the reference checkpoints for the semi-Lagrangian scheme: ADZ_PXYZM and ADZ_WPXYZ,
// registered with GMM_FLAG_RSTR (adz_set.F90:343-360).  The blob is a fixed header, then
// Adz_pxyzm in the context's position storage, then Adz_wpxyz in FP64.  The iteration
// count of the next adz_traject is kept too (the reference restarts at a step boundary,
// where it is Adz_itraj: adz_traject.F90:120, adz_set.F90:424).
namespace {
struct StateHeader {
  char magic[8];
  int32_t pos_dtype, ni, nj, nk, k0m, niter;
  int64_t n_p3, n_wp;
};
constexpr char kStateMagic[8] = {'A', 'D', 'Z', 'S', 'T', 'A', 'T', '1'};

size_t state_bytes(const adz_ctx* c) {
  const size_t sz = c->pos_dtype == ADZ_F32 ? 4 : 8;
  return sizeof(StateHeader) + (size_t)c->n_p3 * sz + (size_t)c->n_wp * 8;
}
}  // namespace

int adz_ctx_state_bytes(const adz_ctx* c, size_t* bytes) {
  if (!c || !bytes) return fail(ADZ_EINVAL, "adz_ctx_state_bytes: null argument");
  *bytes = state_bytes(c);
  return ADZ_OK;
}

int adz_ctx_save_state(const adz_ctx* c, void* host, size_t bytes, adz_stream s) {
  if (!c || !host) return fail(ADZ_EINVAL, "adz_ctx_save_state: null argument");
  if (bytes < state_bytes(c)) return fail(ADZ_EINVAL, "adz_ctx_save_state: buffer too small");
  StateHeader h;
  std::memcpy(h.magic, kStateMagic, 8);
  h.pos_dtype = c->pos_dtype; h.ni = c->P.ni; h.nj = c->P.nj; h.nk = c->P.nk; h.k0m = c->P.k0m;
  h.niter = c->niter; h.n_p3 = c->n_p3; h.n_wp = c->n_wp;
  std::memcpy(host, &h, sizeof(h));
  char* p = (char*)host + sizeof(h);
  const size_t b3 = (size_t)c->n_p3 * (c->pos_dtype == ADZ_F32 ? 4 : 8);
  ADZ_HIP_CHECK(hipMemcpyAsync(p, c->pxyzm, b3, hipMemcpyDeviceToHost, (hipStream_t)s));
  ADZ_HIP_CHECK(hipMemcpyAsync(p + b3, c->wpxyz, (size_t)c->n_wp * 8, hipMemcpyDeviceToHost, (hipStream_t)s));
  ADZ_HIP_CHECK(hipStreamSynchronize((hipStream_t)s));
  return ADZ_OK;
}

int adz_ctx_load_state(adz_ctx* c, const void* host, size_t bytes, adz_stream s) {
  if (!c || !host) return fail(ADZ_EINVAL, "adz_ctx_load_state: null argument");
  if (bytes < sizeof(StateHeader)) return fail(ADZ_EINVAL, "adz_ctx_load_state: buffer too small");
  StateHeader h;
  std::memcpy(&h, host, sizeof(h));
  if (std::memcmp(h.magic, kStateMagic, 8) != 0) return fail(ADZ_EINVAL, "adz_ctx_load_state: not an SL state");
  if (h.pos_dtype != c->pos_dtype || h.ni != c->P.ni || h.nj != c->P.nj || h.nk != c->P.nk || h.k0m != c->P.k0m ||
      h.n_p3 != c->n_p3 || h.n_wp != c->n_wp)
    return fail(ADZ_EINVAL, "adz_ctx_load_state: the state belongs to another grid or position storage");
  if (bytes < state_bytes(c)) return fail(ADZ_EINVAL, "adz_ctx_load_state: buffer too small");
  if (h.niter < 1) return fail(ADZ_EINVAL, "adz_ctx_load_state: bad iteration count");
  const char* p = (const char*)host + sizeof(h);
  const size_t b3 = (size_t)c->n_p3 * (c->pos_dtype == ADZ_F32 ? 4 : 8);
  ADZ_HIP_CHECK(hipMemcpyAsync(c->pxyzm, p, b3, hipMemcpyHostToDevice, (hipStream_t)s));
  ADZ_HIP_CHECK(hipMemcpyAsync(c->wpxyz, p + b3, (size_t)c->n_wp * 8, hipMemcpyHostToDevice, (hipStream_t)s));
  ADZ_HIP_CHECK(hipStreamSynchronize((hipStream_t)s));
  c->niter = h.niter;
  return ADZ_OK;
}

int adz_inittraj(adz_ctx* c, adz_stream s) {
  if (!c) return fail(ADZ_EINVAL, "adz_inittraj: null context");
  long n = (long)c->P.ni * c->P.nj * (c->P.nk - c->P.k0m + 1);
  if (c->pos_dtype == ADZ_F32)
    hipLaunchKernelGGL(k_inittraj<float>, dim3(nb(n)), dim3(256), 0, (hipStream_t)s, (float*)c->pxyzm, c->wpxyz, c->P);
  else
    hipLaunchKernelGGL(k_inittraj<double>, dim3(nb(n)), dim3(256), 0, (hipStream_t)s, (double*)c->pxyzm, c->wpxyz, c->P);
  ADZ_HIP_CHECK(hipGetLastError());
  c->niter = std::max(6, c->itraj);
  return ADZ_OK;
}

int adz_traject(adz_ctx* c, double dt, int schm_advec, double bA_m, double bA, const float* uu_ext,
                const float* vv_ext, const float* ww_ext, const float* ut0, const float* vt0, const float* zdt0,
                adz_stream s) {
  if (!c || !uu_ext || !vv_ext || !ww_ext || !ut0 || !vt0 || !zdt0) return fail(ADZ_EINVAL, "adz_traject: null argument");
  if (schm_advec < 0 || schm_advec > 3) return fail(ADZ_EINVAL, "adz_traject: Schm_advec must be 0..3");
  if (c->pos_dtype == ADZ_F32)
    return run_traject<float>(c, dt, schm_advec, bA_m, bA, uu_ext, vv_ext, ww_ext, ut0, vt0, zdt0, (hipStream_t)s);
  return run_traject<double>(c, dt, schm_advec, bA_m, bA, uu_ext, vv_ext, ww_ext, ut0, vt0, zdt0, (hipStream_t)s);
}

}  // extern "C"
