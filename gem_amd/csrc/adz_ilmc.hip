// ILMC shape preservation (mono = 2; Sorensen et al. 2013, GMD 6, 1029-1042) on gfx950:
// ILMC_LAM.F90:18-273 with its sweep loop ilmc_lam_loop.inc:16-139, for a tile that touches
// the four LAM edges (the domain is F_i0..F_in x F_j0..F_jn x Adz_k0t..nk,
// ILMC_LAM.F90:81-86).
//
// The reference visits every cell of the domain in (k, j, i) order.  A cell above its max
// (below its min) moves mass into (out of) the cells of sweep 1, 2, ..., S around it -- the
// cells at Chebyshev distance s, clipped to the domain -- up to their own max (min), and a
// later visit sees the values the earlier ones left.  That order is kept exactly, in
// parallel:
//   * a cell inside [min, max] never leaves it: mass is added up to a cell's max and
//     removed down to its min, and only where there is room.  So the cells to visit are the
//     cells that violate their bounds before the first visit; the loop skips the others
//     (ilmc_lam_loop.inc:26) and so does this code;
//   * a visit reads and writes only the cube of half-width S around its cell, so two
//     visits commute unless their cells lie within Chebyshev distance 2S.
// A row's cells are taken in windows of kIlWin = 4; a window with violating cells is one
// piece of work, visited cell by cell by one wave.  A window waits for the windows that come
// before it in the sequential order and lie within reach: those to its left, and in earlier
// rows of its level (up to 2S back) and of earlier levels (2S rows either way) those up to
// d = ceil(2S / 4) windows to its left and right.  With wi the window's number in its row,
// all of these have a smaller t = wi + a dj + b dk, a = d + 1, b = d + 2S a + 1 (b = 0 with
// Schm_autobar_L, whose sweeps stay on one level): wi + d - a < wi, and
// wi + d + 2S a - b < wi.
// The windows are listed by t and the waves of ONE launch take them in that order from a
// ticket counter.  A bit per cell says which cells are still to be visited; a wave polls the
// bits it waits for and clears its own when its window's values are written.  Each visit
// sees exactly the values the sequential loop gives it.
//
// Why every wait ends: the list order is a topological order of the waits, and an entry is
// taken from the ticket counter only by a wave that is running, so the first entry not yet
// visited is always held by a running wave that waits for nothing.  The waits are bounded all
// the same: one that gives up raises a flag and ends its wave, as does every wait that sees the
// flag; windows whose waits are over are still visited, and k_il_finish visits what is left in
// list order with one wave, so the result is exact in either case.
//
// The wave holds its window's surroundings, (4 + 2S) x (2S+1) x (2S+1) cells, in LDS: f, its
// bounds and the air mass.  For each visit the lanes form the cube's masses, every lane adds
// a sweep's masses in the reference's order (j, then k, then i), and the lanes redistribute.
//
// What bounds it: the chain of visits that wait for each other.  Fronts of two tracers on
// 384 x 288 x 84 (100 000 to 490 000 violating cells) hold chains of 2000 to 2570 cells; by
// windows of four, about 1000 windows and 2000 to 3900 visits.  A link costs the visits
// (about 1 us each, most of it the sums in the reference's order) and some 3 us of round
// trips to memory (the poll, f, the stores).  With one launch per hyperplane of cells the call
// took 21.1 ms on any front; with one wave per cell in this scheme 7.4 to 16 ms; with windows
// of 16, 6.2 (fronts along j) to 21 ms (along i); of 8, 5.8 to 13.9; of 2, 6.5 to 9.6; of 4,
// 4.9 to 7.9 ms.
//
// f is read and written by agent-scope atomics only, which pass the caches that the XCDs do
// not share, so a window needs no fence that writes back or invalidates a whole L2: it waits
// for its own stores before it clears its bits.  With such fences, and with more waves, the
// waves are in each other's way: 20 tracers of 512 x 384 x 84 with fronts 40 ms as a launch per
// hyperplane, 74 with fences and 2048 waves, 42 with 512 waves, 23 without the fences; 6 smooth
// tracers of 1024 x 512 x 84 37, 41, 30 and 22.5 ms.
// Arithmetic is the reference's `real` arithmetic as written (built without contraction).
#include <algorithm>
#include <cstring>
#include <vector>

#include "adz_common.h"

namespace adz {

constexpr int kIlBlock = 256;
constexpr int kIlScan = 1024;
constexpr int kIlWin = 4;          // cells of a row per piece of work
constexpr uint64_t kIlMask = (1ull << kIlWin) - 1;
constexpr int kIlWaves = 512;      // waves of the visiting launch
constexpr int kIlFew = 128;        // those of them per tracer that visit in any case
constexpr int kIlSpin = 1 << 22;   // polls of one wait (about 1 us each) before it gives up

struct IlmcTr {
  float* f;
  const float* mn;
  const float* mx;
};

struct IlmcArgs {
  const IlmcTr* tr;
  int ntr;
  long nx, nxy;                 // array pitches (pointers address element (1,1,1))
  int i0, j0, k0, ni, nj, nkk;  // domain origin and extents
  int a, b;                     // coefficients of t
  int nplanes;                  // values of t
  int wpr;                      // 64-cell words per row of `pend`
  int spin_limit;               // polls of one wait before it gives up
  const float* air;
  unsigned long long* cnt;  // [nplanes] windows per t, then fill cursors
  unsigned long long* ctl;  // [0] next list entry, [1] nonzero once a wait gave up
  long long* off;           // [nplanes + 1] list starts
  uint64_t* list;           // windows by t: wi | j << 16 | k << 32 | tracer << 44 (domain offsets)
  uint64_t* pend;           // [tracer][k][j][wpr]: bit i of a row set while cell i is to be visited
  long long* counts;
};

__device__ __forceinline__ float il_max(float a, float b) { return (b > a) ? b : a; }
__device__ __forceinline__ float il_min(float a, float b) { return (b < a) ? b : a; }

// Values that visits on different XCDs exchange (f and the pending bits) are read and
// written at agent scope, past the L2 of one XCD.
template <class P>
__device__ __forceinline__ auto il_load(P p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class P, class T>
__device__ __forceinline__ void il_store(P p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Zeros in two arrays of 8-byte words.
__global__ __launch_bounds__(kIlBlock) void k_il_zero(long long* p, long n, long long* q, long m) {
  const long e = (long)blockIdx.x * kIlBlock + threadIdx.x;
  if (e < n) p[e] = 0;
  if (e < m) q[e] = 0;
}

// The cells outside [min, max]: a bit each in `pend`, and their windows counted per t.  One
// wave takes 64 cells of a row at a time, kIlUnroll such words in flight; a block takes `rows`
// rows of one tracer.
constexpr int kIlUnroll = 4;
__global__ __launch_bounds__(kIlBlock) void k_il_mark(IlmcArgs A, int rows) {
  const int n = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row0 = blockIdx.x * rows, nrow = min(rows, A.nj * A.nkk - row0), words = nrow * A.wpr;
  const IlmcTr T = A.tr[n];
  for (int w0 = wave; w0 < words; w0 += kIlBlock / 64 * kIlUnroll) {
    float f[kIlUnroll], mn[kIlUnroll], mx[kIlUnroll];
    int di[kIlUnroll], row[kIlUnroll];
#pragma unroll
    for (int u = 0; u < kIlUnroll; u++) {
      const int w = w0 + u * (kIlBlock / 64), r = w / A.wpr;
      row[u] = row0 + r;
      di[u] = w < words ? (w - r * A.wpr) * 64 + lane : A.ni;
      const int dk = row[u] / A.nj, dj = row[u] - dk * A.nj;
      const long c = (long)(A.i0 - 1) + A.nx * (A.j0 + dj - 1) + A.nxy * (A.k0 + dk - 1) + di[u];
      f[u] = mn[u] = mx[u] = 0.f;
      if (di[u] < A.ni) { f[u] = T.f[c]; mn[u] = T.mn[c]; mx[u] = T.mx[c]; }
    }
#pragma unroll
    for (int u = 0; u < kIlUnroll; u++) {
      const int w = w0 + u * (kIlBlock / 64);
      const float o = il_max(0.f, f[u] - mx[u]), d = il_max(0.f, mn[u] - f[u]);
      const unsigned long long m = __ballot(!(o == 0.f && d == 0.f));
      if (w < words && lane == 0) A.pend[((long)n * A.nj * A.nkk + row0) * A.wpr + w] = m;
      if (!(lane % kIlWin) && ((m >> lane) & kIlMask)) {
        const int dk = row[u] / A.nj, dj = row[u] - dk * A.nj;
        atomicAdd(&A.cnt[di[u] / kIlWin + A.a * dj + A.b * dk], 1ull);
      }
    }
  }
}

// The windows with marked cells into the list, each at its t's cursor (the order among equal t
// does not matter: such windows do not wait for each other).  One lane per word of `pend`.
__global__ __launch_bounds__(kIlBlock) void k_il_fill(IlmcArgs A) {
  const int n = blockIdx.y;
  const long words = (long)A.nj * A.nkk * A.wpr, w = (long)blockIdx.x * kIlBlock + threadIdx.x;
  const uint64_t v = w < words ? A.pend[(long)n * words + w] : 0ull;
  if (!v) return;
  const unsigned row = (unsigned)(w / A.wpr);
  const int dk = (int)(row / (unsigned)A.nj), dj = (int)(row - (unsigned)dk * A.nj);
  const int wi0 = (int)(w - (long)row * A.wpr) * (64 / kIlWin);
  for (int q = 0; q < 64 / kIlWin; q++)
    if ((v >> (kIlWin * q)) & kIlMask) {
      const unsigned long long pos = atomicAdd(&A.cnt[wi0 + q + A.a * dj + A.b * dk], 1ull);
      A.list[pos] = (uint64_t)(wi0 + q) | ((uint64_t)dj << 16) | ((uint64_t)dk << 32) | ((uint64_t)n << 44);
    }
}

// One block: off = exclusive prefix sum of cnt, off[nplanes] = total; cnt becomes the fill
// cursor (= off).
__global__ __launch_bounds__(kIlScan) void k_il_scan(IlmcArgs A) {
  __shared__ long long s[kIlScan];
  const int t = threadIdx.x;
  long long run = 0;
  for (int b0 = 0; b0 < A.nplanes; b0 += kIlScan) {
    const int q = b0 + t;
    const long long v = q < A.nplanes ? (long long)A.cnt[q] : 0;
    s[t] = v;
    __syncthreads();
    for (int o = 1; o < kIlScan; o <<= 1) {
      const long long w = t >= o ? s[t - o] : 0;
      __syncthreads();
      s[t] += w;
      __syncthreads();
    }
    if (q < A.nplanes) {
      A.off[q] = run + s[t] - v;
      A.cnt[q] = (unsigned long long)(run + s[t] - v);
    }
    run += s[kIlScan - 1];
    __syncthreads();
  }
  if (t == 0) A.off[A.nplanes] = run;
}

struct IlWindow {
  int di, dj, dk, n;  // first cell, row, level, tracer
  uint64_t* pend;     // the word that holds the window's bits, at di & 63
  long row0;          // element (from (1,1,1)) of the row's first cell of the domain
};
__device__ __forceinline__ uint64_t* il_row(const IlmcArgs& A, int n, int dj, int dk) {
  return A.pend + (((long)n * A.nkk + dk) * A.nj + dj) * A.wpr;
}
__device__ __forceinline__ IlWindow il_window(const IlmcArgs& A, uint64_t code) {
  IlWindow x;
  x.di = (int)(code & 0xffff) * kIlWin;
  x.dj = (int)((code >> 16) & 0xffff);
  x.dk = (int)((code >> 32) & 0xfff);
  x.n = (int)(code >> 44);
  x.pend = il_row(A, x.n, x.dj, x.dk) + (x.di >> 6);
  x.row0 = (long)(A.i0 - 1) + A.nx * (A.j0 + x.dj - 1) + A.nxy * (A.k0 + x.dk - 1);
  return x;
}

// Waits until no cell that the sequential loop visits before the window and that lies within
// distance D = 2S of it is pending.  Lane l watches the rows l, l + 64, ... of that
// neighbourhood (rows of earlier levels, earlier rows of the window's level, then its own row
// up to it); a row's 4 + 2D <= 20 bits lie in one or two words.  False if the wait gave up.
template <int S, bool AB>
__device__ __forceinline__ bool il_wait(const IlmcArgs& A, const IlWindow& x) {
  constexpr int D = 2 * S, W = 2 * D + 1, RK = AB ? 0 : D * W, R = RK + D + 1;
  const int lane = threadIdx.x;
  int polls = 0;
#pragma unroll 1
  for (int r0 = 0; r0 < R; r0 += 64) {
    const int r = r0 + lane;
    const int ek = r < RK ? -1 - r / W : 0, ej = r < RK ? r % W - D : r - RK - D;
    const int dj = x.dj + ej, dk = x.dk + ek;
    const int lo = max(0, x.di - D), hi = (ek == 0 && ej == 0) ? x.di - 1 : min(A.ni - 1, x.di + kIlWin - 1 + D);
    bool wait = r < R && dj >= 0 && dj < A.nj && dk >= 0 && hi >= lo;
    const int w0 = lo >> 6, w1 = wait ? hi >> 6 : w0;
    uint64_t m0 = ~0ull << (lo & 63), m1 = ~0ull >> (63 - (hi & 63));
    if (w1 == w0) { m0 &= m1; m1 = 0ull; }
    const ADZ_GLOBAL uint64_t* p = (const ADZ_GLOBAL uint64_t*)(wait ? il_row(A, x.n, dj, dk) : A.pend);
    for (;;) {
      if (wait) {
        uint64_t v = il_load(p + w0) & m0;
        if (m1) v |= il_load(p + w1) & m1;
        wait = v != 0ull;
      }
      if (!__any(wait)) break;
      if (polls >= A.spin_limit) {
        il_store(A.ctl + 1, 1ull);
        return false;
      }
      if ((++polls & 15) == 0 && __any(il_load(A.ctl + 1) != 0)) return false;
      // the polls of windows far from their turn would slow the others: with 512 waves and no
      // pause the call above took 6.6 ms where 256 waves with these pauses take 4.9
      const int rows = __popcll(__ballot(wait));
      if (rows > 6) __builtin_amdgcn_s_sleep(64);
      else if (rows > 2) __builtin_amdgcn_s_sleep(8);
    }
  }
  return true;
}

// A window's surroundings in LDS: (4 + 2S) columns x (2S+1) levels x (2S+1) rows, cell e at
// column e % NC, level (e / NC) % NL, row e / (NC NL) (the order j, k, i of the sums).  Cells
// outside the domain hold air = 0 and bounds that leave no room (their masses are +0, which
// leaves a sum of non-negative terms unchanged).
template <int S, bool AB>
struct IlBox {
  static constexpr int W = 2 * S + 1, NL = AB ? 1 : W, NC = kIlWin + 2 * S, N = NC * NL * W, NQ = (N + 63) / 64;
  static constexpr int P = W * NL * W, NP = (P + 63) / 64;  // the cube of one visit
  static constexpr bool kHeld = P <= 128;                   // its masses fit in registers (read as quads)
  static constexpr int kUnroll = kHeld ? NQ : 2;
  float f[N], mn[N], mx[N], air[N];
  float was[N];  // f before the window's visits
  float __attribute__((aligned(16))) mass[(P + 3) / 4 * 4];
};

// What the lanes know of the box and the cube, the same for every window: lane l holds the
// cells l + 64 r.
template <int S, bool AB>
struct IlLane {
  typedef IlBox<S, AB> B;
  int table[B::kHeld ? B::NQ : 1];
  int cube[B::NP];   // cube cell r: place in the box for the box's column S
  int dist[B::NP];   // its sweep (0: the centre, or no cell)
  // Box cell r: column | level << 8 | row << 16, from the box's corner.
  __device__ __forceinline__ static int place(int r) {
    const int e = threadIdx.x + 64 * r, ci = e % B::NC, ck = (e / B::NC) % B::NL, cj = e / (B::NC * B::NL);
    return ci | (AB ? S : ck) << 8 | cj << 16;
  }
  __device__ __forceinline__ int at(int r) const {
    if constexpr (B::kHeld) return table[r];
    else return place(r);
  }
  __device__ __forceinline__ void init() {
    if constexpr (B::kHeld) {
#pragma unroll
      for (int r = 0; r < B::NQ; r++) table[r] = place(r);
    }
#pragma unroll
    for (int r = 0; r < B::NP; r++) {
      const int p = threadIdx.x + 64 * r, ci = p % B::W, row = p / B::W, ck = AB ? S : row % B::NL, cj = row / B::NL;
      cube[r] = p < B::P ? row * B::NC + ci - S : 0;
      dist[r] = p < B::P ? max(abs(ci - S), max(abs(ck - S), abs(cj - S))) : 0;
    }
  }
  // Box cell r: its element from the window's first cell.
  __device__ __forceinline__ long off(const IlmcArgs& A, int r) const {
    const int w = at(r);
    return (w & 255) - S + A.nx * ((w >> 16) - S) + A.nxy * (((w >> 8) & 255) - S);
  }
  // Is box cell r of window x in the domain?
  __device__ __forceinline__ bool in(const IlmcArgs& A, const IlWindow& x, int r) const {
    const int w = at(r);
    const int di = x.di + (w & 255) - S, dk = x.dk + ((w >> 8) & 255) - S, dj = x.dj + (w >> 16) - S;
    return (unsigned)di < (unsigned)A.ni && (unsigned)dj < (unsigned)A.nj && (unsigned)dk < (unsigned)A.nkk &&
           threadIdx.x + 64 * r < B::N;
  }
};

typedef ADZ_GLOBAL float* IlPtr;
typedef const ADZ_GLOBAL float* IlCPtr;

// What no visit changes: bounds and air mass.
template <int S, bool AB>
__device__ __forceinline__ void il_fetch(const IlmcArgs& A, const IlmcTr& T, const IlWindow& x, const IlLane<S, AB>& K,
                                         IlBox<S, AB>& L) {
  typedef IlBox<S, AB> B;
  const long q0 = x.row0 + x.di;
#pragma unroll(B::kUnroll)
  for (int r = 0; r < B::NQ; r++) {
    float mn = 0.f, mx = 0.f, air = 0.f;
    if (K.in(A, x, r)) {
      mn = ((IlCPtr)T.mn)[q0 + K.off(A, r)];
      mx = ((IlCPtr)T.mx)[q0 + K.off(A, r)];
      air = ((IlCPtr)A.air)[q0 + K.off(A, r)];
    }
    const int e = threadIdx.x + 64 * r;
    if (e < B::N) { L.mn[e] = mn; L.mx[e] = mx; L.air[e] = air; }
  }
}

// One sweep of the visit of a cell (ilmc_lam_loop.inc:30-76, :82-128): true if it moved mass.
// `mass(p)` gives the cube's masses; f, bnd and w are those of the lane's cube cells.
template <int s, int S, bool AB, class Mass>
__device__ __forceinline__ bool il_sweep(IlBox<S, AB>& L, const IlLane<S, AB>& K, int c, const Mass& mass, const float* f,
                                         const float* bnd, const float* w, bool over, float& fc, float& o, float& u,
                                         float mnc, float mxc, float airc) {
  typedef IlBox<S, AB> B;
  float msum = 0.f;  // :34-45 (:86-97): masses in the sweep's order
  auto row = [&](int ej, bool edge) {
#pragma unroll
    for (int ek = AB ? 0 : -s; ek <= (AB ? 0 : s); ek++) {
      const bool whole = edge || (!AB && (ek == s || ek == -s));
#pragma unroll
      for (int ei = -s; ei <= s; ei++)
        if (whole || ei == s || ei == -s) msum = mass(((ej + S) * B::NL + (AB ? 0 : ek + S)) * B::W + ei + S) + msum;
    }
  };
  row(-s, true);
#pragma unroll(B::kHeld ? 2 * s : 1)
  for (int ej = 1 - s; ej < s; ej++) row(ej, false);
  row(s, true);
  const float m_use = il_min(msum, (over ? o : u) * airc);  // :47 (:99)
  if (!(m_use > 0.f)) return false;                         // :51 (:103)
  if (over) {
    fc = il_max(fc - m_use / airc, mnc);
    o = il_max(0.f, fc - mxc);
  } else {
    fc = il_min(fc + m_use / airc, mxc);
    u = il_max(0.f, mnc - fc);
  }
  const float ratio = m_use / msum;
#pragma unroll
  for (int r = 0; r < B::NP; r++)
    if (K.dist[r] == s && w[r] > 0.f)
      L.f[K.cube[r] + c] = over ? il_min(f[r] + w[r] * ratio, bnd[r]) : il_max(f[r] - w[r] * ratio, bnd[r]);
  return true;
}

// The visits of a window's marked cells, in order, at the present values; the cells they
// changed are written back.  Returns the number of sweeps that moved mass.
template <int S, bool AB>
__device__ __forceinline__ int il_visit(const IlmcArgs& A, const IlmcTr& T, const IlWindow& x, unsigned marked,
                                        const IlLane<S, AB>& K, IlBox<S, AB>& L) {
  typedef IlBox<S, AB> B;
  const IlPtr tf = (IlPtr)T.f + x.row0 + x.di;
  constexpr int kG = B::kHeld ? B::NQ : 4;  // loads in flight
#pragma unroll 1
  for (int r0 = 0; r0 < B::NQ; r0 += kG) {
    float v[kG];
#pragma unroll
    for (int g = 0; g < kG; g++) {
      v[g] = 0.f;
      if (r0 + g < B::NQ && K.in(A, x, r0 + g)) v[g] = il_load(tf + K.off(A, r0 + g));
    }
#pragma unroll
    for (int g = 0; g < kG; g++) {
      const int e = threadIdx.x + 64 * (r0 + g);
      if (e < B::N) L.f[e] = L.was[e] = v[g];
    }
  }
  __syncthreads();
  int moved = 0;
  for (; marked; marked &= marked - 1) {
    const int c = __ffs((int)marked) - 1 + S, ec = (S * B::NL + (AB ? 0 : S)) * B::NC + c;
    float fc = L.f[ec];
    const float mnc = L.mn[ec], mxc = L.mx[ec], airc = L.air[ec];
    float o = il_max(0.f, fc - mxc), u = il_max(0.f, mnc - fc);  // :23-26
    if (o == 0.f && u == 0.f) continue;                          // put back in bounds by earlier visits
    const bool over = o > 0.f;
    float f[B::NP], bnd[B::NP], w[B::NP];
#pragma unroll
    for (int r = 0; r < B::NP; r++) {
      const int e = K.cube[r] + c, p = threadIdx.x + 64 * r;
      f[r] = L.f[e];
      bnd[r] = over ? L.mx[e] : L.mn[e];
      w[r] = over ? il_max(0.f, bnd[r] - f[r]) : il_max(0.f, f[r] - bnd[r]);
      if (p < B::P) L.mass[p] = w[r] * L.air[e];
    }
    __syncthreads();
    // a sweep that leaves the cell in bounds ends the visit: the next would compute
    // m_use = min(m_sweep, 0) and move nothing (:47, :51)
    int m = 0;
    auto sweeps = [&](auto mass) {
      m = il_sweep<1, S, AB>(L, K, c, mass, f, bnd, w, over, fc, o, u, mnc, mxc, airc);
      if constexpr (S >= 2)
        if ((over ? o : u) != 0.f) m += il_sweep<2, S, AB>(L, K, c, mass, f, bnd, w, over, fc, o, u, mnc, mxc, airc);
      if constexpr (S >= 3)
        if ((over ? o : u) != 0.f) m += il_sweep<3, S, AB>(L, K, c, mass, f, bnd, w, over, fc, o, u, mnc, mxc, airc);
      if constexpr (S >= 4)
        if ((over ? o : u) != 0.f) m += il_sweep<4, S, AB>(L, K, c, mass, f, bnd, w, over, fc, o, u, mnc, mxc, airc);
    };
    if constexpr (B::kHeld) {
      typedef float f32x4 __attribute__((ext_vector_type(4)));
      f32x4 v[(B::P + 3) / 4];
#pragma unroll
      for (int q = 0; q < (B::P + 3) / 4; q++) v[q] = ((const f32x4*)L.mass)[q];
      sweeps([&](int p) { return v[p / 4][p % 4]; });
    } else {
      sweeps([&](int p) { return L.mass[p]; });
    }
    if (m && threadIdx.x == 0) L.f[ec] = fc;
    moved += m;
    __syncthreads();
  }
#pragma unroll(B::kUnroll)
  for (int r = 0; r < B::NQ; r++) {
    if (K.in(A, x, r)) {
      const float f = L.f[threadIdx.x + 64 * r], w = L.was[threadIdx.x + 64 * r];
      if (__builtin_bit_cast(unsigned, f) != __builtin_bit_cast(unsigned, w)) il_store(tf + K.off(A, r), f);
    }
  }
  __syncthreads();  // the box is reused by the next window
  return moved;
}

// The visits: single-wave blocks take windows from the ticket counter until none is left or
// a wait gave up.  128 waves per tracer, and where that is more, three for every window that the
// values of t have on average, as many as their order lets run at a time; others would only poll.
// ms, with 128 (256, 512, 1024) waves: two tracers of 384 x 288 x 84 with a front 7.3 (7.6, 8.0,
// 8.7), one of 100 x 80 x 40 with 30 % of the cells out of bounds 2.2 (1.9, 3.3, 3.9), one of
// 512 x 384 x 84 with 2 % 9.1 (4.8, 3.5, 4.2), with 30 % 98 (50, 34, 35; 61 as a launch per
// hyperplane).
template <int S, bool AB>
__global__ __launch_bounds__(64) void k_il_visit(IlmcArgs A) {
  __shared__ IlBox<S, AB> L;
  __shared__ long long ticket;
  IlLane<S, AB> K;
  K.init();
  const int lane = threadIdx.x;
  const long long total = A.off[A.nplanes];
  if (blockIdx.x >= (long long)kIlFew * A.ntr && blockIdx.x >= 3 * total / A.nplanes) return;
  for (;;) {
    // through LDS and barriers: a readfirstlane here would hang on where the lanes reconverge
    // after the branches on lane 0
    __syncthreads();
    if (lane == 0) ticket = (long long)atomicAdd(A.ctl, 1ull);
    __syncthreads();
    const long long e = ticket;
    if (e >= total) return;
    const IlWindow x = il_window(A, A.list[e]);
    const IlmcTr T = A.tr[x.n];
    const unsigned marked = (unsigned)((il_load(x.pend) >> (x.di & 63)) & kIlMask);
    il_fetch<S, AB>(A, T, x, K, L);
    if (!il_wait<S, AB>(A, x)) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");  // f is loaded after the polls came back clear
    const int moved = il_visit<S, AB>(A, T, x, marked, K, L);
    // the window's values are out before its bits go: the stores of f, agent-scope atomics that
    // go through to where every XCD sees them, have been acknowledged
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    if (lane == 0) {
      __hip_atomic_fetch_and(x.pend, ~((uint64_t)marked << (x.di & 63)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (A.counts && moved) atomicAdd((unsigned long long*)&A.counts[3 * x.n], (unsigned long long)moved);
    }
  }
}

// What follows the visits.  If a wait gave up, block 0 first visits the windows still
// pending, in list order, and the other blocks leave.  Then the reset to [min, max]
// (ILMC_LAM.F90:249-273) and its counts: only cells that were out of bounds before the first
// visit can be so now, so the reset goes over the listed windows, 16 to a wave.
template <int S, bool AB>
__global__ __launch_bounds__(64) void k_il_finish(IlmcArgs A, int reset) {
  __shared__ IlBox<S, AB> L;
  const int lane = threadIdx.x;
  const long long total = A.off[A.nplanes];
  long long step = gridDim.x;
  if (A.ctl[1]) {
    if (blockIdx.x) return;
    step = 1;
    IlLane<S, AB> K;
    K.init();
    for (long long e = 0; e < total; e++) {
      const IlWindow x = il_window(A, A.list[e]);
      const unsigned marked = (unsigned)((*x.pend >> (x.di & 63)) & kIlMask);
      if (!marked) continue;
      const IlmcTr T = A.tr[x.n];
      il_fetch<S, AB>(A, T, x, K, L);
      const int moved = il_visit<S, AB>(A, T, x, marked, K, L);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (A.counts && lane == 0 && moved) atomicAdd((unsigned long long*)&A.counts[3 * x.n], (unsigned long long)moved);
    }
  }
  if (!reset) return;
  constexpr int kPer = 64 / kIlWin;
  for (long long b = (long long)blockIdx.x * kPer; b < total; b += step * kPer) {
    const long long e = b + lane / kIlWin;
    int n = -1;
    bool lo = false, hi = false;
    if (e < total) {
      const IlWindow x = il_window(A, A.list[e]);
      const int di = x.di + lane % kIlWin;
      n = x.n;
      if (di < A.ni) {
        const IlmcTr T = A.tr[n];
        const long c = x.row0 + di;
        float f = il_load(T.f + c);
        const float mn = T.mn[c], mx = T.mx[c];
        lo = f < mn;
        if (lo) f = mn;
        hi = f > mx;
        if (hi) f = mx;
        if (lo || hi) T.f[c] = f;
      }
    }
    if (!A.counts) continue;
    for (unsigned long long todo = __ballot(lo || hi); todo;) {  // one add per tracer and wave
      const int l = __ffsll(todo) - 1, nl = __builtin_amdgcn_readlane(n, l);
      const unsigned long long same = __ballot(n == nl);
      const int a = __popcll(__ballot(lo) & same), c = __popcll(__ballot(hi) & same);
      if (lane == l) {
        if (a) atomicAdd((unsigned long long*)&A.counts[3 * nl + 1], (unsigned long long)a);
        if (c) atomicAdd((unsigned long long*)&A.counts[3 * nl + 2], (unsigned long long)c);
      }
      todo &= ~same;
    }
  }
}

}  // namespace adz

using namespace adz;

struct adz_ilmc {
  IlmcArgs a;
  int sweep_max, autobar, min_max;
  void* mem;
};

namespace {

template <int S, bool AB>
void launch_visits(const IlmcArgs& a, int reset, hipStream_t st) {
  hipLaunchKernelGGL((k_il_visit<S, AB>), dim3(kIlWaves), dim3(64), 0, st, a);
  hipLaunchKernelGGL((k_il_finish<S, AB>), dim3(kIlWaves), dim3(64), 0, st, a, reset);
}

}  // namespace

extern "C" {

int adz_ilmc_create(const adz_ilmc_tracer* tr, int ntr, const adz_ilmc_domain* dom, adz_ilmc** out) {
  if (!tr || ntr <= 0 || !dom || !out) return fail(ADZ_EINVAL, "adz_ilmc_create: bad argument");
  const adz_ilmc_domain& d = *dom;
  if (d.in < d.i0 || d.jn < d.j0 || d.nk < d.k0 || d.i0 < d.minx || d.in > d.maxx || d.j0 < d.miny ||
      d.jn > d.maxy || d.k0 < 1)
    return fail(ADZ_EINVAL, "adz_ilmc_create: domain outside the arrays");
  if (d.sweep_max < 1 || d.sweep_max > 4)
    return fail(ADZ_EINVAL, "adz_ilmc_create: ILMC_sweep_max must be 1..4 (the sweep arrays hold 400 cells)");
  const int ni = d.in - d.i0 + 1, nj = d.jn - d.j0 + 1, nkk = d.nk - d.k0 + 1;
  // window and row offsets are packed in 16 bits each, levels in 12, tracers in the remaining 20;
  // k_il_mark launches a 256-lane block for every few rows of the domain (at most 2^32 lanes)
  if (ni > 65535 || nj > 65535 || nkk > 4095 || ntr > 65535 || (long)nj * nkk > (1L << 24))
    return fail(ADZ_EINVAL, "adz_ilmc_create: domain or tracer count too large");
  std::vector<IlmcTr> h(ntr);
  for (int n = 0; n < ntr; n++) {
    if (!tr[n].f || !tr[n].mn || !tr[n].mx) return fail(ADZ_EINVAL, "adz_ilmc_create: null tracer array");
    h[n] = IlmcTr{(float*)tr[n].f, (const float*)tr[n].mn, (const float*)tr[n].mx};
  }
  IlmcArgs a;
  std::memset(&a, 0, sizeof(a));
  a.ntr = ntr;
  a.nx = d.maxx - d.minx + 1;
  a.nxy = a.nx * (long)(d.maxy - d.miny + 1);
  a.i0 = d.i0; a.j0 = d.j0; a.k0 = d.k0; a.ni = ni; a.nj = nj; a.nkk = nkk;
  const int reach = (2 * d.sweep_max + kIlWin - 1) / kIlWin;  // windows to the left or right
  a.a = reach + 1;
  a.b = d.autobar ? 0 : reach + a.a * 2 * d.sweep_max + 1;
  const int nwin = (ni + kIlWin - 1) / kIlWin;
  const long np = (long)(nwin - 1) + (long)a.a * (nj - 1) + (long)a.b * (nkk - 1) + 1;
  const long cap = (long)ntr * nwin * nj * nkk;
  if (np > (1L << 30)) return fail(ADZ_EINVAL, "adz_ilmc_create: domain too large");
  a.nplanes = (int)np;
  const size_t tb = (sizeof(IlmcTr) * ntr + 255) / 256 * 256;
  const size_t cb = (sizeof(long long) * (np + 2) + 255) / 256 * 256, ob = (sizeof(long long) * (np + 1) + 255) / 256 * 256;
  const size_t lb = sizeof(uint64_t) * cap;
  a.wpr = (ni + 63) / 64;
  const size_t wb = sizeof(uint64_t) * (size_t)ntr * nj * nkk * a.wpr;
  void* mem = nullptr;
  if (hipMalloc(&mem, tb + cb + ob + lb + wb) != hipSuccess) return fail(ADZ_ENOMEM, "adz_ilmc_create: hipMalloc");
  if (hipMemcpy(mem, h.data(), sizeof(IlmcTr) * ntr, hipMemcpyHostToDevice) != hipSuccess) {
    (void)hipFree(mem);
    return fail(ADZ_EHIP, "adz_ilmc_create: upload");
  }
  char* p = (char*)mem;
  a.tr = (const IlmcTr*)p;
  a.cnt = (unsigned long long*)(p + tb);
  a.ctl = a.cnt + np;
  a.off = (long long*)(p + tb + cb);
  a.list = (uint64_t*)(p + tb + cb + ob);
  a.pend = (uint64_t*)(p + tb + cb + ob + lb);
  a.spin_limit = kIlSpin;
  adz_ilmc* r = new adz_ilmc;
  r->a = a;
  r->sweep_max = d.sweep_max; r->autobar = d.autobar != 0; r->min_max = d.min_max != 0;
  r->mem = mem;
  *out = r;
  return ADZ_OK;
}

int adz_ilmc_lam(adz_ilmc* il, const void* air_m, long long* counts, adz_stream stream) {
  if (!il || !air_m) return fail(ADZ_EINVAL, "adz_ilmc_lam: null argument");
  hipStream_t st = (hipStream_t)stream;
  IlmcArgs a = il->a;
  a.air = (const float*)air_m;
  a.counts = counts;
  const long nz = (long)a.nplanes + 2, nc = counts ? 3L * a.ntr : 0;  // cnt and, behind it, ctl; counts
  hipLaunchKernelGGL(k_il_zero, dim3((unsigned)((std::max(nz, nc) + kIlBlock - 1) / kIlBlock)), dim3(kIlBlock), 0, st,
                     (long long*)a.cnt, nz, counts, nc);
  const int nrows = a.nj * a.nkk, rows = std::max(1, kIlBlock / 64 * kIlUnroll / a.wpr);
  hipLaunchKernelGGL(k_il_mark, dim3((unsigned)((nrows + rows - 1) / rows), (unsigned)a.ntr), dim3(kIlBlock), 0, st, a,
                     rows);
  hipLaunchKernelGGL(k_il_scan, dim3(1), dim3(kIlScan), 0, st, a);
  hipLaunchKernelGGL(k_il_fill, dim3((unsigned)(((long)nrows * a.wpr + kIlBlock - 1) / kIlBlock), (unsigned)a.ntr),
                     dim3(kIlBlock), 0, st, a);
  const int reset = il->min_max;
  switch (il->sweep_max * 2 + il->autobar) {
    case 2: launch_visits<1, false>(a, reset, st); break;
    case 3: launch_visits<1, true>(a, reset, st); break;
    case 4: launch_visits<2, false>(a, reset, st); break;
    case 5: launch_visits<2, true>(a, reset, st); break;
    case 6: launch_visits<3, false>(a, reset, st); break;
    case 7: launch_visits<3, true>(a, reset, st); break;
    case 8: launch_visits<4, false>(a, reset, st); break;
    default: launch_visits<4, true>(a, reset, st); break;
  }
  ADZ_HIP_CHECK(hipGetLastError());
  return ADZ_OK;
}

int adz_ilmc_set_spin_limit(adz_ilmc* il, int polls) {
  if (!il || polls < 0) return fail(ADZ_EINVAL, "adz_ilmc_set_spin_limit: bad argument");
  il->a.spin_limit = polls;
  return ADZ_OK;
}

int adz_ilmc_free(adz_ilmc* il) {
  if (!il) return ADZ_OK;
  hipError_t e = hipFree(il->mem);
  delete il;
  if (e != hipSuccess) return fail(ADZ_EHIP, "adz_ilmc_free: hipFree");
  return ADZ_OK;
}

}  // extern "C"
