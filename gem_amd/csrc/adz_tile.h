// Pieces shared by the kernels that stage a tile's source box in LDS (gfx950).
#pragma once
#include "adz_common.h"

namespace adz {

// Buffer descriptor of `bytes` bytes from `base`, both wave-uniform: loads beyond them return
// zeros and stores are dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t field_rsrc(const void* base, unsigned bytes) {
  // the field pointer is uniform across the wave: keep the descriptor in SGPRs
  unsigned long long a = (unsigned long long)base;
  unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a), hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
  void* p = (void*)(((unsigned long long)hi << 32) | lo);
  return __builtin_amdgcn_make_buffer_rsrc(p, (short)0, (int)__builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

// Block-wide minimum of 6 values, returned as scalars, with one barrier and no reading of
// other waves' words: each wave reduces by DPP moves (pairs, quads, half-rows, rows of 16, then
// the row broadcasts of 15 and 31 leave the minimum in lane 63), lanes 0..5 of the wave put
// the six into LDS with one min each, and after the barrier lanes 0..5 read them back.  `red`
// holds three sets of 6 words, all `kFar` at first; tile number t uses set t % 3 and clears
// set (t + 1) % 3, which was last read before the barrier of tile t - 1.
constexpr int kFar = 1 << 30;
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ int dpp_min(int v) {
  if constexpr (ROWS == 0xF) return min(v, __builtin_amdgcn_mov_dpp(v, CTRL, 0xF, 0xF, true));
  else return min(v, __builtin_amdgcn_update_dpp(0x7fffffff, v, CTRL, ROWS, 0xF, false));
}
__device__ __forceinline__ void tile_min6(int* v, int* red, unsigned t) {
  const int lane = threadIdx.x & 63;
  int mine = kFar;
#pragma unroll
  for (int q = 0; q < 6; q++) {
    int m = v[q];
    m = dpp_min<0xB1>(m);        // quad_perm [1,0,3,2]
    m = dpp_min<0x4E>(m);        // quad_perm [2,3,0,1]
    m = dpp_min<0x141>(m);       // row_half_mirror
    m = dpp_min<0x140>(m);       // row_mirror
    m = dpp_min<0x142, 0xA>(m);  // row_bcast:15 into rows 1 and 3
    m = dpp_min<0x143, 0xC>(m);  // row_bcast:31 into rows 2 and 3
    int w = __builtin_amdgcn_readlane(m, 63);
    asm volatile("" : "+s"(w));  // here, by every lane: the reduction must not sink into a branch
    mine = lane == q ? w : mine;
  }
  int* set = red + 6 * (t % 3);
  if (lane < 6) atomicMin(set + lane, mine);
  if (threadIdx.x < 6) red[6 * ((t + 1) % 3) + threadIdx.x] = kFar;
  __syncthreads();
  const int r = set[min(lane, 5)];
#pragma unroll
  for (int q = 0; q < 6; q++) v[q] = __builtin_amdgcn_readlane(r, q);
}

// Tile of this block, >= n where it has none: in the order of the blocks, or (chunks) an
// eighth of the list for each of the 8 XCDs, to which the hardware deals blocks in turn.
// The grid has two dimensions, since one holds less than 2^32 threads.
constexpr long kGridX = 1L << 21;  // blocks per row of the grid: a multiple of 8
__device__ __forceinline__ long tile_of_block(long n, int chunks) {
  const long b = (long)blockIdx.y * kGridX + blockIdx.x;
  if (!chunks) return b;
  const long per = (n + 7) / 8, l = b / 8;
  return l < per ? b % 8 * per + l : n;
}
inline dim3 tile_grid(long n) {
  const long b = 8 * ((n + 7) / 8);
  return dim3((unsigned)(b < kGridX ? b : kGridX), (unsigned)((b + kGridX - 1) / kGridX));
}

}  // namespace adz
