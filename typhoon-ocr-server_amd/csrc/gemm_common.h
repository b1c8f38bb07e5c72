// gemm_common.h -- device-side pieces shared by the tiled GEMMs and the kernels
// that write their activations: the plane layout, 16-bit packing, tile order.
#pragma once
#include "tl_common.h"

namespace tl {

// Code row of plane p of token t: 4t + p, or grouped, where row group 4T + p
// holds plane p of tokens 16T .. 16T + 15 (the layout of the quadrant GEMM);
// and the code row groups of `rows` tokens.
__host__ __device__ __forceinline__ int planes_row(int t, int p, bool grouped) {
  return grouped ? 64 * (t >> 4) + 16 * p + (t & 15) : 4 * t + p;
}
__host__ __device__ __forceinline__ int planes_groups(int rows, bool grouped) {
  return grouped ? 4 * cdiv(rows, 16) : cdiv(4 * rows, 16);
}

// two fp32 as packed fp16, rounded to nearest even (v_cvt_pkrtz truncates)
__device__ inline uint32_t pack_f16x2(float a, float b) {
  return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)a) | ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)b) << 16);
}

// Orders a wave's LDS accesses across it: what its lanes wrote before is what
// other lanes of the same wave read after, and no later write moves above an
// earlier read.  (LDS works a wave's accesses off in order, so nothing waits.)
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Tile order of the tiled GEMMs, for any tile counts (work-group b runs on XCD
// b % 8): XCD x owns an eighth of the tiles, consecutive in an order that walks
// bands of gm tile rows column by column, so that the tiles an XCD runs at once
// are a patch of gm rows and its L2 fills gm row panels and as many columns
// (against the int8 LDS-staged kernel's order over a sweep of 130 shapes: 6 %
// faster where the columns divide over the XCDs and tiles number more than 128,
// 10 % where they do not, equal below).
__device__ __forceinline__ void tile_patch(int b, int ntm, int ntn, int gm, int& tm, int& tn) {
  const int n = ntm * ntn, x = b % 8;
  const int u = x * (n / 8) + min(x, n % 8) + b / 8;      // a bijection of [0, n)
  const int grp = u / (gm * ntn), r = u - grp * gm * ntn;
  const int rows = min(gm, ntm - gm * grp);
  tm = gm * grp + r % rows;
  tn = r / rows;
}

}  // namespace tl
