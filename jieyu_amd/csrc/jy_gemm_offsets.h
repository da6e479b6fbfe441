// jy_gemm_offsets.h — where the matrix-core prompt GEMM (jy_gemm_mfma.hip) reads a matrix's copy
// (Q8MfmaDev): plain C++, so that the same arithmetic can be checked over whole grids on the host.
#pragma once

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>

#define JY_HD __host__ __device__ __forceinline__
#else
#define JY_HD inline
#endif

namespace jy {

// Every offset lies inside the copy by itself: waves past the last column tile, the second tile
// of a pair and the blocks of a step past the matrix (and of the step after the last one, whose
// loads are issued and never used) read the last tile or block there is.  The buffer
// descriptor's range check is not relied on: the scalar offset is no part of it.
//
// A load = base of tile gm_base_tile + lane part (a vector register per 32-column tile) +
// block part (scalar).

JY_HD int gm_min(int a, int b) { return a < b ? a : b; }

// tilet: the wave's first 16-column tile
JY_HD int gm_base_tile(int tilet, int tiles) { return gm_min(tilet, tiles - 1); }

// tiles past the base of lane l's column in the wave's nt-th 32-column tile
JY_HD int gm_lane_tile(int tilet, int nt, int l, int tiles) {
    return gm_min(tilet + 2 * nt + ((l & 31) >> 4), tiles - 1) - gm_base_tile(tilet, tiles);
}

// weights, bytes: slot l % 16 + 16 (l / 32) of block b (the lane's halves of 16 k: jy_gemm_mfma.hip)
JY_HD int gm_q_lane(int tilet, int nt, int l, int tiles, int nb) {
    return gm_lane_tile(tilet, nt, l, tiles) * nb * 512 + (l & 15) * 16 + 256 * (l >> 5);
}
JY_HD int gm_q_block(int b, int nb) { return gm_min(b, nb - 1) * 512; }

// scales, bytes: row l % 16 of the four blocks around b
JY_HD int gm_d_lane(int tilet, int nt, int l, int tiles, int nb4) {
    return gm_lane_tile(tilet, nt, l, tiles) * nb4 * 256 + (l & 15) * 16;
}
JY_HD int gm_d_block(int b, int nb4) { return gm_min(b >> 2, nb4 - 1) * 256; }

}  // namespace jy
