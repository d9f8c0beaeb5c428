// Where the mask builder's score kernels want the block means (block_map.hip; the quantisers of sage.hip write them too).
#pragma once
#include "common.h"

namespace sla {

// 16-bit dtypes, head dim 64 or 128: the means are written in the order the matrix products of the scores read them, in whole
// tiles of 32 blocks per head; other dtypes and head dims take rows, and so does a workspace with no room for the tiles.
static inline int score_takes_tiled(int dtype, int D) { return dtype != SLA_F32 && (D == 64 || D == 128); }

// Rows of at most this many key blocks are always scored and selected from in one launch (block_map.hip) and need no memory for
// scores.  (Longer ones up to 256 are where their workgroups are few; their workspace has room for scores all the same.)
constexpr int SELECT_FUSED_N = 128;
static inline bool scores_in_memory(int N, int D) { return N > SELECT_FUSED_N || (D != 64 && D != 128); }

// Operand order: tiles of 32 blocks; per tile and 16 columns a fragment of 64 lanes x 8 elements, lane (r, h) = (block % 32,
// column % 2), element j = columns 16 c + 2 j + h: what lane r + 32 h feeds the 32x32x2 product chain, two columns a step.
static __host__ __device__ __forceinline__ size_t tiled_head(int bh, int nblk, int D) {
  return (size_t)bh * (size_t)((nblk + 31) & ~31) * (size_t)D;
}
static __host__ __device__ __forceinline__ size_t tiled_pos(int blk, int d, int D) {
  return ((size_t)((blk >> 5) * (D >> 4) + (d >> 4)) * 64 + 32 * (d & 1) + (blk & 31)) * 8 + ((d & 15) >> 1);
}

}  // namespace sla
