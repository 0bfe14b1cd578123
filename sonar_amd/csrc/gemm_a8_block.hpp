// Interface of gemm_a8_block.hip to the dispatcher of the W4A8 calls (gemm_a8.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sonar {

struct A8BlockParams {
  const uint8_t* a;          // [M] rows of K bytes, `lda` apart
  long lda;
  uint16_t* c;               // [M][N], float16 or bfloat16
  const uint32_t* w;         // gfx950 order
  const uint16_t* scales;    // [groups][N], single-permuted inside every 32 columns
  const uint32_t* zeros;     // [groups][N/8] or null
  const float* a_scales;     // [M]
  const uint16_t* bias;      // [N], permuted like the scales, or null
  int size_m, size_n, size_k;
  int group_chunks;          // 32-row chunks per group: 1 (int8 only), 2, 4; 0: channelwise
  int bf16;                  // output (and scale) type
  uint32_t* partial;         // [splits][M][N] raw totals when splits > 1
  int tiles_m, tiles, splits, split_steps;   // filled in by a8_block_gemm
};

// Tile of a workgroup: 32 * rows rows of C, 64 * strips columns, K in `ranges` parts; K split over `splits` workgroups,
// whose raw totals the caller adds.
struct A8BlockShape {
  int rows, strips, ranges, splits;
};

// Most row blocks whose tiles are built: what 256 registers hold.  (More scales in flight with small groups.)
constexpr int a8_max_row_blocks(bool fp8, bool zero_points, int group_chunks) {
  if (group_chunks == 0 || (group_chunks == 4 && !fp8 && !zero_points)) return 4;
  return group_chunks == 1 && zero_points ? 2 : 3;
}

int a8_block_gemm(A8BlockParams p, bool fp8, A8BlockShape shape, hipStream_t st);

}  // namespace sonar
