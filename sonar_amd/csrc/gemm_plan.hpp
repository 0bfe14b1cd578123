// Which kernel a dense call takes and how much scratch it needs: shared by the
// dispatcher, the tile kernels and sonar_marlin_gemm_scratch_bytes.
#pragma once

#include <stdint.h>

namespace sonar {

struct GemmPlan {
  bool tile;        // MFMA-tiled kernel (else the streaming kernels, in 64-row slabs)
  int tile_rows;    // rows of a tile: 256, or 128 (the wide tile kernel's form for calls with few tiles)
  int k_splits;     // workgroups per split tile along K (tile kernel only)
  int k_steps_per_split;
  // With k_splits > 1: the first `whole_tiles` tiles of the tile numbering are
  // each computed by one workgroup over the whole of K, the rest are split.
  int64_t whole_tiles;
};

// 97..128 rows on a matrix with more strips than compute units (N > 16384) and K <= 8192: the wide tile
// kernel's 128-row form with K in two ranges is ahead of blocks of rows in the decode kernel (measured at
// K = 4096, N = 28672: M = 128: 45 us against 55; M = 72 and 96: level; with 64 to 96 strips, N = 4096 / 6144,
// the decode kernel is two times ahead).  `wide128`: the call is one that form takes (4-bit integer codes
// with groups of 64 * 2^i rows or one group, no act-order gather).
inline bool plan_rows_97_128(int64_t size_m, int64_t size_n, int64_t size_k, bool wide128) {
  // (up to 128 tiles of 256 columns: beyond that K is not split and the tile kernel is not planned)
  return wide128 && size_m > 96 && size_m <= 128 && size_n > 16384 && size_n <= 32768 && size_k <= 8192 &&
         size_k % 256 == 0;
}

inline GemmPlan plan_gemm(int64_t size_m, int64_t size_n, int64_t size_k, bool async_tile, int tile_rows = 256,
                          bool rows_97_128 = false) {
  GemmPlan plan = {false, tile_rows, 1, 0, 0};
  if (size_m <= 64 || size_k % 64 != 0) return plan;
  const int64_t tiles = ((size_m + tile_rows - 1) / tile_rows) * ((size_n + 255) / 256);
  const int k_steps = (int)(size_k / 64);
  plan.k_steps_per_split = k_steps;
  // Few tiles leave compute units idle: split K so that about 256 workgroups
  // run, each with at least eight K steps.  Partial tiles cost 256 KiB of
  // fp32 traffic each way (128 with 128-row tiles), so up to 128 rows the streaming kernels
  // stay ahead.
  int splits = 1;
  if (async_tile && tiles < 256) {
    splits = (int)(256 / tiles);
    if (splits > k_steps / 8) splits = k_steps / 8;
    if (splits > 16) splits = 16;
    if (splits < 1) splits = 1;
  }
  // More tiles than compute units, the last round of workgroups a half or less
  // of the chip: split the tiles of that round so that it is as wide as the
  // others and 1 / splits as long.  Worth the partial-tile traffic (at most
  // 64 MiB each way, about 30 us) once a tile takes about 80 us (48 K steps).
  int64_t whole_tiles = 0;
  if (async_tile && tiles > 256 && k_steps >= 48) {
    const int64_t last_round = tiles % 256;
    if (last_round != 0 && last_round <= 128) {
      splits = (int)(256 / last_round);
      if (splits > k_steps / 8) splits = k_steps / 8;
      if (splits > 16) splits = 16;
      if (splits < 2) splits = 1;
      else whole_tiles = tiles - last_round;
    }
  }
  // (with a long K the partial tiles are a small part of the work: measured at K = 14336, N = 4096,
  // M = 96 / 128: 47 / 53 us in slabs)
  if (size_m <= 128 && !(async_tile && (size_k >= 8192 || rows_97_128) && splits > 1)) return plan;
  if (splits == 1 && size_m <= 512 && tiles < 64) return plan;  // slabs use every compute unit
  plan.tile = true;
  plan.k_splits = splits;
  plan.k_steps_per_split = (k_steps + splits - 1) / splits;
  // ranges of a multiple of four steps, a whole pass of the wide tile kernel's loop, where K allows it
  if (k_steps % 4 == 0) plan.k_steps_per_split = (plan.k_steps_per_split + 3) / 4 * 4;
  plan.k_splits = (k_steps + plan.k_steps_per_split - 1) / plan.k_steps_per_split;  // no empty split
  plan.whole_tiles = plan.k_splits > 1 ? whole_tiles : tiles;
  return plan;
}

inline size_t plan_partial_bytes(const GemmPlan& plan, int64_t size_m, int64_t size_n) {
  if (!plan.tile || plan.k_splits <= 1) return 0;
  const int64_t tiles = ((size_m + plan.tile_rows - 1) / plan.tile_rows) * ((size_n + 255) / 256);
  return (size_t)plan.k_splits * (size_t)(tiles - plan.whole_tiles) * plan.tile_rows * 1024;
}

// The 128-row form pays when 256-row tiles would leave more than half of the compute units to
// K ranges of the same tile: twice the tiles, half the ranges, half the partial-tile bytes.  With
// a long K the partial tiles are a smaller part of the work and the larger tile is ahead again
// from 48 tiles on (measured at K = 14336, N = 4096, 128-row against 256-row tiles: M = 256:
// 44.4 against 50.9 us; 384: 62.0 against 75.4; 512: 72.7 against 74.6; 768: 109 against 101;
// 1024: 126 against 120).
inline bool plan_prefers_128_rows(int64_t size_m, int64_t size_n, int64_t size_k) {
  const int64_t tiles256 = ((size_m + 255) / 256) * ((size_n + 255) / 256);
  // up to 128 rows (calls that plan_gemm gives to the tile kernel at all: a long K, or rows_97_128) half of a
  // 256-row tile would be padding (K = 14336, N = 4096, M = 72 / 96 / 128: 47.3 / 47.8 / 49.0 -> 29.8 / 30.0 /
  // 30.0 us; K = 8192, N = 8192, M = 65 / 128: 54.4 / 52.9 -> 32.3 / 32.7)
  if (size_m <= 128) return size_m > 64 && tiles256 <= 128;
  return tiles256 <= (size_k <= 8192 ? 128 : 32);
}

// Whether the 64 rows of a dense call's A that a wavefront of the wide tile kernel copies are within 32-bit offsets of the first.
// (The other tile kernels have 64-bit addresses.)
inline bool wide_rows_within_32_bits(int64_t a_row_stride) { return a_row_stride < (int64_t)1 << 25; }

// What the tile kernels are launched with, given room for the partial tiles.  `rows128`: the call's format has 128-row tiles.
inline GemmPlan tile_plan(int64_t size_m, int64_t size_n, int64_t size_k, bool rows128, bool rows_97_128) {
  if (rows128 && plan_prefers_128_rows(size_m, size_n, size_k)) {
    const GemmPlan plan = plan_gemm(size_m, size_n, size_k, true, 128, rows_97_128);
    if (plan.tile) return plan;
  }
  return plan_gemm(size_m, size_n, size_k, true, 256, rows_97_128);
}

constexpr double kTileStepInt4 = 1.21, kTileStepMxFp4 = 1.14;   // `step` of tile_estimate

// Microseconds the tile kernels take: rounds of workgroups, each 11.2 us around its loop and `step` us per 64 rows of K for a
// 256-row tile (0.58 of both for a 128-row one), 3.3 us for the launch, and for K in ranges a second launch and its bytes.  A fit
// of 168 random calls of 220 to 8192 rows in all formats: 90 % within 14 % below and 13 % above.
inline double tile_estimate(int64_t size_m, int64_t size_n, int64_t size_k, double step, bool rows128, bool rows_97_128) {
  const GemmPlan plan = tile_plan(size_m, size_n, size_k, rows128, rows_97_128);
  const bool small = plan.tile_rows == 128;
  const int64_t rows = plan.tile_rows, steps = size_k / 64, tiles = ((size_m + rows - 1) / rows) * ((size_n + 255) / 256);
  const double unit = small ? 0.58 : 1.0, whole = unit * (step * steps + 11.2);
  const double range = unit * (step * plan.k_steps_per_split + 11.2), sum = 1.1 + 1.24e-6 * plan.k_splits * size_m * size_n;
  if (plan.k_splits > 1 && plan.whole_tiles == 0) return 3.3 + (tiles * plan.k_splits + 255) / 256 * range + sum;
  const int64_t last = tiles % 256;
  double us = 3.3 + tiles / 256 * whole;
  if (last > 128 || (last > 0 && plan.k_splits < 3 && (tiles < 256 || !rows128))) us += whole;
  else if (last > 0) us += plan.k_splits >= 3 ? range + 1.1 : 0.58 * whole;
  return us;
}

// Microseconds of marlin_tile_twin_kernel (128-row tiles over the whole of K, two at a time on a compute unit): so many pairs of tiles
// as a compute unit gets, and a single one where their number is odd.  A fit of 156 random calls of 256 to 8192 rows, K = 512 to
// 7168: 80 % within 9 %.  Taken where this is below tile_estimate, it is 0.7 % (float16), 1.0 % (bfloat16 integers) and 0.1 % (MXFP4)
// above the better of the two on those, no call more than 1.7 % slower than before.
inline double twin_estimate(int64_t size_m, int64_t size_n, int64_t size_k, bool float16, bool fp4) {
  const double pair_step = fp4 ? 1.25 : float16 ? 1.34 : 1.41, one_step = fp4 ? 0.78 : float16 ? 0.93 : 1.02;
  const int64_t steps = size_k / 64, tiles = ((size_m + 127) / 128) * ((size_n + 255) / 256), most = (tiles + 255) / 256;
  return 3.3 + most / 2 * (pair_step * steps + 6.4) + most % 2 * (one_step * steps + 1.0);
}
// Whether a dense call that could have such tiles has them: where 256-row tiles would run otherwise (more than half a round of them),
// and the estimates say so; by 3 % where it is at most one round of them, as both take a round then (M = 2834, K = 2304, N = 4352, AWQ,
// fp16: 56.5 us there, 58.8 here; M = 2755, K = 1664, N = 3712, groups of 32 39.5 / 41.0).  On 246 random calls in turn with the
// tree before, 0.965 times the time: M = 332, K = 3200, N = 17728, AWQ, fp16 (140 tiles of 256 rows, 210 of 128) 64.5 -> 43.0; M = 855,
// K = 1024, N = 17472, MXFP4 (276 / 483) 48.2 -> 32.4; M = 4000, K = 512, N = 28672 148 -> 115; M = 569, K = 2944, N = 24512, bf16 110 -> 75.
inline bool twin_pays(int64_t size_m, int64_t size_n, int64_t size_k, bool float16, bool fp4, bool rows128, bool rows_97_128) {
  const double least = ((size_m + 255) / 256) * ((size_n + 255) / 256) <= 256 ? 0.97 : 1.0;
  return tile_plan(size_m, size_n, size_k, rows128, rows_97_128).tile_rows == 256 &&
         twin_estimate(size_m, size_n, size_k, float16, fp4) <
             least * tile_estimate(size_m, size_n, size_k, fp4 ? kTileStepMxFp4 : kTileStepInt4, rows128, rows_97_128);
}

// Scratch for the partial tiles of either tiling.
inline size_t plan_partial_bytes_any(int64_t size_m, int64_t size_n, int64_t size_k) {
  const bool r = plan_rows_97_128(size_m, size_n, size_k, true);
  const size_t a = plan_partial_bytes(plan_gemm(size_m, size_n, size_k, true, 256, r), size_m, size_n);
  const size_t b = plan_partial_bytes(plan_gemm(size_m, size_n, size_k, true, 128, r), size_m, size_n);
  return a > b ? a : b;
}

}  // namespace sonar
