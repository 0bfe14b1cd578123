// Interface of gemm_mid.hip to the dispatchers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>

#include "gemm_plan.hpp"

namespace sonar {

// Weight formats of the kernel in gemm_mid.hip.
enum MidFormat { kMidInt4 = 0, kMidInt4Zp = 1, kMidInt8 = 2, kMidFp8 = 3, kMidMxFp4 = 4, kMidNvFp4 = 5 };

constexpr int kMidMostSplits = 8;
constexpr int kMidMostRawRows = 4;   // row blocks of a tile with MidParams::raw_codes

struct MidParams {
  const uint16_t* a;
  long lda;                  // elements between rows of a
  uint16_t* c;
  const uint4* b;            // gfx950 streaming order
  const uint16_t* bias;
  const uint16_t* scales;
  const uint32_t* zeros;
  const float* global_scale;   // NVFP4
  int size_m, size_n, size_k, num_groups;
  int group_shift;           // log2 of the 64-row steps per group; -1: groups of 32 or 16 rows
  int chunks_per_strip;
  int cus;                   // compute units
  int splits;                // of K over workgroups; their totals go to `partial` and a second kernel adds them
  float4* partial;           // [splits][M][N / 4]
  // 4-bit integers with one group or groups of 128 * 2^i rows, K % 128 == 0: feed the matrix cores the integers and apply
  // scales to fp32 sums, as the decode kernel does, instead of rounding every scaled weight to 16 bits
  bool raw_codes;
  int tiles_m, tiles, split_steps;   // filled in by mid_gemm
};
// Grouped (mixture-of-experts) calls: a row tile is a block of 32, 48 or 64 slots of one expert.  (Arguments of their own: every
// launch of the dense kernel and of its sum reads its arguments first, and 92 bytes more of them took 0.3 us: 64 rows, K 9600, N 1408, MXFP8 17.2 -> 16.8,
// int4 with groups of 32 15.0 -> 14.5, one scale a column 14.7 -> 14.0; 40 rows, K 6016, N 2048, MXFP8 13.0 -> 12.6.)
struct MidMoe {
  const int32_t* sorted_ids;   // slot -> row id of C (row id / top_k of A), >= rows_total: padding
  const int32_t* expert_ids;   // of a block; not 0 .. num_experts - 1: nothing to do
  const int32_t* num_post_pad;
  const float* topk_weights;
  int block_size, top_k, mul_topk, num_experts, rows_total, sorted_len;
  int a_by_slot;               // row of A = slot (a column-permuted copy made per slot), else row id / top_k
  long expert_b_stride;        // uint4 units between experts in b
  long expert_s_stride, expert_z_stride, expert_bias_stride;   // elements between experts
  // if not null: the gated activation of C, (rows_total, size_n / 2), in place of C.  `gated_halves`: silu_and_mul, a workgroup has
  // as many strips of the gate half as of the up half; else swigluoai, whose gate and up columns alternate
  uint16_t* gated;
  int gated_halves;
  float gated_limit, gated_alpha;
};
struct MidMoeParams : MidParams {
  MidMoe moe;
  int strips_each;   // of a workgroup: filled in by mid_moe_gemm
};

// Whether the kernel can run a call (no act-order gather; rows of a within 4 GiB; groups of 16, 32 or 64 * 2^i rows or
// one group).
inline bool mid_applies(int64_t size_m, int64_t size_k, int64_t lda, int64_t num_groups, int group_size) {
  if (size_k % 64 != 0 || size_m * lda * 2 >= (1LL << 32)) return false;
  if (num_groups == 1 || group_size == 16 || group_size == 32) return true;
  const int per = group_size / 64;
  return group_size % 64 == 0 && (per & (per - 1)) == 0;
}

// Strips of a workgroup, two or four, in a grouped call and in dense 64-row tiles of raw codes with K in one piece.  A round of
// workgroups takes as long as six steps beside its loop (start, first bytes, the sum of the ranges), so that twice the columns and half
// the ranges, whose activations are copied half as often, pay where rounds are many; in whole rounds, less `slack`.
// Grouped calls (slack 0.1, the second blocks of uneven routing counted by mid_moe_strips) are what this was fitted to: both forms of
// 242 GEMMs of 23 to 57 slots an expert (blocks of 48 and 64): 0.5 % slower than the better of the two, two strips always 16 %; at
// worst 1.2 times two strips.
// Dense calls take it as it stands with slack 0, as their tiles are counted and not estimated.  Timed on 150 random calls against the
// tree that had two strips only: it changes 10 of them, to 0.67 to 0.93 times the time.
// Us, two -> four strips: 64 of 56, K = 2304, N = 6656, bf16 346 -> 242; 64 of 49, AWQ, 1664 x 8704 291 -> 220; 32 of 42, 1152 x 15360
// 187 -> 132; 64 of 29, MXFP4, 640 x 2688 51 -> 35; 8 of 49, 1536 x 5888 26.5 -> 21.1; 16 of 52, 1152 x 1536, three quarters of a
// round 14.9 -> 18.0.
inline int mid_strips_by_rounds(double row_tiles, double slack, int64_t size_n, int64_t size_k, bool units, int cus) {
  if (size_k < 512) return 2;   // (not timed)
  double cost[2];
  for (int four = 0; four < 2; ++four) {
    const int64_t across = (size_n / 64 + (four ? 3 : 1)) / (four ? 4 : 2), ranges = four ? 2 : 4;
    int64_t steps = (size_k / 64 + ranges - 1) / ranges;
    if (units) steps = (steps + 1) & ~(int64_t)1;
    cost[four] = std::ceil(row_tiles * across / cus - slack) * (6 + steps);
  }
  return cost[1] < 1.06 * cost[0] ? 4 : 2;
}

// Microseconds a call takes in tiles of the best number of row blocks and splits of K, which are returned in
// `row_blocks` and `splits`.  A fit of measured times (K = 2048 and 4096, N = 2048, 6144 and 20032, 17 to 768 rows, all
// formats, on weights that a cache holds, mostly within 15 %; from memory two rounds of tiles take 15 to 20 % more): 4 us
// around the loop of a round of workgroups, and per 4096 rows of K 1.5 us for a row block's matrix instructions and a time
// that depends on the format for the dequantisation, which the matrix instructions do not hide; more at the clock of a
// full chip than of a half empty one; no less than the weights take from memory.  K is split where the tiles leave
// compute units idle, if the totals fit `room` bytes; the pass that adds them is 3.3 us and its bytes.  `raw_codes` (see
// MidParams) has a fit of its own (K = 1024 to 14336, N = 2048 to 28672, 17 to 256 rows, weights from memory: 90 % within
// 6 % below and 13 % above): fewer instructions a chunk for the dequantisation, more a row block for the fold.  Workgroups of four strips
// (mid_strips_by_rounds) have their own: the fuller their one round, the slower (111 calls of up to 127 rows, K = 512 to 11520, N up to
// 57344, both types, 5.6 % rms; with two strips' term, which grows with the bytes, 8192 x 57344 was put at twice its time and
// 49 rows left for the decode kernel: K = 7424, N = 51968, fp16 94 us there, 65 here).
inline double mid_estimate(int64_t size_m, int64_t size_n, int64_t size_k, int64_t num_groups, int dtype, int format,
                           bool raw_codes, int cus, size_t room, int& row_blocks, int& splits) {
  static const double kDequant[6][2] = {   // float16, bfloat16
      {6.8, 8.8}, {8.3, 10.0}, {6.0, 10.2}, {8.0, 15.5}, {5.3, 5.3}, {9.0, 13.3}};
  const double dequant = kDequant[format][dtype == 0 ? 0 : 1] + (num_groups > 1 && size_k / num_groups == 32 && format != kMidMxFp4 ? 0.8 : 0.0);
  static const double kRaw[2][2][2] = {   // without and with zero points, float16 and bfloat16: a strip's share, a row block's
      {{8.2, 1.83}, {6.2, 2.8}}, {{9.55, 1.77}, {6.7, 2.8}}};
  const double* raw = kRaw[format == kMidInt4Zp][dtype == 0 ? 0 : 1];
  const int64_t steps = size_k / 64;
  const double memory = 4.0 + size_n * size_k * (format == kMidInt8 || format == kMidFp8 ? 1.0 : 0.5) / 4.5e6;
  double best = 1e30;
  for (int mb = 2; mb <= (raw_codes ? kMidMostRawRows : 6); ++mb) {
    const int64_t tiles = ((size_m + 16 * mb - 1) / (16 * mb)) * ((size_n + 127) / 128);
    for (int n = 1; n <= kMidMostSplits; ++n) {
      if (n > 1 && (tiles * n > cus || steps < 8 * n || (size_t)n * size_m * size_n * 4 > room)) break;
      const double k = (raw_codes ? 2 * (((steps / 2 + n - 1) / n + 3) / 4) : ((steps + n - 1) / n + 3) / 4) * 256 / 4096.0;
      const int64_t groups = tiles * n, rounds = (groups + cus - 1) / cus;
      double us = 1.5 + rounds * (4.0 + k * (dequant + 1.5 * mb) * (rounds > 2 ? 1.3 : 2 * groups > cus ? 1.1 : 0.85));
      if (raw_codes) {   // (one round: slower the more bytes its weights are)
        const double slow = rounds > 1 ? 0.95 : (2 * groups > cus ? 0.86 : 0.8) + 2.5e-9 * size_n * size_k;
        us = 1.4 + rounds * (2.4 + 0.3 * mb + k * (raw[0] + raw[1] * mb) * slow);
        if (mb == kMidMostRawRows && n == 1 && mid_strips_by_rounds((double)((size_m + 16 * mb - 1) / (16 * mb)), 0.0, size_n, size_k, true, cus) == 4) {
          const int64_t fours = ((size_m + 16 * mb - 1) / (16 * mb)) * ((size_n + 255) / 256), rounds4 = (fours + cus - 1) / cus;
          const double k4 = 2 * ((steps / 2 + 1) / 2) * 256 / 4096.0;
          const double slow4 = rounds4 > 1 ? 1.0 : 0.63 + 0.58 * fours / cus;
          us = 1.4 + rounds4 * (2.4 + 0.3 * mb + k4 * (raw[0] + raw[1] * mb) * slow4);
        }
      }
      if (us < memory) us = memory;
      if (n > 1) us += raw_codes ? 3.0 + 1.6e-6 * n * size_m * size_n : 3.3 + 2e-6 * n * size_m * size_n;
      if (us < best) best = us, row_blocks = mb, splits = n;
    }
  }
  return best;
}

// Whether a call that the tile kernels could take runs in this kernel, whose time mid_estimate puts at `mid_us`, with K in
// `splits` ranges.  `twin`: tile_twin_applies.
// What mid_estimate lacks on the calls tile_estimate was fitted to, with K in one piece: kSlow.  (A time of the tile kernels that
// grows with the operations alone, and 0.93 for either kernel: 2.7 % slower than the better of the two on 147 random calls, at
// worst 1.6 times; so 0.6 %, 1.3 times.)
// 8-bit codes with one scale a column in bf16 have factors of their own: this kernel multiplies them unscaled, with fewer
// instructions than mid_estimate's fit of all 8-bit codes, and the tile kernels take longer for fp8 codes in bf16 than
// tile_estimate has it (199 random calls of 65 to 3000 rows: slower than the better of the two by 5.6 % (fp8) and 1.4 % (integers),
// at worst 1.5 times, with the other formats' factors; so 0.3 % and 0.5 %, 1.17 times.  Us, before -> now: fp8, M = 271,
// K = 6144, N = 6400 51.4 -> 34.9; M = 134, K = 3968, N = 26240 71.8 -> 53.0; integers, M = 196, K = 1664, N = 11392
// 29.9 -> 24.0).
inline bool mid_beats_tiles(double mid_us, int splits, int64_t size_m, int64_t size_n, int64_t size_k, int64_t num_groups,
                            int group_size, bool float16, int format, bool rows_97_128, bool twin) {
  static const double kStep[6] = {kTileStepInt4, kTileStepInt4, 1.27, 1.27, kTileStepMxFp4, 1.30};
  static const double kSlow[6][2] = {   // float16, bfloat16
      {1.12, 1.10}, {1.18, 1.10}, {1.30, 1.12}, {1.13, 1.05}, {1.22, 1.22}, {1.03, 1.0}};
  const bool is_8bit = format == kMidInt8 || format == kMidFp8, groups_of_32 = num_groups > 1 && group_size == 32;
  if (is_8bit && num_groups == 1 && !float16) mid_us *= format == kMidFp8 ? 0.77 : 0.92;
  else if (splits > 1) mid_us *= 0.94;
  else mid_us *= format == kMidFp8 && groups_of_32 ? 0.97 : kSlow[format][float16 ? 0 : 1];
  const bool rows128 = format != kMidNvFp4 && !(is_8bit && groups_of_32);
  if (twin && twin_pays(size_m, size_n, size_k, float16, format == kMidMxFp4, rows128, rows_97_128) &&
      twin_estimate(size_m, size_n, size_k, float16, format == kMidMxFp4) <= mid_us)
    return false;
  return mid_us < tile_estimate(size_m, size_n, size_k, kStep[format], rows128, rows_97_128);
}

// Up to 16 rows of 8-bit codes or NVFP4, which the decode kernel does not have: into how many parts K is split, in
// tiles of one row block and one strip.  Never more workgroups than compute units (two on one share its vector unit:
// K = 4096, N = 11008, fp8, 172 strips: 14.8 us, 17.4 with K in two), and as many parts as pay for the pass that adds them:
// about 1.2 us for 64 rows in each of a workgroup's eight ranges, 3 us for the pass (N = 4096, 64 strips, K = 1 / 2 / 4 parts:
// 13.2 / 11.4 / 10.0 us; K = 1024, N = 1024: 5.1 / 6.4 / 6.5).
inline int mid_splits_16_rows(int64_t size_n, int64_t size_k, int cus) {
  const int64_t strips = size_n / 64, steps = size_k / 64;
  double best = 1e30;
  int splits = 1;
  for (int n = 1; n <= kMidMostSplits && (n == 1 || (strips * n <= cus && steps >= 8 * n)); ++n) {
    const double us = 1.2 * (((steps + n - 1) / n + 7) / 8) + (n > 1 ? 3.0 + 0.1 * n : 0.0);
    if (us < best) best = us, splits = n;
  }
  return splits;
}

inline int mid_moe_strips(int64_t block_size, int64_t slots, int64_t num_experts, int64_t size_n, int64_t size_k, bool units, int cus) {
  const int64_t most = block_size * 7 / 8, even = block_size == 64 ? 44 : block_size * 5 / 8;
  const double second = slots > even ? 0.0009 * (slots - even) * (slots - even) : 0.0;   // second blocks, for each first one
  return mid_strips_by_rounds((double)num_experts * (slots <= most ? 1.0 + second : slots / most + 1), 0.1, size_n, size_k, units, cus);
}

// Strips of a workgroup in the calling thread's last GEMM; 0: that ran in another kernel.
extern thread_local int g_last_mid_strips;

// `row_blocks`: 16-row blocks of a tile, 1 to 6.
int mid_gemm(MidParams p, int dtype, int format, int row_blocks, hipStream_t st);

// Grouped: 4-bit integers as `raw_codes` has them, or MXFP4; blocks of 32, 48 or 64 slots, `blocks` of them at most.
int mid_moe_gemm(MidMoeParams p, int dtype, int format, int blocks, hipStream_t st);

}  // namespace sonar
