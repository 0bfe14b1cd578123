// Tiled W4A16 GEMM for more than 64 activation rows (the MFMA-bound regime).
//
// A workgroup of eight wavefronts owns a 256 (rows of A) x 256 (columns of W)
// tile of C and walks K in steps of 64.  Per step, four wavefronts each fetch
// one 1-KiB chunk of packed weights per 32 rows (64 columns x 32 rows, already
// in operand order), dequantise it in registers and store the result to LDS as
// four 16-column operand blocks; all eight wavefronts fetch the 256 x 64 slice
// of A and store it to LDS as 16-row operand blocks.  An operand block is 64
// lanes x 16 bytes: exactly what one v_mfma_f32_16x16x32 reads, so every LDS
// read of the inner loop is a linear, conflict-free ds_read_b128.  LDS is
// double-buffered; the global loads of step i+1 are issued before the matrix
// work of step i and land in registers meanwhile.  Each wavefront computes a
// 128 x 64 sub-tile: 8 x 4 accumulator tiles, weights as the row operand
// (D[n][m]) so a lane ends up with four consecutive columns of one row of C.
//
// Workgroup ids are dealt so that the 32 workgroups resident on one XCD (ids
// congruent mod 8) take neighbouring tiles (tile_of_workgroup).
#include <cstdlib>
#include <type_traits>

#include "dequant.hpp"
#include "gemm_plan.hpp"
#include "moe_activation.hpp"

namespace sonar {
namespace {

constexpr int kTileM = 256;
constexpr int kTileN = 256;
constexpr int kTileK = 64;
constexpr int kTileWaves = 8;
constexpr int kBlockBytes = 1024;                          // one operand block
constexpr int kStageA = (kTileM / 16) * (kTileK / 32) * kBlockBytes;  // 32 KiB
constexpr int kStageB = (kTileN / 16) * (kTileK / 32) * kBlockBytes;  // 32 KiB
constexpr int kStageBytes = kStageA + kStageB;
constexpr int kTileLds = 2 * kStageBytes;                  // 128 KiB

struct TileParams {
  const uint16_t* a;
  long lda;
  uint16_t* c;
  const uint4* b;
  const uint16_t* bias;
  const float* global_scale;   // NVFP4: one number the output is multiplied by; else nullptr
  const uint16_t* scales;
  const uint32_t* zeros;
  const int32_t* perm;
  int size_m, size_n, size_k;
  int num_groups, group_size;
  int chunks_per_strip;
  int tiles_m, tiles_n;
  int tile_rows;               // rows of a tile: 256 (128: marlin_tile_wide_kernel with 8 row blocks)
  int tile_band;               // rows of tiles per band of the tile numbering (tile_of_workgroup)
  // split K (k_splits > 1): workgroup (tile, split) of a split tile covers K steps
  // [split * k_steps_per_split, ...) and leaves its fp32 tile in `partial` for tile_reduce_kernel
  int k_splits, k_steps_per_split;
  int whole_tiles;             // with k_splits > 1: tiles 0..whole_tiles-1 of the numbering are not split
  float4* partial;
  // grouped (mixture-of-experts) calls only
  const int32_t* sorted_ids;   // slot -> row id of C (row id / top_k of A), >= rows_total: padding
  const float* topk_weights;
  const int32_t* tile_table;   // [0]: number of row tiles, then (first block, blocks, expert) per tile
  // launches with both tile sizes (marlin_tile_wide_pair_kernel): dense, the first `big_tiles` tiles of the 256-row
  // numbering as they are and the others as two 128-row tiles each; grouped, `tile_table` of 256-row tiles and
  // `table_small` of 128-row tiles (pair_word says what their first words hold)
  int big_tiles;
  const int32_t* table_small;
  float4* partial_small;       // partial tiles of the 128-row tiles
  int rows_total, top_k, mul_topk;
  int a_by_slot;               // grouped: row of A = slot index (a column-permuted copy made per slot), else row id / top_k
  long expert_b_stride;        // uint4 units between experts in b
  long expert_s_stride, expert_z_stride, expert_bias_stride;  // elements between experts
  // grouped, wide kernel: the gated activation of C, (rows_total, size_n / 2), in place of C; `gated_halves`: silu_and_mul of the
  // columns' two halves, else swigluoai_and_mul of alternating columns
  uint16_t* gated;
  int gated_halves;
  float gated_limit, gated_alpha;
};

// 16 bytes (8 consecutive k) of row `row` of A, gathered through perm when given.
template <bool HAS_PERM>
__device__ __forceinline__ uint4 load_a16(const TileParams& p, int row, int k0) {
  const uint16_t* arow = p.a + (long)(row < p.size_m ? row : p.size_m - 1) * p.lda;
  if (!HAS_PERM) return *reinterpret_cast<const uint4*>(arow + k0);
  const int4 p0 = *reinterpret_cast<const int4*>(p.perm + k0);
  const int4 p1 = *reinterpret_cast<const int4*>(p.perm + k0 + 4);
  uint4 v;
  v.x = (uint32_t)arow[p0.x] | ((uint32_t)arow[p0.y] << 16);
  v.y = (uint32_t)arow[p0.z] | ((uint32_t)arow[p0.w] << 16);
  v.z = (uint32_t)arow[p1.x] | ((uint32_t)arow[p1.y] << 16);
  v.w = (uint32_t)arow[p1.z] | ((uint32_t)arow[p1.w] << 16);
  return v;
}

// Tiles are numbered band by band (tile_band rows of tiles), inside a band
// column by column: with bands of 4 rows, 32 consecutive tiles are 4 panels
// of A x 8 panels of W.
__host__ __device__ __forceinline__ void tile_coords(const TileParams& p, int tile, int& tile_m, int& tile_n) {
  const int band = tile / (p.tile_band * p.tiles_n);
  const int rem = tile - band * p.tile_band * p.tiles_n;
  const int rows = min(p.tile_band, p.tiles_m - band * p.tile_band);
  tile_n = rem / rows;
  tile_m = band * p.tile_band + rem - tile_n * rows;
}
// Tiles of the launch, and those of them computed by one workgroup over the whole of K (the first ones).
__host__ __device__ __forceinline__ int launch_tiles(const TileParams& p) {
  return p.tiles_m * p.tiles_n;
}
__host__ __device__ __forceinline__ int whole_tiles(const TileParams& p) {
  return p.k_splits > 1 ? p.whole_tiles : launch_tiles(p);
}

// Workgroup id -> (tile, K range).  Workgroups whose ids are congruent mod 8
// run on one XCD and share its L2: each XCD takes a contiguous run of the
// whole tiles, rows of A innermost, so the workgroups resident on it share a
// few panels of W, and after those a contiguous run of the (tile, split) pairs
// of the split tiles, so that the short workgroups start last on every XCD.
// Returns false for the padding ids of a run.
__host__ __device__ __forceinline__ bool tile_of_block(const TileParams& p, int block, int& tile, int& split,
                                                       bool& whole_k) {
  const int tiles = launch_tiles(p);
  const int whole = whole_tiles(p);
  const int split_tiles = tiles - whole;
  const int whole_per_xcd = (whole + 7) / 8;
  const int split_per_xcd = (split_tiles * p.k_splits + 7) / 8;
  const int xcd = block & 7, i = block >> 3;
  whole_k = i < whole_per_xcd;
  if (whole_k) {
    tile = xcd * whole_per_xcd + i;
    split = 0;
    return tile < whole;
  }
  // (a grouped launch is sized for the most tiles there could be: ids past this XCD's share do nothing)
  if (i - whole_per_xcd >= split_per_xcd) return false;
  const int t = xcd * split_per_xcd + (i - whole_per_xcd);
  if (t >= split_tiles * p.k_splits) return false;
  split = t / split_tiles;
  tile = whole + t - split * split_tiles;
  return true;
}
__device__ __forceinline__ bool tile_of_workgroup(const TileParams& p, int& tile, int& split, bool& whole_k) {
  return tile_of_block(p, blockIdx.x, tile, split, whole_k);
}

// Grouped calls learn the number of their tiles on the device (the routing decides it), so the
// kernel plans the K split itself, by plan_gemm's rules: fewer tiles than compute units, or a last
// round of workgroups that fills half of the chip or less, are cut along K into about 256
// workgroups, in ranges of a multiple of four steps (the caller has checked that K allows it).
constexpr int kLiveSplitTilesMax = 128;   // tiles that can be split, and
constexpr int kLiveSplitWorkMax = 256;    // (tile, K range) pairs, i.e. partial tiles, there can be
struct LiveSplit {
  int whole, splits, steps;   // tiles computed over the whole of K; K ranges per split tile; steps per range
};
__host__ __device__ __forceinline__ LiveSplit plan_live_split(int tiles, int k_steps) {
  LiveSplit s = {tiles, 1, k_steps};
  int split_tiles = 0;
  if (tiles < 256) split_tiles = tiles;
  else if (k_steps >= 48 && tiles % 256 <= 128) split_tiles = tiles % 256;
  if (split_tiles == 0 || split_tiles > kLiveSplitTilesMax) return s;
  int splits = 256 / split_tiles;
  if (splits > k_steps / 8) splits = k_steps / 8;
  if (splits > 16) splits = 16;
  if (splits < 2) return s;
  const int steps = ((k_steps + splits - 1) / splits + 3) / 4 * 4;
  splits = (k_steps + steps - 1) / steps;   // no empty range
  if (splits < 2) return s;
  s.whole = tiles - split_tiles;
  s.splits = splits;
  s.steps = steps;
  return s;
}
// The tiles there are in a grouped call (`row_tiles` of them down the rows), with the K split
// planned from them when the call has room for partial tiles.
__host__ __device__ __forceinline__ TileParams live_tiles_of(const TileParams& p, int row_tiles) {
  TileParams live = p;
  live.tiles_m = row_tiles;
  live.tile_band = 4;
  if (p.partial != nullptr) {
    const LiveSplit s = plan_live_split(live.tiles_m * live.tiles_n, p.size_k / kTileK);
    live.k_splits = s.splits;
    live.whole_tiles = s.whole;
    live.k_steps_per_split = s.steps;
  }
  return live;
}
__device__ __forceinline__ TileParams live_tiles(const TileParams& p) { return live_tiles_of(p, p.tile_table[0]); }

// ---- Launches with both tile sizes (marlin_tile_wide_pair_kernel).
// What a 128-row tile takes of a 256-row tile's time.
constexpr float kPairBig = 1.f, kPairSmall = 0.58f;
// (A power of two, and floats below: these run in a kernel that is all latency.)
constexpr int kPairCus = 256;
// When the last of `big` longer and `small` shorter tiles ends, the longer ones started first and every tile on the compute
// unit that is free first.
__host__ __device__ __forceinline__ float pair_makespan(int big, float big_time, int small, float small_time) {
  const int rounds = big / kPairCus, extra = big % kPairCus;
  float t0 = rounds * big_time, t1 = t0 + big_time;      // compute units with `rounds` and one more of them
  float end = extra > 0 ? t1 : t0;
  if (small > 16 * kPairCus) return end + small * small_time * (1.f / kPairCus);
  while (small > 0) {
    const bool first = extra == 0 || t0 <= t1;
    small -= first ? kPairCus - extra : extra;
    (first ? t0 : t1) += small_time;
    end = fmaxf(end, first ? t0 : t1);
  }
  return end;
}
// Steps of a range when K is cut into about `splits`, and the ranges there are then.
__host__ __device__ __forceinline__ int pair_range(int k_steps, int splits) {
  return splits > 1 ? ((k_steps + splits - 1) / splits + 3) / 4 * 4 : k_steps;
}
__host__ __device__ __forceinline__ int pair_ranges(int k_steps, int splits) {
  const int range = pair_range(k_steps, splits);
  return (k_steps + range - 1) / range;
}
// How a grouped call's rows are cut: of `big` 256-row and `small` 128-row row tiles at first, the last `halved` 256-row ones
// become two 128-row tiles each, and K of the tiles of each size is cut into `splits[size]` ranges, whose partial tiles a second
// kernel adds.
struct PairPlan {
  int halved, splits[2];
};
// The time that takes, and a little of the work it is (a launch with less of it leaves more of the power limit).
__host__ __device__ __forceinline__ float pair_cost(int big, int small, const PairPlan& plan, int tiles_n, int k_steps) {
  int tiles[2] = {(big - plan.halved) * tiles_n, (small + 2 * plan.halved) * tiles_n};
  float time[2] = {kPairBig, kPairSmall}, extra = 0.f;
  for (int i = 0; i < 2; ++i)
    // (a K step of a 256-row tile is about 1.4 us, its start and end 13 us, the sum of the partial tiles 8 us: as measured with
    // results stored from the registers; whole lines have made the end shorter since, and a gated activation longer)
    if (plan.splits[i] > 1) {
      tiles[i] *= plan.splits[i];
      time[i] *= (k_steps / (float)plan.splits[i] + 11.f) / (k_steps + 9.f);
      extra = 8.f / (1.4f * k_steps + 13.f);
    }
  const float work = (tiles[0] * time[0] + tiles[1] * time[1]) * (1.f / kPairCus);
  return pair_makespan(tiles[0], time[0], tiles[1], time[1]) + extra + 0.125f * work;
}
// Whether the partial tiles of a plan have room: K is cut for all tiles of a size, while they are few.
__host__ __device__ __forceinline__ bool pair_has_room(int big, int small, const PairPlan& plan, int tiles_n, int k_steps) {
  const int tiles[2] = {(big - plan.halved) * tiles_n, (small + 2 * plan.halved) * tiles_n};
  for (int i = 0; i < 2; ++i)
    if (plan.splits[i] > 1 && (tiles[i] == 0 || tiles[i] > kLiveSplitTilesMax || tiles[i] * plan.splits[i] > kLiveSplitWorkMax ||
                               k_steps < 8 * plan.splits[i]))
      return false;
  return true;
}
// Plans by number, at most 256: the first is none halved, nothing cut.
__host__ __device__ __forceinline__ int pair_halved_step(int big, bool may_split) { return may_split ? big / 16 + 1 : big / 128 + 1; }
__host__ __device__ __forceinline__ int pair_plans(int big, bool may_split) {
  return (big / pair_halved_step(big, may_split) + 1) * (may_split ? 16 : 1);
}
__host__ __device__ __forceinline__ PairPlan pair_plan(int number, int big, bool may_split) {
  PairPlan plan = {0, {1, 1}};
  if (may_split) {
    plan.splits[0] = number % 4 + 1;
    plan.splits[1] = 1 << (number / 4 % 4);
    number /= 16;
  }
  plan.halved = number * pair_halved_step(big, may_split);
  return plan;
}
// The first word of a table of such a launch: its tiles, and above them the K ranges asked for less one.
constexpr int kPairSplitShift = 27;
__host__ __device__ __forceinline__ int pair_word(int tiles, int splits) { return tiles | ((splits - 1) << kPairSplitShift); }
// The tiles of one size, from the first word of its table, in the terms that moe_tile_reduce_kernel reads.
__host__ __device__ __forceinline__ TileParams pair_params(const TileParams& p, bool small, int word) {
  TileParams q = p;
  const int splits = (word >> kPairSplitShift) + 1, k_steps = p.size_k / kTileK;
  q.tile_rows = small ? 128 : kTileM;
  q.tile_table = small ? p.table_small : p.tile_table;
  q.tiles_m = word & ((1 << kPairSplitShift) - 1);
  q.tile_band = small ? 8 : 4;   // the same rows of A per band with either tile size
  q.k_steps_per_split = pair_range(k_steps, splits);
  q.k_splits = pair_ranges(k_steps, splits);
  q.whole_tiles = 0;   // read only with k_splits > 1
  if (small) q.partial = p.partial_small;
  return q;
}
struct PairTile {
  int rows, tile_m, tile_n, k_first, k_tiles;
  int partial_at;   // -1: the whole of K
};
// Workgroup id -> tile.  Each XCD takes a contiguous run of the 256-row tiles and then one of the 128-row tiles.
// Grouped: `big_word` and `small_word` are the first words of the two tables.  False: nothing to do.
__host__ __device__ __forceinline__ bool pair_tile_of_block(const TileParams& p, int big_word, int small_word, int block,
                                                            PairTile& out) {
  const bool grouped = p.tile_table != nullptr;
  const int xcd = block & 7, k_steps = p.size_k / kTileK;
  int i = block >> 3;
  TileParams q;
  for (int size = 0; size < 2; ++size) {
    int tiles, first = 0;
    if (grouped) {
      q = pair_params(p, size == 1, size == 1 ? small_word : big_word);
      tiles = q.tiles_m * q.tiles_n;
    } else {
      q = p;
      q.k_splits = 1;
      tiles = p.big_tiles;
      if (size == 1) {   // tile t of the 256-row numbering is tiles 2 t and 2 t + 1 of the 128-row one, in bands twice as high
        q.tiles_m = 2 * p.tiles_m;
        q.tile_band = 2 * p.tile_band;
        first = 2 * p.big_tiles;
        tiles = q.tiles_m * q.tiles_n - first;
      }
    }
    const int work = tiles * q.k_splits;
    const int begin = (int)((int64_t)work * xcd >> 3), end = (int)((int64_t)work * (xcd + 1) >> 3);
    if (i < end - begin) {
      i += begin;
      const int split = q.k_splits > 1 ? i / tiles : 0;
      out.rows = size == 1 ? 128 : kTileM;
      out.partial_at = q.k_splits > 1 ? i : -1;
      out.k_first = split * q.k_steps_per_split;
      out.k_tiles = q.k_splits > 1 && out.k_first + q.k_steps_per_split < k_steps ? out.k_first + q.k_steps_per_split : k_steps;
      tile_coords(q, first + i - split * tiles, out.tile_m, out.tile_n);
      return grouped || out.tile_m * out.rows < p.size_m;   // (the second half of a ragged last tile may have no rows)
    }
    i -= end - begin;
  }
  return false;
}
inline int pair_grid(const TileParams& p, int max_tiles) {
  if (p.tile_table == nullptr) {
    const int smalls = 2 * (p.tiles_m * p.tiles_n - p.big_tiles);
    return 8 * ((p.big_tiles + 7) / 8 + (smalls + 7) / 8);
  }
  // a tile has at least one block; K ranges: at most kLiveSplitWorkMax of either size
  return 8 * ((max_tiles * p.tiles_n + 7) / 8 + 2 + (p.partial != nullptr ? 2 * kLiveSplitWorkMax / 8 : 0));
}

inline int tile_grid(const TileParams& p) {
  const int whole = whole_tiles(p);
  const int split_work = (launch_tiles(p) - whole) * p.k_splits;
  // (a grouped call with room for partial tiles: the kernel may turn up to 128 of its tiles into 256 K ranges)
  const int live_split = p.tile_table != nullptr && p.partial != nullptr ? kLiveSplitWorkMax : 0;
  return 8 * ((whole + 7) / 8 + (split_work + live_split + 7) / 8);
}

template <typename T, bool HAS_ZP, bool HAS_PERM>
__global__ __launch_bounds__(kTileWaves * 64) void marlin_tile_kernel(const TileParams p) {
  typedef typename Dq<T>::vec8 vec8;
  typedef typename Dq<T>::Col Col;
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col16 = lane & 15;
  const int kb = lane >> 4;
  const uint32_t magic = magic_register();
  const bool grouped = p.num_groups > 1;

  int tile, tile_m, tile_n, split;
  bool whole_k;
  if (!tile_of_workgroup(p, tile, split, whole_k)) return;  // this kernel is launched with k_splits == 1
  tile_coords(p, tile, tile_m, tile_n);
  const int m0 = tile_m * kTileM;
  const int strip0 = tile_n * (kTileN / kStripN);
  const int strips_here = min(kTileN / kStripN, p.size_n / kStripN - strip0);

  // ---- what this thread fetches per K step
  // A: the 256 x 64 slice is 32 operand blocks (16 row blocks x 2 k blocks);
  // thread t fills lane t%64 of blocks t/64 + 8*i, i = 0..3.
  // W: wavefronts 0..3 each own one strip of the tile and fetch its two chunks.
  const bool loads_b = wave < strips_here;
  const uint4* b_src = p.b + (size_t)(unsigned)((strip0 + (loads_b ? wave : 0)) * p.chunks_per_strip) * 64 + lane;
  const uint16_t* s_src = p.scales + (strip0 + (loads_b ? wave : 0)) * kStripN;
  const uint32_t* z_src = HAS_ZP ? p.zeros + (strip0 + (loads_b ? wave : 0)) * 8 + zero_point_word(col16) : nullptr;
  int s_slot[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) s_slot[j] = scale_slot(16 * j + col16, grouped);

  // ---- what this wavefront computes
  const int wm = wave >> 2;   // rows 128*wm .. +128 of the tile
  const int wn = wave & 3;    // strip wn of the tile
  floatx4_t acc[4][8];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int mb = 0; mb < 8; ++mb) acc[nb][mb] = floatx4_t{0.f, 0.f, 0.f, 0.f};

  uint4 a_reg[4];
  uint4 b_reg[2];
  uint32_t s_reg[2][4];
  uint32_t z_reg[2];

  auto fetch = [&](int kt) {
    const int k0 = kt * kTileK;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int blk = wave + 8 * i;          // 0..31: row block blk>>1, k block blk&1
      a_reg[i] = load_a16<HAS_PERM>(p, m0 + 16 * (blk >> 1) + col16, k0 + 32 * (blk & 1) + 8 * kb);
    }
    if (loads_b) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int chunk = kt * 2 + h;
        b_reg[h] = b_src[(size_t)chunk * 64];
        const int g = grouped ? (chunk * kChunkK) / p.group_size : 0;
        const uint16_t* srow = s_src + (long)g * p.size_n;
#pragma unroll
        for (int j = 0; j < 4; ++j) s_reg[h][j] = srow[s_slot[j]];
        if (HAS_ZP) z_reg[h] = z_src[(long)g * (p.size_n / 8)];
      }
    }
  };

  auto stash = [&](int stage) {
    char* sa = smem + stage * kStageBytes;
    char* sb = sa + kStageA;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<uint4*>(sa + (wave + 8 * i) * kBlockBytes + lane * 16) = a_reg[i];
    if (loads_b) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        Col cols[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          int z = 8;
          if (HAS_ZP) z = (int)((z_reg[h] >> zero_point_shift(16 * j + col16)) & 0xFu);
          cols[j] = Dq<T>::make_col((uint16_t)s_reg[h][j], z);
        }
        const uint32_t words[4] = {b_reg[h].x, b_reg[h].y, b_reg[h].z, b_reg[h].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const vec8 w = Dq<T>::word(words[j], cols[j], magic);
          // column block 4*wave + j of the tile, k block h
          *reinterpret_cast<vec8*>(sb + ((4 * wave + j) * 2 + h) * kBlockBytes + lane * 16) = w;
        }
      }
    }
  };

  const int k_tiles = p.size_k / kTileK;
  fetch(0);
  stash(0);
  __syncthreads();

  for (int kt = 0; kt < k_tiles; ++kt) {
    if (kt + 1 < k_tiles) fetch(kt + 1);
    const char* sa = smem + (kt & 1) * kStageBytes;
    const char* sb = sa + kStageA;
    if (wn < strips_here) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        vec8 wv[4];
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
          wv[nb] = *reinterpret_cast<const vec8*>(sb + ((4 * wn + nb) * 2 + h) * kBlockBytes + lane * 16);
#pragma unroll
        for (int mb = 0; mb < 8; ++mb) {
          const vec8 av =
              *reinterpret_cast<const vec8*>(sa + ((8 * wm + mb) * 2 + h) * kBlockBytes + lane * 16);
#pragma unroll
          for (int nb = 0; nb < 4; ++nb) acc[nb][mb] = Dq<T>::mfma(wv[nb], av, acc[nb][mb]);
        }
      }
    }
    if (kt + 1 < k_tiles) stash((kt + 1) & 1);
    __syncthreads();
  }

  // ---- epilogue: lane holds C[m][n .. n+3] for m = row block + lane%16
  if (wn >= strips_here) return;
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    const int n = (strip0 + wn) * kStripN + 16 * nb + 4 * kb;
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (p.bias) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        bias[r] = Dq<T>::to_float(p.bias[(strip0 + wn) * kStripN + scale_slot(16 * nb + 4 * kb + r, false)]);
    }
#pragma unroll
    for (int mb = 0; mb < 8; ++mb) {
      const int m = m0 + 128 * wm + 16 * mb + col16;
      if (m < p.size_m) {
        const floatx4_t v = acc[nb][mb];
        uint2 o;
        o.x = (uint32_t)Dq<T>::from_float(v.x + bias[0]) | ((uint32_t)Dq<T>::from_float(v.y + bias[1]) << 16);
        o.y = (uint32_t)Dq<T>::from_float(v.z + bias[2]) | ((uint32_t)Dq<T>::from_float(v.w + bias[3]) << 16);
        *reinterpret_cast<uint2*>(p.c + (long)m * p.size_n + n) = o;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The same tile with every operand arriving through asynchronous global -> LDS
// copies, three K steps deep, so no vector register holds bytes in flight and
// the copies of step i+2 are issued before the matrix work of step i.
//   * A: a ring of three 32-KiB stages shared by the workgroup, each 32
//     regions of 8 rows x 128 bytes; wavefront w copies regions 4w..4w+3, one
//     copy per region, eight whole 128-byte lines per copy.
//   * W: the packed chunks are already in operand order.  Every wavefront
//     copies the two chunks of its strip (and the scale / zero-point row of the
//     step's group) into a private ring and dequantises them in registers.
// The eight wavefronts form two groups (wm = 0: rows 0..127 of the tile, wm = 1:
// rows 128..255); each SIMD holds one wavefront of either group.  A K step is
// two half steps (k blocks 0 and 1), a half step is a "fetch" phase (the copies
// of a later stage, the LDS read of one packed chunk, dequantisation: VALU
// work) followed by a "multiply" phase (32 MFMAs and, behind the four of a row
// block, the LDS read of that row block's operand of the next half step; a
// group reads only rows of A that its own wavefronts copied).  Phases end with
// a workgroup barrier and group 1 runs one phase behind group 0, so that on
// every SIMD one wavefront multiplies while the other fetches.  The fetch phase
// is the longer one: while its sibling issues MFMAs a wavefront gets a VALU
// instruction through every eight cycles or so, and its copies and LDS
// instructions take their issue time on top of that.
// Copies of a wavefront complete in issue order, seven per stage, so "stage i
// has landed" is s_waitcnt vmcnt(7) while the copies of stage i+1 are
// outstanding.  With p = 4 kt + 2 b (+1 for group 1) the phase in which the
// fetch of (step kt, k block b) runs: stage kt is read in phases 4kt..4kt+3; the
// copies of stage kt+2 go to the slot of stage kt-1 and are issued in the two
// fetch phases of step kt, phases 4kt..4kt+3, after the barrier that ends
// phase 4kt-1; every wavefront waits for its copies of stage kt+1 at the end of
// its fetch of (kt, 1), phases 4kt+2 and 4kt+3, before the barrier that starts
// phase 4kt+4.
// LDS is read from asm blocks only (the compiler cannot tell which LDS bytes a
// copy writes and would otherwise wait for all copies before any LDS access).
// Needs groups of a multiple of 64 rows (or one group) and no act-order, or MXFP4: what the wide kernel does not take
// (groups of 192 rows and the like, and dense MXFP4 calls of few tiles).
constexpr int kAsyncStages = 3;
// g32: groups of 32 rows (MXFP4), i.e. one group per k block: a stage then carries two
// scale rows (256 bytes each) and takes one copy more.
constexpr int wave_stage(bool g32) { return 2 * kBlockBytes + (g32 ? 512 : 256); }   // two weight chunks + scale rows
constexpr int kAsyncA = kAsyncStages * kStageA;
constexpr int async_lds(bool g32) { return kAsyncA + kTileWaves * kAsyncStages * wave_stage(g32); }
constexpr int async_copies(bool g32) { return g32 ? 8 : 7; }
// 8-bit codes (W8: uint8b128): a K step of a strip is four 1-KiB blocks
// of 16 rows (block 2 b holds the low four, block 2 b + 1 the high four of the eight
// consecutive rows of a lane's operand of k block b).  Private rings of that size would not
// fit, so the two wavefronts of a strip (one per group of rows) share one ring: the
// wavefront of group 0 copies the two blocks of k block 0, that of group 1 those of k block
// 1, the same number of copies per stage as with 4-bit codes.  The barriers that order the
// shared stages of A order these too: group 1 reads k block 0 one phase after group 0 has
// waited for its copies, group 0 reads k block 1 two barriers after group 1 has.
constexpr int strip_stage8() { return 4 * kBlockBytes + 256; }
constexpr int async_lds8() { return kAsyncA + (kTileN / kStripN) * kAsyncStages * strip_stage8(); }

template <typename T, bool HAS_ZP, bool GROUPED, bool FP4 = false, bool W8 = false>
__global__ __launch_bounds__(kTileWaves * 64) void marlin_tile_async_kernel(const TileParams p) {
  typedef typename Dq<T>::vec8 vec8;
  typedef typename Dq4Of<T, FP4, false>::type D4;   // integer codes, or float4_e2m1f (MXFP4)
  typedef typename Dq8Of<T, false>::type D8;
  typedef typename std::conditional<W8, typename D8::Col, typename D4::Col>::type Col;
  static_assert(!W8 || (!HAS_ZP && !FP4), "8-bit codes are symmetric");
  constexpr bool G32 = FP4;
  constexpr int kWaveStage = W8 ? strip_stage8() : wave_stage(G32);
  constexpr int kWeightBytes = (W8 ? 4 : 2) * kBlockBytes;   // packed weights of a stage, scale rows behind them
  constexpr int kAsyncCopies = async_copies(G32);
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col16 = lane & 15;
  const int kb = lane >> 4;
  const uint32_t magic = magic_register();
  const bool grouped = p.num_groups > 1;

  int tile, tile_m, tile_n, split;
  bool whole_k;
  if (!tile_of_workgroup(p, tile, split, whole_k)) return;
  tile_coords(p, tile, tile_m, tile_n);
  // Grouped calls: row tile t is up to four consecutive 64-slot blocks of one
  // expert, listed in tile_table; rows are slots of sorted_ids.
  int first_slot = 0, tile_rows = kTileM;
  long expert = 0;
  if (GROUPED) {
    if (tile_m >= p.tile_table[0]) return;
    first_slot = p.tile_table[1 + 3 * tile_m] * 64;
    tile_rows = p.tile_table[2 + 3 * tile_m] * 64;
    expert = p.tile_table[3 + 3 * tile_m];
  }
  const int m0 = tile_m * kTileM;
  const int strip0 = tile_n * (kTileN / kStripN);
  const int strips_here = min(kTileN / kStripN, p.size_n / kStripN - strip0);
  const int wm = wave >> 2;
  const int wn = wave & 3;
  const bool active = wn < strips_here;
  // a wavefront past the last strip copies the last strip again and computes nothing
  const int strip = strip0 + (active ? wn : strips_here - 1);

  // ---- copy sources
  // A stage is 32 regions of 1 KiB: region 2 rb + h holds rows 8h..8h+7 of row
  // block rb, 128 bytes (both k blocks) each.  One copy fills one region: its
  // lanes 8r..8r+7 fetch the eight 16-byte pieces of one 128-byte line of row r,
  // so an instruction touches 8 whole lines (16 rows x 64 bytes per instruction,
  // the operand-block shape, moves a third of the bytes per cycle).  Piece q of
  // row r sits at 16-byte slot q ^ r of the row, which keeps the operand reads
  // (16 rows, one piece each) off each other's banks.  Wavefront w fills
  // regions 4w..4w+3.
  const char* a_src[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int region = 4 * wave + i;
    const int r8 = lane >> 3;
    const int in_tile = 16 * (region >> 1) + 8 * (region & 1) + r8;
    int row;
    if (GROUPED) {
      const int id = in_tile < tile_rows ? p.sorted_ids[first_slot + in_tile] : p.rows_total;
      // padding slots read row 0, never stored
      row = (unsigned)id < (unsigned)p.rows_total ? (p.a_by_slot ? first_slot + in_tile : id / p.top_k) : 0;
    } else {
      row = m0 + in_tile;
      if (row >= p.size_m) row = p.size_m - 1;  // rows past M are computed and never stored
    }
    a_src[i] = reinterpret_cast<const char*>(p.a) + ((long)row * p.lda + 8 * ((lane & 7) ^ r8)) * 2;
  }
  const uint4* b_src = p.b + expert * p.expert_b_stride +
                       (size_t)(unsigned)(strip * p.chunks_per_strip) * (W8 ? 128 : 64) + lane;
  const char* s_src;
  long s_group_stride;
  if (HAS_ZP && lane >= 32) {
    s_src = reinterpret_cast<const char*>(p.zeros + expert * p.expert_z_stride + strip * 8 + (lane & 7));
    s_group_stride = (long)(p.size_n / 8) * 4;
  } else {
    s_src = reinterpret_cast<const char*>(p.scales + expert * p.expert_s_stride + strip * kStripN) + 4 * (lane & 31);
    s_group_stride = (long)p.size_n * 2;
  }
  // the weight ring: private to the wavefront, or shared by the two wavefronts of a strip (8-bit codes)
  char* wring = smem + kAsyncA + (W8 ? wn : wave) * (kAsyncStages * kWaveStage);
  const uint32_t a_lds = (uint32_t)(uintptr_t)(lds_void_t*)smem;
  const uint32_t w_lds = (uint32_t)(uintptr_t)(lds_void_t*)wring;

  // copy `idx` (0..6) of the stage of step kt: four blocks of A, two weight chunks, one scale row
  auto issue_one = [&](int kt, int slot, int idx) {
    if (idx < 4) {
      char* sa = smem + slot * kStageA;
      __builtin_amdgcn_global_load_lds((glb_void_t*)(a_src[idx] + (long)kt * (kTileK * 2)),
                                       (lds_void_t*)(sa + (4 * wave + idx) * kBlockBytes), 16, 0, 0);
      return;
    }
    char* sw = wring + slot * kWaveStage;
    if (idx < 6) {
      if (W8) {   // blocks 2 wm, 2 wm + 1 of the four of this step: the two of k block wm
        const int blk = 2 * wm + (idx - 4);
        const uint4* g = b_src + (size_t)(4 * kt + blk) * 64;
        __builtin_amdgcn_global_load_lds((glb_void_t*)g, (lds_void_t*)(sw + blk * kBlockBytes), 16, 0, 0);
        return;
      }
      const uint4* g = b_src + (size_t)(2 * kt + (idx - 4)) * 64;   // the two chunks of this step
      __builtin_amdgcn_global_load_lds((glb_void_t*)g, (lds_void_t*)(sw + (idx - 4) * kBlockBytes), 16, 0, 0);
      return;
    }
    // the scale rows (with a shared ring both wavefronts of the strip copy them: the same bytes twice)
    if (G32) {   // idx 6 / 7: the rows of groups 2 kt and 2 kt + 1
      __builtin_amdgcn_global_load_lds((glb_void_t*)(s_src + (long)(2 * kt + idx - 6) * s_group_stride),
                                       (lds_void_t*)(sw + kWeightBytes + 256 * (idx - 6)), 4, 0, 0);
      return;
    }
    const int grp = grouped ? (kt * kTileK) / p.group_size : 0;
    __builtin_amdgcn_global_load_lds((glb_void_t*)(s_src + (long)grp * s_group_stride),
                                     (lds_void_t*)(sw + kWeightBytes), 4, 0, 0);
  };
  auto issue = [&](int kt, int slot) {
#pragma unroll
    for (int idx = 0; idx < kAsyncCopies; ++idx) issue_one(kt, slot, idx);
  };

  uint32_t s_off[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) s_off[j] = kWeightBytes + 2 * scale_slot(16 * j + col16, grouped);
  const uint32_t z_off = kWeightBytes + 128 + 4 * zero_point_word(col16);

  floatx4_t acc[4][8];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int mb = 0; mb < 8; ++mb) acc[nb][mb] = floatx4_t{0.f, 0.f, 0.f, 0.f};

  // K steps [k_first, k_tiles) of this workgroup
  const int k_first = whole_k ? 0 : split * p.k_steps_per_split;
  const int k_tiles = whole_k ? p.size_k / kTileK : min(p.size_k / kTileK, k_first + p.k_steps_per_split);
  issue(k_first, 0);
  issue(min(k_first + 1, k_tiles - 1), 1);

  u32x4_t av[8], wv[4], qraw;
  u32x4_t qhigh = u32x4_t{0u, 0u, 0u, 0u};   // 8-bit codes: the block with the high four rows
  uint32_t sb0 = 0, sb1 = 0, sb2 = 0, sb3 = 0, zw = 0;
  Col cols[4];
// Starts one 16-byte LDS read into `dst`; the data is there after the next
// s_waitcnt lgkmcnt(0) that names `dst` as an operand.  Until then nothing may
// name `dst` (the hardware does not interlock).
#define SONAR_TILE_READ(dst, base, off) \
  asm volatile("ds_read_b128 %0, %1 offset:" #off : "=&v"(dst) : "v"(base) : "memory")
// Waits for every LDS read in flight; the registers they fill are operands so
// that no use of them can be scheduled ahead of the wait.
#define SONAR_TILE_LANDED()                                                                        \
  asm volatile("s_waitcnt lgkmcnt(0)"                                                              \
               : "+v"(av[0]), "+v"(av[1]), "+v"(av[2]), "+v"(av[3]), "+v"(av[4]), "+v"(av[5]),     \
                 "+v"(av[6]), "+v"(av[7])                                                          \
               :                                                                                   \
               : "memory")
  // Starts the reads of the packed chunk of (stage in `slot`, k block b), with
  // the scales and zero points of the step when `with_scales` (they hold for
  // both k blocks: a step lies inside one group).  The wavefront's own copies of
  // that stage must have landed.  The data is picked up by the next fetch().
  auto raw_start = [&](int slot, int b, bool with_scales) {
    const uint32_t w_at = w_lds + slot * kWaveStage;
    const uint32_t q_at = w_at + (W8 ? 2 * b : b) * kBlockBytes + lane * 16;
    const uint32_t r_at = w_at + (G32 ? 256 * b : 0);   // this k block's scale row
    if constexpr (W8) asm volatile("ds_read_b128 %0, %1 offset:1024" : "=&v"(qhigh) : "v"(q_at) : "memory");
    if (with_scales) {
      asm volatile(
          "ds_read_b128 %0, %6\n\t"
          "ds_read_u16 %1, %7\n\t"
          "ds_read_u16 %2, %8\n\t"
          "ds_read_u16 %3, %9\n\t"
          "ds_read_u16 %4, %10\n\t"
          "ds_read_b32 %5, %11"
          : "=&v"(qraw), "=&v"(sb0), "=&v"(sb1), "=&v"(sb2), "=&v"(sb3), "=&v"(zw)
          : "v"(q_at), "v"(r_at + s_off[0]), "v"(r_at + s_off[1]), "v"(r_at + s_off[2]), "v"(r_at + s_off[3]),
            "v"(r_at + z_off)
          : "memory");
    } else {
      asm volatile("ds_read_b128 %0, %1" : "=&v"(qraw) : "v"(q_at) : "memory");
    }
  };
  // Fetch phase of a half step: picks up the packed chunk started by raw_start
  // and dequantises it, then waits for the operands of A the last multiply
  // phase started to read.
  auto fetch = [&](int slot, int b, bool with_scales) {
    if constexpr (W8) {
      asm volatile("s_waitcnt lgkmcnt(0)"
                   : "+v"(qraw), "+v"(qhigh), "+v"(sb0), "+v"(sb1), "+v"(sb2), "+v"(sb3), "+v"(zw)
                   :
                   : "memory");
    } else {
      asm volatile("s_waitcnt lgkmcnt(0)"
                   : "+v"(qraw), "+v"(sb0), "+v"(sb1), "+v"(sb2), "+v"(sb3), "+v"(zw)
                   :
                   : "memory");
    }
    if (with_scales) {
      const uint32_t sbits[4] = {sb0, sb1, sb2, sb3};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (W8) {
          cols[j] = D8::make_col((uint16_t)sbits[j]);
        } else {
          int z = 8;
          if (HAS_ZP) z = (int)((zw >> zero_point_shift(16 * j + col16)) & 0xFu);
          cols[j] = D4::make_col((uint16_t)sbits[j], z);
        }
      }
    }
    if constexpr (W8) {
      const uint32_t lo[4] = {qraw.x, qraw.y, qraw.z, qraw.w}, hi[4] = {qhigh.x, qhigh.y, qhigh.z, qhigh.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint2 w_lo = D8::word4(lo[j], cols[j], magic), w_hi = D8::word4(hi[j], cols[j], magic);
        wv[j] = u32x4_t{w_lo.x, w_lo.y, w_hi.x, w_hi.y};
      }
    } else {
      wv[0] = __builtin_bit_cast(u32x4_t, D4::word(qraw.x, cols[0], magic));
      wv[1] = __builtin_bit_cast(u32x4_t, D4::word(qraw.y, cols[1], magic));
      wv[2] = __builtin_bit_cast(u32x4_t, D4::word(qraw.z, cols[2], magic));
      wv[3] = __builtin_bit_cast(u32x4_t, D4::word(qraw.w, cols[3], magic));
    }
    SONAR_TILE_LANDED();
  };
  // operand lane (kb, col16) of row block rb, k block b: piece 4 b + kb of row col16
  auto a_address = [&](int slot, int b) {
    return a_lds + slot * kStageA + (8 * wm * 2 + (col16 >> 3)) * kBlockBytes + (col16 & 7) * 128 +
           (((4 * b + kb) ^ (col16 & 7)) * 16);
  };
  // Multiply phase: 32 MFMAs, ahead of the other wavefront's VALU work in the
  // issue order; behind the four of a row block, the read of that row block's
  // operand of half step (slot, b), which the next multiply phase uses: the
  // reads of A cost the fetch phases nothing.
  auto multiply_and_read = [&](int slot, int b) {
    const uint32_t a_at = a_address(slot, b);
    __builtin_amdgcn_s_setprio(2);
#define SONAR_TILE_ROW(i, off)                                                                          \
  _Pragma("unroll") for (int j = 0; j < 4; ++j) acc[j][i] =                                             \
      Dq<T>::mfma(__builtin_bit_cast(vec8, wv[j]), __builtin_bit_cast(vec8, av[i]), acc[j][i]);         \
  SONAR_TILE_READ(av[i], a_at, off)
    SONAR_TILE_ROW(0, 0);
    SONAR_TILE_ROW(1, 2048);
    SONAR_TILE_ROW(2, 4096);
    SONAR_TILE_ROW(3, 6144);
    SONAR_TILE_ROW(4, 8192);
    SONAR_TILE_ROW(5, 10240);
    SONAR_TILE_ROW(6, 12288);
    SONAR_TILE_ROW(7, 14336);
#undef SONAR_TILE_ROW
    __builtin_amdgcn_s_setprio(0);
  };
  // end of a phase; nothing may be scheduled across it
  auto phase_end = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  // The loop body has no branches: a wavefront past the last strip of the
  // matrix works on a second copy of the last strip (its results are dropped),
  // and the copies for steps past the end fetch the last step again, into a
  // slot nobody reads any more.  So seven copies are outstanding at every wait.
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kAsyncCopies) : "memory");  // stage k_first has landed
  // a shared ring: the blocks of k block 0 are the copies of the strip's wavefront of group 0,
  // which the wavefront of group 1 may read only behind a barrier that follows that wait
  if constexpr (W8) phase_end();
  raw_start(0, 0, true);
  phase_end();
  {
    const uint32_t a_at = a_address(0, 0);
    SONAR_TILE_READ(av[0], a_at, 0);
    SONAR_TILE_READ(av[1], a_at, 2048);
    SONAR_TILE_READ(av[2], a_at, 4096);
    SONAR_TILE_READ(av[3], a_at, 6144);
    SONAR_TILE_READ(av[4], a_at, 8192);
    SONAR_TILE_READ(av[5], a_at, 10240);
    SONAR_TILE_READ(av[6], a_at, 12288);
    SONAR_TILE_READ(av[7], a_at, 14336);
  }
  if (wm == 1) phase_end();  // group 1 runs one phase behind

  int slot = 0;        // stage of step kt
  int fill = 2;        // stage step kt + 2 goes to
  for (int kt = k_first; kt < k_tiles; ++kt) {
    const int next_slot = slot == kAsyncStages - 1 ? 0 : slot + 1;
    // ---- half step (kt, 0)
    // the copies of stage kt + 2 go out in the fetch phases, four and three: a
    // wavefront waits at a copy while the memory pipeline is busy, which would
    // starve the matrix cores if it happened between MFMAs
    const int copy_kt = min(kt + 2, k_tiles - 1);
#pragma unroll
    for (int idx = 0; idx < 4; ++idx) issue_one(copy_kt, fill, idx);
    fetch(slot, 0, true);
    raw_start(slot, 1, G32);
    phase_end();
    multiply_and_read(slot, 1);
    phase_end();
    // ---- half step (kt, 1)
#pragma unroll
    for (int idx = 4; idx < kAsyncCopies; ++idx) issue_one(copy_kt, fill, idx);
    fetch(slot, 1, G32);
    // stage kt + 1 has landed once nothing but the copies of stage kt + 2 is outstanding
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kAsyncCopies) : "memory");
    raw_start(next_slot, 0, true);
    phase_end();
    // the rows of stage kt + 1 this group reads are the ones it copied, and its four
    // wavefronts have waited for their copies before the barrier above
    multiply_and_read(next_slot, 0);
    phase_end();
    slot = next_slot;
    fill = fill == kAsyncStages - 1 ? 0 : fill + 1;
  }
  if (wm == 0) phase_end();  // the barrier that ends group 1's last phase
  // the last copies and the last read started by raw_start must not outlive the wavefront
  if constexpr (W8) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)"
                 : "+v"(qraw), "+v"(qhigh), "+v"(sb0), "+v"(sb1), "+v"(sb2), "+v"(sb3), "+v"(zw)::"memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" : "+v"(qraw), "+v"(sb0), "+v"(sb1), "+v"(sb2), "+v"(sb3), "+v"(zw)::"memory");
  }
  SONAR_TILE_LANDED();   // the operand reads started by the last multiply phase
#undef SONAR_TILE_LANDED
#undef SONAR_TILE_READ

  if (!active) return;
  if (!GROUPED && !whole_k) {
    // partial tile of this K range: one 1-KiB block per accumulator tile
    const int first_split = whole_tiles(p);
    const int split_tiles = p.tiles_m * p.tiles_n - first_split;
    float4* dst = p.partial + ((size_t)(split * split_tiles + tile - first_split) * 256 + wave * 32) * 64 + lane;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int mb = 0; mb < 8; ++mb) {
        const floatx4_t v = acc[nb][mb];
        dst[(nb * 8 + mb) * 64] = make_float4(v.x, v.y, v.z, v.w);
      }
    return;
  }
  // rows of C this lane writes: one per row block
  long c_row[8];
  float row_w[8];
#pragma unroll
  for (int mb = 0; mb < 8; ++mb) {
    const int r = 128 * wm + 16 * mb + col16;
    c_row[mb] = -1;
    row_w[mb] = 1.f;
    if (GROUPED) {
      const int id = r < tile_rows ? p.sorted_ids[first_slot + r] : p.rows_total;
      if ((unsigned)id < (unsigned)p.rows_total) {
        c_row[mb] = id;
        // the routing weight is rounded to the activation type and the product is
        // formed and rounded in that type (marlin_template.h(moe):1893-1897)
        if (p.mul_topk) row_w[mb] = Dq<T>::to_float(Dq<T>::from_float(p.topk_weights[id]));
      }
    } else if (m0 + r < p.size_m) {
      c_row[mb] = m0 + r;
    }
  }
  const uint16_t* bias_src = p.bias ? p.bias + expert * p.expert_bias_stride + strip * kStripN : nullptr;
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    const int n = strip * kStripN + 16 * nb + 4 * kb;
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias_src) {
#pragma unroll
      for (int r = 0; r < 4; ++r) bias[r] = Dq<T>::to_float(bias_src[scale_slot(16 * nb + 4 * kb + r, false)]);
    }
#pragma unroll
    for (int mb = 0; mb < 8; ++mb) {
      if (c_row[mb] < 0) continue;
      const floatx4_t v = acc[nb][mb];
      uint16_t o[4] = {Dq<T>::from_float(v.x + bias[0]), Dq<T>::from_float(v.y + bias[1]),
                       Dq<T>::from_float(v.z + bias[2]), Dq<T>::from_float(v.w + bias[3])};
      if (GROUPED && p.mul_topk) {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = Dq<T>::from_float(Dq<T>::to_float(o[r]) * row_w[mb]);
      }
      uint2 packed;
      packed.x = (uint32_t)o[0] | ((uint32_t)o[1] << 16);
      packed.y = (uint32_t)o[2] | ((uint32_t)o[3] << 16);
      *reinterpret_cast<uint2*>(p.c + c_row[mb] * p.size_n + n) = packed;
    }
  }
}

// ---------------------------------------------------------------------------
// The wide form of the asynchronous tile kernel: the same 256 x 256 tile and K
// step, four wavefronts instead of eight, one per SIMD with the whole register
// file (256 accumulator registers for 256 rows x 64 columns: a strip over all
// rows of the tile).  A chunk of weights is dequantised once per workgroup
// instead of once per group of rows and feeds 64 MFMAs; with no second
// wavefront on the SIMD the other work (dequantising the next chunk, the LDS
// reads of A four row blocks ahead, the copies of a later stage) sits between
// the MFMAs of the wavefront's own instruction stream, one to two instructions
// behind each MFMA, where the matrix pipeline hides them.
//   * A: a ring of four 32-KiB stages filled by LDS-DMA, wavefront w copying
//     row blocks 4w..4w+3 (eight 1-KiB regions, the layout of the kernel above).
//   * W: the two chunks of a step go from memory straight into registers (one
//     16-byte load per lane and chunk), a ring of four register sets.
//   * scales / zero points: one 256-byte row per step through a private LDS
//     ring of sixteen rows, fetched a step earlier than the rest.
// The eleven memory operations a wavefront issues per step (8 + 1 + 2: stage
// kt + 3 of A and W, the scale row of step kt + 4) go out in the second half of
// step kt.  One barrier per step, between its halves: before it a wavefront
// waits until only the eleven youngest operations are outstanding, so behind it
// stage kt + 1 has landed for everyone and the slot of stage kt - 1 is free.
// The MFMAs are written as asm statements with the accumulator as a tied
// operand: 224 accumulator registers in AGPRs, 32 in VGPRs, every one updated in
// place (left to the register allocator, the 256 accumulators of this loop get
// copied between registers all the time).  The compiler therefore does not see
// MFMAs here and pads no matrix-core hazard: none arises inside the loop (an
// accumulator is touched again 64 MFMAs later, operands are written long before
// they are read), and the results are read after the pipeline has drained
// (s_nop below).
// 4-bit or symmetric 8-bit codes with groups of 64 * 2^i rows or one group, MXFP4 (float4_e2m1f codes,
// bf16, a scale per 32 rows: one hardware conversion and half a byte permute behind each row
// block), integer / 8-bit floating-point codes with a scale per 32 rows (MXFP8 among them), or NVFP4
// (float4_e2m1f codes with a scale per 16 rows and a global scale, either activation type); no
// act-order; dense and grouped (mixture-of-experts) calls.  A pass of the loop is four steps, whose ring positions
// are static; up to three steps that are no whole pass follow the loop.
constexpr int kWideStages = 4;
constexpr int kWideScaleRows = 16;   // a ring of 16 rows per wavefront: eight steps of one row, or of two (groups of 32 rows)
// RB: row blocks of 16 rows a wavefront owns: 16 (a 256-row tile) or 8 (a 128-row tile, for
// calls with few tiles: twice the tiles, half the K ranges and half the partial-tile traffic).
constexpr int wide_stage(int rb) { return rb * 2 * kBlockBytes; }                    // one stage of A
constexpr int wide_a(int rb) { return kWideStages * wide_stage(rb); }                // 128 / 64 KiB
constexpr int wide_lds(int rb) { return wide_a(rb) + 4 * kWideScaleRows * 256; }     // + the scale rows of four wavefronts
// memory operations per wavefront and step: its blocks of A, the scale row (groups of 32 / 16 rows: two, one per
// k block), two chunks (8-bit codes: four blocks)
constexpr int wide_ops(int rb, bool fp4 = false, bool w8 = false) { return rb / 2 + (fp4 ? 2 : 1) + (w8 ? 4 : 2); }

// A scale row of ones in bf16: what 8-bit codes with one scale a column are dequantised with.  Every code is a bf16 number, so
// the matrix cores get it exact and the column's scale goes into the fp32 sums, as in marlin_mid_gemm, between which and this
// kernel the estimates choose.  (Error against 64 bits in units of the output's rounding, scaled weights rounded to bf16: 1.38
// to 1.41, so: 1.00.  A row of ones instead of a form without scales: the same instructions in the loop, and no branch.)
template <bool FP8>
struct OnesRow {
  uint16_t bits[kStripN];
  constexpr OnesRow() : bits() {
    for (int i = 0; i < kStripN; ++i) bits[i] = Raw8<FP8>::kOne;
  }
};
__device__ __attribute__((aligned(128))) const OnesRow<false> kOnesInt8 = {};
__device__ __attribute__((aligned(128))) const OnesRow<true> kOnesFp8 = {};

// The end of a grouped tile whose rows go through the gated activation: the rows lie turned in LDS as wide_tile left them, a
// wavefront's at wave * kRows * 128, and every value is rounded as the GEMM's result would be, so that the bits are those of
// the GEMM and the activation after one another.  Bound by vector instructions (20 to 30 a result).  A launch and two passes over
// the rows of gate and up less; us a layer, activation in a launch of its own -> here: Mixtral-8x7B shapes, 4096 tokens 2500 -> 2395,
// 2000 tokens 1310 -> 1255; 8 experts 1024 x 2688, AWQ, 6002 tokens 298 -> 273; 16 of 2048 x 2816, 3000 tokens, top 4 481 -> 450; 64
// MXFP4 experts 2048 x 768, 4000 tokens, top 8 437 -> 426; 32 of 2880 x 2880, swigluoai, 2000 tokens, top 4 480 -> 465 (of which the
// tiles take 15 us longer and the activation took 30), 6000 tokens 1171 -> 1131.
//   alternating columns: a wavefront's own 64 columns are 32 results; `strip` is its strip
//   halves: wavefronts 0 and 1 have two strips of the gate half, 2 and 3 the same strips of the up half; wavefront w
//   then takes half w / 2 of the rows of strip `strip` + w % 2
// The ids of the rows go through `ids_lds`, 1 KiB of the wavefront's own, so that the rows are a loop: unrolled, its code would be
// fetched once a tile (with the division and expf of the library as well: 467 us for the 2000 tokens above that take 457
// with a launch of their own).
template <typename T, int RB>
__device__ __forceinline__ void store_gated(const TileParams& p, uint32_t a_lds, uint32_t ids_lds, int wave, int lane, int strip,
                                            const int (&ids)[RB]) {
  constexpr int kRows = 16 * RB;
  const int r8 = lane >> 3;
#pragma unroll
  for (int mb = 0; mb < RB; ++mb)
    asm volatile("ds_write_b32 %0, %1 offset:%2" ::"v"(ids_lds + 4 * (lane & 15)), "v"(ids[mb]), "i"(mb * 64) : "memory");
  const bool halves = p.gated_halves != 0;
  uint32_t at = a_lds + r8 * 128 + (((lane & 7) ^ r8) * 16), row_at = ids_lds + 4 * r8;
  if (halves) {
    at += (wave & 1) * (kRows * 128) + (wave >> 1) * (RB * 1024);
    row_at += (wave >> 1) * (8 * RB * 4);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();   // the rows of the other wavefronts
  } else {
    at += wave * (kRows * 128);
  }
  uint16_t* to_strip = p.gated + (halves ? (strip + (wave & 1)) * kStripN + 8 * (lane & 7) : strip * (kStripN / 2) + 4 * (lane & 7));
  const int steps = halves ? RB / 4 : RB / 2;   // of 32 rows
#pragma unroll 1
  for (int i = 0; i < steps; ++i, at += 4096, row_at += 128) {
    u32x4_t g[4], v[4];
    int row[4];
#define SONAR_READ_ROWS(IDS)                                                                                       \
  "ds_read_b32 %4, " IDS "\n\tds_read_b32 %5, " IDS " offset:32\n\tds_read_b32 %6, " IDS " offset:64\n\t"          \
  "ds_read_b32 %7, " IDS " offset:96\n\t"
#define SONAR_READ_LINES(A, B, C, D, AT)                                                                           \
  "ds_read_b128 " A ", " AT "\n\tds_read_b128 " B ", " AT " offset:1024\n\tds_read_b128 " C ", " AT " offset:2048\n\t" \
  "ds_read_b128 " D ", " AT " offset:3072\n\t"
#define SONAR_LINES_AND_ROWS "=&v"(g[0]), "=&v"(g[1]), "=&v"(g[2]), "=&v"(g[3]), "=&v"(row[0]), "=&v"(row[1]), "=&v"(row[2]), "=&v"(row[3])
    if (halves) {
      asm volatile(SONAR_READ_ROWS("%12") SONAR_READ_LINES("%0", "%1", "%2", "%3", "%13")
                       SONAR_READ_LINES("%8", "%9", "%10", "%11", "%14") "s_waitcnt lgkmcnt(0)"
                   : SONAR_LINES_AND_ROWS, "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
                   : "v"(row_at), "v"(at), "v"(at + 2 * (kRows * 128))
                   : "memory");
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        u32x4_t o;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o[j] = (uint32_t)silu_times<T>((uint16_t)g[u][j], (uint16_t)v[u][j]) |
                 ((uint32_t)silu_times<T>((uint16_t)(g[u][j] >> 16), (uint16_t)(v[u][j] >> 16)) << 16);
        if (row[u] >= 0) *reinterpret_cast<u32x4_t*>(to_strip + (long)row[u] * (p.size_n / 2)) = o;
      }
    } else {
      asm volatile(SONAR_READ_ROWS("%8") SONAR_READ_LINES("%0", "%1", "%2", "%3", "%9") "s_waitcnt lgkmcnt(0)"
                   : SONAR_LINES_AND_ROWS
                   : "v"(row_at), "v"(at)
                   : "memory");
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o[j] = swiglu_oai<T>((uint16_t)g[u][j], (uint16_t)(g[u][j] >> 16), p.gated_limit, p.gated_alpha);
        if (row[u] >= 0)
          *reinterpret_cast<uint2*>(to_strip + (long)row[u] * (p.size_n / 2)) = make_uint2(o[0] | (o[1] << 16), o[2] | (o[3] << 16));
      }
    }
#undef SONAR_READ_ROWS
#undef SONAR_READ_LINES
#undef SONAR_LINES_AND_ROWS
  }
}

// G32: a scale (and zero point) per 32 rows, i.e. one row of them per k block: MXFP4 always, integer codes when asked.
// NV (with FP4): NVFP4, a scale per 16 rows: the row of a k block then holds two groups of 128 bytes (the copy
// fetches one per half of the wavefront), and a lane, whose eight rows of a k block lie in one group, reads group
// kb / 2; the global scale multiplies the sums at the end.
// TWIN (with RB = 8): the form of marlin_tile_twin_kernel.
// The tile (tile_m, tile_n) of a launch, over K steps [k_first, k_tiles); `table`: of the row tiles of a grouped call;
// partial_at: index of the workgroup's partial tile in `partial`, or -1 when it has the whole of K.
template <typename T, bool HAS_ZP, bool GROUPED, int RB, bool FP4, int W8, bool G32, bool NV, bool TWIN = false>
__device__ __forceinline__ void wide_tile(const TileParams& p, const int32_t* table, float4* partial, const int tile_m,
                                          const int tile_n, const int k_first, const int k_tiles, const int partial_at) {
  typedef typename Dq<T>::vec8 vec8;
  typedef typename Dq4Of<T, FP4, NV>::type D4;   // integer codes, or float4_e2m1f (MXFP4: bf16; NVFP4)
  typedef typename Dq8Of<T, W8 == 2>::type D8;   // 8-bit integer (W8 = 1) or floating-point (W8 = 2) codes
  typedef typename std::conditional<W8 != 0, typename D8::Col, typename D4::Col>::type Col;
  typedef typename Dq<T>::Mid Mid;
  static_assert(W8 == 0 || (!HAS_ZP && !FP4), "8-bit codes: symmetric");
  static_assert(wide_ops(RB, G32, W8 != 0) <= 2 * RB, "a step's memory operations go out behind its row blocks");
  static_assert(!FP4 || G32, "MXFP4 has a scale per 32 rows");
  constexpr int kChunkLoads = W8 ? 2 : 1;   // 16-byte loads per lane and k block: 8-bit codes come as a block of
                                            // the low four and a block of the high four of a lane's eight rows
  static_assert(!FP4 || ((NV || std::is_same<T, __bf16>::value) && !HAS_ZP), "MXFP4: bf16; float4 codes: no zero points");
  static_assert(!NV || (FP4 && RB == 16), "NVFP4 is float4 codes; 256-row tiles");
  static_assert(!(W8 != 0 && G32) || RB == 16, "8-bit codes with groups of 32 rows: 256-row tiles");
  static_assert(RB == 16 || RB == 8, "256-row tiles or 128-row tiles");
  static_assert(!TWIN || (RB == 8 && W8 == 0 && !NV), "4-bit integers and MXFP4");
  constexpr int kRows = 16 * RB;
  constexpr int kStage = wide_stage(RB), kWideA = wide_a(RB), kWideOps = wide_ops(RB, G32, W8 != 0);
  constexpr int kAgprBlocks = RB == 16 ? 14 : RB;   // row blocks whose accumulators sit in AGPRs
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col16 = lane & 15;
  const int kb = lane >> 4;
  const uint32_t magic = magic_register();
  const bool grouped = p.num_groups > 1;
  constexpr bool kScaleSums = W8 != 0 && !G32 && std::is_same<T, __bf16>::value;   // with one group (OnesRow)

  // Grouped calls: row tile t is up to four consecutive 64-slot blocks of one expert, listed in
  // tile_table; rows are slots of sorted_ids (as in marlin_tile_async_kernel).
  int first_slot = 0, tile_rows = kRows;
  long expert = 0;
  if (GROUPED) {
    first_slot = table[1 + 3 * tile_m] * 64;
    tile_rows = table[2 + 3 * tile_m] * 64;
    expert = __builtin_amdgcn_readfirstlane(table[3 + 3 * tile_m]);
  }
  const int m0 = tile_m * kRows;
  const int strip0 = tile_n * (kTileN / kStripN);
  const int strips_here = min(kTileN / kStripN, p.size_n / kStripN - strip0);
  const bool active = wave < strips_here;
  // a wavefront past the last strip works on the last strip again and stores nothing
  int strip = strip0 + (active ? wave : strips_here - 1);
  // silu_and_mul at the end: a tile is 128 columns of the gate and the same 128 of the up half (the host checks: all strips are there)
  if (GROUPED && p.gated != nullptr && p.gated_halves)
    strip = 2 * tile_n + (wave & 1) + (wave >> 1) * (p.size_n / (2 * kStripN));

  // ---- sources (regions of A as in marlin_tile_async_kernel; wavefront w fills RB / 2 regions)
  // Memory operations take a scalar base and a 32-bit offset a lane where they can: with a 64-bit address a lane each holds up the
  // wavefront's other instructions 20 cycles longer.  (M = 8192, K = 4096, N = 28672, fp16 1368 -> 1355 us; one tile alone 74.2 -> 73.4.)
  // Dense calls: a wavefront's rows of A are within 32 bits of its first (wide_rows_within_32_bits); the rows of a grouped tile
  // may be anywhere.
  const int a_first = GROUPED ? 0 : min(m0 + 4 * RB * wave, p.size_m - 1);
  const char* a_rows = reinterpret_cast<const char*>(p.a + (long)a_first * p.lda);
  constexpr bool kFarRows = GROUPED && !TWIN;
  typename std::conditional<kFarRows, const char*, uint32_t>::type a_src[RB / 2];
#pragma unroll
  for (int i = 0; i < RB / 2; ++i) {
    const int region = (RB / 2) * wave + i;
    const int r8 = lane >> 3;
    const int in_tile = 16 * (region >> 1) + 8 * (region & 1) + r8;
    int row;
    if (GROUPED) {
      const int id = in_tile < tile_rows ? p.sorted_ids[first_slot + in_tile] : p.rows_total;
      // padding slots read row 0, never stored
      row = (unsigned)id < (unsigned)p.rows_total ? (p.a_by_slot ? first_slot + in_tile : id / p.top_k) : 0;
    } else {
      row = m0 + in_tile;
      if (row >= p.size_m) row = p.size_m - 1;   // rows past M are computed and never stored
    }
    if constexpr (kFarRows) a_src[i] = a_rows + ((long)row * p.lda + 8 * ((lane & 7) ^ r8)) * 2;
    else a_src[i] = (uint32_t)(row - a_first) * (uint32_t)(p.lda * 2) + 16 * ((lane & 7) ^ r8);
  }
  const char* b_base = reinterpret_cast<const char*>(p.b + expert * p.expert_b_stride) +
                       (size_t)(unsigned)(strip * p.chunks_per_strip) * (1024 * kChunkLoads);
  const uint32_t b_off = 16 * lane;
  // (zero points: the lower half of the wavefront copies scales, the upper half zero points, from bases of their own)
  const char* s_base = reinterpret_cast<const char*>(p.scales + expert * p.expert_s_stride + strip * kStripN);
  if (kScaleSums && !grouped) s_base = W8 == 2 ? reinterpret_cast<const char*>(&kOnesFp8) : reinterpret_cast<const char*>(&kOnesInt8);
  const char* z_src = reinterpret_cast<const char*>(p.zeros + expert * p.expert_z_stride + strip * 8 + (lane & 7));
  const long s_group_stride = (long)p.size_n * 2;
  const uint32_t sz_group_stride = HAS_ZP && lane >= 32 ? (uint32_t)p.size_n / 2 : (uint32_t)s_group_stride;
  const char* sz_src = HAS_ZP && lane >= 32 ? z_src : s_base + 4 * (lane & 31);
  const uint32_t s_lane = 4 * (lane & 31) + (NV ? (lane >> 5) * (uint32_t)s_group_stride : 0);   // (NVFP4: the next group's row)
  // steps per group as a shift (the host checks: group_size = 64 * 2^i)
  const int group_shift = grouped ? 31 - __builtin_clz(p.group_size / kTileK) : 0;
  char* sring = smem + kWideA + wave * (kWideScaleRows * 256);
  const uint32_t a_lds = (uint32_t)(uintptr_t)(lds_void_t*)smem;
  const uint32_t s_lds = (uint32_t)(uintptr_t)(lds_void_t*)sring;

  u32x4_t wq[kWideStages][2 * kChunkLoads];   // packed chunks in flight or waiting (8-bit: [2 b + h], h = high rows)
  // the scale row of step kt (clamped to the last step) into its ring position; MXFP4: the row of
  // k block h of the step (groups of 32 rows), ring position 2 (kt - k_first) + h
  auto issue_scales = [&](int kt, int h) __attribute__((always_inline)) {
    const int k = min(kt, k_tiles - 1);
    const int grp = G32 ? (NV ? 2 : 1) * (2 * k + h) : (grouped ? k >> group_shift : 0);
    const int at = G32 ? 2 * (kt - k_first) + h : kt - k_first;
    if constexpr (HAS_ZP)
      __builtin_amdgcn_global_load_lds((glb_void_t*)(sz_src + (uint64_t)(uint32_t)grp * sz_group_stride),
                                       (lds_void_t*)(sring + (at & (kWideScaleRows - 1)) * 256), 4, 0, 0);
    else
      copy_to_lds<4>(s_lds + (at & (kWideScaleRows - 1)) * 256, s_lane, s_base + grp * s_group_stride);
  };
  // memory operation `idx` (0..kWideOps-1) issued for step kt into ring position `slot`: first the
  // blocks of A of step kt, then the scale row of step kt + 1, then the two chunks of step kt
  auto issue_one = [&](int kt, int slot, int idx) __attribute__((always_inline)) {
    const int k = min(kt, k_tiles - 1);
    if (idx < RB / 2) {
      const uint32_t to = slot * kStage + ((RB / 2) * wave + idx) * kBlockBytes;
      if constexpr (kFarRows)
        __builtin_amdgcn_global_load_lds((glb_void_t*)(a_src[idx] + (long)k * (kTileK * 2)), (lds_void_t*)(smem + to), 16, 0, 0);
      else
        copy_to_lds<16>(a_lds + to, a_src[idx], a_rows + (long)k * (kTileK * 2));
    } else if (idx < RB / 2 + (G32 ? 2 : 1)) {
      issue_scales(kt + 1, idx - RB / 2);
    } else {
      const int c = idx - RB / 2 - (G32 ? 2 : 1);
      asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3"
                   : "=&v"(wq[slot][c]) : "v"(b_off), "s"(b_base + (size_t)k * (2048 * kChunkLoads)), "i"(c * 1024) : "memory");
    }
  };

  uint32_t s_off[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) s_off[j] = 2 * scale_slot(16 * j + col16, TWIN || grouped);
  const uint32_t z_off = 128 + 4 * zero_point_word(col16);
  // operand lane (kb, col16) of row block 0, k block b of stage 0: piece 4 b + kb of row col16
  uint32_t a_base[2];
#pragma unroll
  for (int b = 0; b < 2; ++b)
    a_base[b] = a_lds + (col16 >> 3) * kBlockBytes + (col16 & 7) * 128 + (((4 * b + kb) ^ (col16 & 7)) * 16);

  floatx4_t acc[4][RB];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int mb = 0; mb < RB; ++mb) {
      if constexpr (TWIN) {   // (copies of one register of zeros need that register beside the 128 AGPRs there are)
        asm volatile("s_nop 1\n\tv_mfma_f32_16x16x32_f16 %0, %1, %1, 0" : "=a"(acc[nb][mb]) : "v"(u32x4_t{0, 0, 0, 0}));
        continue;
      }
      acc[nb][mb] = floatx4_t{0.f, 0.f, 0.f, 0.f};
      // the zeros sit where the MFMAs will hold the accumulator, so that the value has one home
      // on every path to the stores
      if (mb < kAgprBlocks) asm volatile("" : "+a"(acc[nb][mb]));
      else asm volatile("" : "+v"(acc[nb][mb]));
    }

  constexpr int kAhead = TWIN ? 3 : 4, kAv = TWIN ? 4 : 8;   // operands of A are read this many row blocks ahead
  u32x4_t av[kAv];        // row block rb in av[rb % kAv]
  uint32_t wb[2][4][4];   // dequantised chunk of k block b: four operand blocks of 16 columns, four pairs each
  uint32_t sb0 = 0, sb1 = 0, sb2 = 0, sb3 = 0, zw = 0;
  // a shift more for two nibbles of a word, and half the constants, which would not fit the registers
  constexpr bool kOneForm = TWIN && HAS_ZP && std::is_same<T, __bf16>::value;
  constexpr int kColSets = TWIN ? 1 : 2;
  Col cols[kColSets][4];  // by the parity of the step (MXFP4: of the k block); TWIN: a column block's are replaced behind its last use

#define SONAR_WIDE_READ(dst, base, off) \
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(dst) : "v"(base), "i"(off) : "memory")
#define SONAR_WIDE_LANDED(n, reg) asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(reg) : "n"(n) : "memory")

  auto scales_start = [&](int kt, int h) __attribute__((always_inline)) {
    const uint32_t r_at = s_lds + ((G32 ? 2 * (kt - k_first) + h : kt - k_first) & (kWideScaleRows - 1)) * 256 +
                          (NV ? 128 * (kb >> 1) : 0);
    if constexpr (TWIN) {
      asm volatile(
          "ds_read_u16 %0, %5\n\t"
          "ds_read_u16 %1, %5 offset:4\n\t"
          "ds_read_u16 %2, %5 offset:8\n\t"
          "ds_read_u16 %3, %5 offset:12\n\t"
          "ds_read_b32 %4, %6"
          : "=&v"(sb0), "=&v"(sb1), "=&v"(sb2), "=&v"(sb3), "=&v"(zw)
          : "v"(r_at + s_off[0]), "v"(HAS_ZP ? r_at + z_off : r_at + s_off[0])
          : "memory");
      return;
    }
    asm volatile(
        "ds_read_u16 %0, %5\n\t"
        "ds_read_u16 %1, %6\n\t"
        "ds_read_u16 %2, %7\n\t"
        "ds_read_u16 %3, %8\n\t"
        "ds_read_b32 %4, %9"
        : "=&v"(sb0), "=&v"(sb1), "=&v"(sb2), "=&v"(sb3), "=&v"(zw)
        : "v"(r_at + s_off[0]), "v"(r_at + s_off[1]), "v"(r_at + s_off[2]), "v"(r_at + s_off[3]),
          "v"(NV ? r_at + s_off[0] : r_at + z_off)
        : "memory");
  };
  auto make_col = [&](int set, int j) __attribute__((always_inline)) {
    const uint32_t sbits = j == 0 ? sb0 : j == 1 ? sb1 : j == 2 ? sb2 : sb3;
    int z = 8;
    if (HAS_ZP) z = (int)((zw >> zero_point_shift(16 * j + col16)) & 0xFu);
    if constexpr (W8 != 0) cols[set % kColSets][j] = D8::make_col((uint16_t)sbits);
    else cols[set % kColSets][j] = D4::make_col((uint16_t)sbits, z);
  };
  auto word_of = [](const u32x4_t& q, int j) __attribute__((always_inline)) -> uint32_t {
    return j == 0 ? q.x : j == 1 ? q.y : j == 2 ? q.z : q.w;
  };
  // acc[j][rb] += W block j (16 columns) x A row block rb, in place; with 16 row blocks the last two in VGPRs
  auto mfma = [&](int B, int j, int rb) __attribute__((always_inline)) {
    const u32x4_t w = u32x4_t{wb[B][j][0], wb[B][j][1], wb[B][j][2], wb[B][j][3]};
    if constexpr (std::is_same<T, _Float16>::value) {
      if (rb < kAgprBlocks) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[j][rb]) : "v"(w), "v"(av[rb % kAv]));
      else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(acc[j][rb]) : "v"(w), "v"(av[rb % kAv]));
    } else {
      if (rb < kAgprBlocks) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[j][rb]) : "v"(w), "v"(av[rb % kAv]));
      else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc[j][rb]) : "v"(w), "v"(av[rb % kAv]));
    }
  };

  // One k block of step kt: RB row blocks of four MFMAs.  R: ring position of the step's
  // stage, B: the k block.  Behind the MFMAs of a row block, one instruction each: one pair
  // (with 8 row blocks: two) of the 16 of the next half step's chunk; then B = 0: the scales of
  // step kt + 1 become per-column constants; B = 1: one memory operation of step kt + 3.
  auto chunk = [&](const int R, const int B, const int kt) __attribute__((always_inline)) {
    const int NR = B ? (R + 1) & 3 : R;   // stage and k block of the half step after this one
    const int NB = B ^ 1;
    // constants of the step the next half step belongs to (MXFP4: of the next k block)
    const int set = G32 ? NB : (B ? (R + 1) & 1 : R & 1);
    const uint32_t a_cur = a_base[B] + R * kStage;
    const uint32_t a_next = a_base[NB] + NR * kStage;
    const u32x4_t& q4 = B ? wq[NR][0] : wq[R][kChunkLoads];                         // 8-bit: the low four rows
    const u32x4_t& q4h = B ? wq[NR][kChunkLoads - 1] : wq[R][2 * kChunkLoads - 1];   // 8-bit: the high four rows
    constexpr int kPairs = 16 / RB;   // pairs of weights dequantised per row block
    uint32_t r_lo = 0;     // MXFP4: rows (0, 2) or (4, 6) of the word in hand, waiting for their odd partners
    uint32_t nv_lo = 0, nv_hi = 0;   // NVFP4, bf16: the same rows as fp32 products
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const int j = (kPairs * rb) >> 2, part = (kPairs * rb) & 3;
      // reads started after the one of this row block: those of the next kAhead - 1 row blocks,
      // and the five scale reads of slot 0 (first half; MXFP4: either half)
      if ((B == 0 || G32) && rb >= 1 && rb <= kAhead) SONAR_WIDE_LANDED(kAhead - 1 + 5, av[rb % kAv]);
      else SONAR_WIDE_LANDED(kAhead - 1, av[rb % kAv]);
      // behind this wait the scale reads of slot 0 have landed: from here on the registers they fill
      // hold the scales (without this the compiler is free to use them any time after slot 0)
      if ((B == 0 || G32) && rb == (kAhead + 1 < RB ? kAhead + 1 : RB - 1))
        asm volatile("" : "+v"(sb0), "+v"(sb1), "+v"(sb2), "+v"(sb3), "+v"(zw) : : "memory");
      if (rb + kAhead < RB) SONAR_WIDE_READ(av[(rb + kAhead) % kAv], a_cur, (rb + kAhead) * 2048);
      else SONAR_WIDE_READ(av[(rb + kAhead) % kAv], a_next, (rb + kAhead - RB) * 2048);
      // the scales of the step after this one (MXFP4: of its k block B, two half steps ahead)
      if (rb == 0 && (B == 0 || G32)) scales_start(kt + 1, B);
      const uint32_t qw = word_of(q4, j);
      if constexpr (W8 != 0) {
        // a register of half a column block (two of four rows of 16 columns; with 8 row blocks: both), spread over three
        // matrix instructions.  (Half a column block in one piece behind every second row block, 14 instructions behind
        // one that hides four: fp8, bf16, M = 2000, K = 2944, N = 8832 167 -> 133 us; M = 1323, K = N = 8832 235 -> 203; MXFP8,
        // M = 3000, K = 2944, N = 6144 168 -> 150; uint8b128, M = 1000, K = 4096, N = 6144 68 -> 58.)
        const int piece = RB == 8 ? rb : rb >> 1, jj = piece >> 1, half = piece & 1, first = RB == 8 ? 0 : rb & 1;
        const uint32_t w8 = word_of(half ? q4h : q4, jj);
        mfma(B, 0, rb);
        const uint32_t x = D8::stage1(w8, first, magic);
        uint32_t x2 = 0;
        if (RB == 8) x2 = D8::stage1(w8, 1, magic);
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 1, rb);
        const typename D8::Mid y = D8::stage2(x, cols[set % kColSets][jj]);
        typename D8::Mid y2 = y;
        if (RB == 8) y2 = D8::stage2(x2, cols[set % kColSets][jj]);
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 2, rb);
        wb[NB][jj][2 * half + first] = D8::stage3(y, cols[set % kColSets][jj]);
        if (RB == 8) wb[NB][jj][2 * half + 1] = D8::stage3(y2, cols[set % kColSets][jj]);
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 3, rb);
      } else if constexpr (NV && std::is_same<T, _Float16>::value) {
        // the pair of codes read as fp16 numbers (value * 2^-14) times scale * 2^14 in one packed multiply
        // (DqNvF4<_Float16>::pair, a piece behind each MFMA)
        mfma(B, 0, rb);
        const uint32_t y = part == 3 ? qw : qw << (12 - 4 * part);
        const uint32_t mag = (y >> 3) & 0x0E000E00u;
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 1, rb);
        const uint32_t hbits = (y & 0x80008000u) | mag;
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 2, rb);
        wb[NB][j][part] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, hbits) *
                                                           __builtin_bit_cast(half2_t, cols[set % kColSets][j].s2));
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 3, rb);
      } else if constexpr (FP4 && kPairs == 2) {
        // MXFP4 with 8 row blocks: the conversions of an even and an odd part (rows (0,2) and (1,3), or (4,6) and
        // (5,7)) and their two byte permutes behind one row block
        mfma(B, 0, rb);
        const float sc = cols[set % kColSets][j].s;
        const uint32_t r_e = __builtin_bit_cast(uint32_t, part == 0 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(qw, sc, 0)
                                                                    : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(qw, sc, 1));
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 1, rb);
        const uint32_t r_o = __builtin_bit_cast(uint32_t, part == 0 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(qw, sc, 2)
                                                                    : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(qw, sc, 3));
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 2, rb);
        wb[NB][j][part] = __builtin_amdgcn_perm(r_o, r_e, 0x05040100u);
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 3, rb);
        wb[NB][j][part + 1] = __builtin_amdgcn_perm(r_o, r_e, 0x07060302u);
      } else if constexpr (NV) {
        // bf16: one hardware conversion with a unit scale per row block (rows (0,2), (1,3), (4,6), (5,7) of the
        // column), the two values times the scale in fp32; behind the second and the fourth, the two byte
        // permutes that cut the products back to bf16 and put four rows in order (DqNvF4<__bf16>::word)
        mfma(B, 0, rb);
        const float sc = cols[set % kColSets][j].s;
        const uint32_t r = __builtin_bit_cast(
            uint32_t, part == 0   ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(qw, 1.0f, 0)
                      : part == 1 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(qw, 1.0f, 2)
                      : part == 2 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(qw, 1.0f, 1)
                                  : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(qw, 1.0f, 3));
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 1, rb);
        const float f_lo = __uint_as_float(r << 16), f_hi = __uint_as_float(r & 0xFFFF0000u);
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 2, rb);
        const uint32_t p_lo = __float_as_uint(f_lo * sc), p_hi = __float_as_uint(f_hi * sc);
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 3, rb);
        if (part & 1) {
          wb[NB][j][part - 1] = __builtin_amdgcn_perm(p_lo, nv_lo, 0x07060302u);
          wb[NB][j][part] = __builtin_amdgcn_perm(p_hi, nv_hi, 0x07060302u);
        } else {
          nv_lo = p_lo;
          nv_hi = p_hi;
        }
      } else if constexpr (FP4) {
        // one hardware conversion per row block (two rows of the column each: (0,2), (1,3), (4,6),
        // (5,7)); behind the second and the fourth, the two byte permutes that put four rows in order
        mfma(B, 0, rb);
        const float sc = cols[set % kColSets][j].s;
        const uint32_t r = __builtin_bit_cast(
            uint32_t, part == 0   ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(qw, sc, 0)
                      : part == 1 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(qw, sc, 2)
                      : part == 2 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(qw, sc, 1)
                                  : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(qw, sc, 3));
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 1, rb);
        if (part & 1) wb[NB][j][part - 1] = __builtin_amdgcn_perm(r, r_lo, 0x05040100u);
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 2, rb);
        if (part & 1) wb[NB][j][part] = __builtin_amdgcn_perm(r, r_lo, 0x07060302u);
        else r_lo = r;
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 3, rb);
      } else {
        mfma(B, 0, rb);
        const uint32_t x = Dq<T>::stage1(part < 2 ? qw : qw >> 8, part, magic);
        uint32_t x2 = 0;
        if (kPairs == 2) x2 = kOneForm ? Dq<T>::stage1(qw >> (part < 2 ? 4 : 12), part, magic) : Dq<T>::stage1(part < 2 ? qw : qw >> 8, part + 1, magic);
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 1, rb);
        const Mid y = Dq<T>::stage2(x, cols[set % kColSets][j], part);
        Mid y2 = y;
        if (kPairs == 2) y2 = Dq<T>::stage2(x2, cols[set % kColSets][j], kOneForm ? part : part + 1);
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 2, rb);
        wb[NB][j][part] = Dq<T>::stage3(y, cols[set % kColSets][j]);
        if (kPairs == 2) wb[NB][j][part + 1] = Dq<T>::stage3(y2, cols[set % kColSets][j]);
        __builtin_amdgcn_sched_barrier(0);
        mfma(B, 3, rb);
      }
      if (B == 0 || G32) {
        // the scale reads of slot 0 have landed behind the wait of slot kAhead + 1; they become the
        // constants of the step after this one (MXFP4: of its k block B, whose set the chunk being
        // dequantised here does not use)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (rb == (kAhead + 1 + c < RB ? kAhead + 1 + c : RB - 1)) make_col(G32 ? B : (R + 1) & 1, c);
      }
      if (B == 1 && rb < kWideOps) issue_one(kt + 3, (R + 3) & 3, rb);
      // (8-bit codes with 8 row blocks: nine operations, the ninth behind the first row block too)
      if (B == 1 && RB + rb < kWideOps) issue_one(kt + 3, (R + 3) & 3, RB + rb);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto step = [&](const int R, int kt) __attribute__((always_inline)) {
    chunk(R, 0, kt);
    // stage kt + 1 (its blocks of A, its two chunks) and the scale row of step kt + 2 have landed
    // once only the operations issued in step kt - 1 are outstanding
    asm volatile("s_waitcnt vmcnt(%2)"
                 : "+v"(wq[(R + 1) & 3][0]), "+v"(wq[(R + 1) & 3][1])
                 : "n"(kWideOps)
                 : "memory");
    if constexpr (W8 != 0) asm volatile("" : "+v"(wq[(R + 1) & 3][2]), "+v"(wq[(R + 1) & 3][3]) : : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    chunk(R, 1, kt);
    // the chunk of the next step is dequantised up to here: without this the compiler moves all of it behind the branch
    // between the steps, where no matrix instruction hides it
#pragma unroll
    for (int j = 0; j < 4; ++j)
      asm volatile("" : "+v"(wb[0][j][0]), "+v"(wb[0][j][1]), "+v"(wb[0][j][2]), "+v"(wb[0][j][3]));
  };

  // ---- prologue: the scale row of the first step, then what steps k_first - 3 .. k_first - 1 would have issued
  issue_scales(k_first, 0);
  if (G32) issue_scales(k_first, 1);
#pragma unroll
  for (int idx = 0; idx < kWideOps; ++idx) issue_one(k_first, 0, idx);
#pragma unroll
  for (int idx = 0; idx < kWideOps; ++idx) issue_one(k_first + 1, 1, idx);
#pragma unroll
  for (int idx = 0; idx < kWideOps; ++idx) issue_one(k_first + 2, 2, idx);
  asm volatile("s_waitcnt vmcnt(%2)" : "+v"(wq[0][0]), "+v"(wq[0][1]) : "n"(2 * kWideOps) : "memory");
  if constexpr (W8 != 0) asm volatile("" : "+v"(wq[0][2]), "+v"(wq[0][3]) : : "memory");
  __builtin_amdgcn_s_barrier();
  auto second_block = [&]() __attribute__((always_inline)) {   // the constants of k block 1 of the first step
    scales_start(k_first, 1);
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(sb0), "+v"(sb1), "+v"(sb2), "+v"(sb3), "+v"(zw) : : "memory");
#pragma unroll
    for (int j = 0; j < 4; ++j) make_col(1, j);
  };
  if (G32 && !TWIN) second_block();
  scales_start(k_first, 0);
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(sb0), "+v"(sb1), "+v"(sb2), "+v"(sb3), "+v"(zw) : : "memory");
#pragma unroll
  for (int j = 0; j < 4; ++j) make_col(0, j);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    u32x4_t w;
    if constexpr (W8 != 0) {
      const uint2 lo = D8::word4(word_of(wq[0][0], j), cols[0][j], magic);
      const uint2 hi = D8::word4(word_of(wq[0][1], j), cols[0][j], magic);
      w = u32x4_t{lo.x, lo.y, hi.x, hi.y};
    } else {
      w = __builtin_bit_cast(u32x4_t, D4::word(word_of(wq[0][0], j), cols[0][j], magic));
    }
    wb[0][j][0] = w.x;
    wb[0][j][1] = w.y;
    wb[0][j][2] = w.z;
    wb[0][j][3] = w.w;
  }
  if (G32 && TWIN) second_block();
#pragma unroll
  for (int rb = 0; rb < kAhead; ++rb) SONAR_WIDE_READ(av[rb], a_base[0], rb * 2048);
  __builtin_amdgcn_sched_barrier(0);

  // Whole passes without a branch between their steps, then up to three steps.  (With a branch behind every step: int4, M = 8192,
  // K = 4096, N = 28672 1520 us against 1498, M = 4000, K = 1152, N = 6144 71 against 64.)
  int kt = k_first;
  for (; kt + 4 <= k_tiles; kt += 4) {
    step(0, kt);
    step(1, kt + 1);
    step(2, kt + 2);
    step(3, kt + 3);
  }
  if (kt < k_tiles) {
    step(0, kt);
    if (kt + 1 < k_tiles) {
      step(1, kt + 1);
      if (kt + 2 < k_tiles) step(2, kt + 2);
    }
  }
  // nothing in flight may outlive the wavefront (the copies of the steps past the end, the two
  // operand reads of the last half step), and the matrix pipeline drains before the results are read
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
  // the registers those operations were still to fill stay untouched up to here
#pragma unroll
  for (int i = 0; i < kWideStages; ++i)
#pragma unroll
    for (int c = 0; c < 2 * kChunkLoads; ++c) asm volatile("" : "+v"(wq[i][c]) : : "memory");
#pragma unroll
  for (int i = 0; i < kAv; ++i) asm volatile("" : "+v"(av[i]) : : "memory");
  asm volatile("" : "+v"(sb0), "+v"(sb1), "+v"(sb2), "+v"(sb3), "+v"(zw) : : "memory");
  __builtin_amdgcn_sched_barrier(0);
#undef SONAR_WIDE_LANDED
#undef SONAR_WIDE_READ

  __builtin_amdgcn_s_barrier();   // nobody reads the stages of A any more
  if (!active) return;
  floatx4_t sum_scale[4];
  if constexpr (kScaleSums) {
    const uint16_t* row = p.scales + expert * p.expert_s_stride + strip * kStripN;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sum_scale[nb][r] = grouped ? 1.f : Raw8<W8 == 2>::column_scale(row[scale_slot(16 * nb + 4 * kb + r, false)]);
  }
  if (!TWIN && partial_at >= 0) {
    // partial tile of this K range, in the order tile_reduce_kernel reads: 1-KiB blocks
    // (half of the rows, strip, column block, row block)
    float4* dst = partial + ((size_t)partial_at * kRows + wave * 32) * 64 + lane;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int mb = 0; mb < RB; ++mb) {
        if (mb < kAgprBlocks) asm volatile("" : "+a"(acc[nb][mb]));   // still in its AGPRs here
        const floatx4_t v = kScaleSums ? acc[nb][mb] * sum_scale[nb] : acc[nb][mb];
        dst[((mb >> 3) * 128 + nb * 8 + (mb & 7)) * 64] = make_float4(v.x, v.y, v.z, v.w);
        __builtin_amdgcn_sched_barrier(0);   // one accumulator at a time leaves the AGPRs
      }
    return;
  }
  const uint16_t* bias_src = p.bias ? p.bias + expert * p.expert_bias_stride + strip * kStripN : nullptr;
  float gs = 1.f;   // NVFP4: the global scale multiplies the sum before anything else (marlin_template.h:1661-1665)
  if (NV && p.global_scale) gs = p.global_scale[GROUPED ? expert : 0];
  float bias[4][4];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      bias[nb][r] = bias_src ? Dq<T>::to_float(bias_src[scale_slot(16 * nb + 4 * kb + r, false)]) : 0.f;
  // Grouped: the rows of C, and their weights, of all row blocks at once.  (One row block after the other, every one waited
  // for two loads, and the sixteen waits took about 15 us: 32 MXFP4 experts 2880 x 2880, 2000 tokens 504 -> 470 us; 8
  // experts 1280 x 1408, 3655 tokens 279 -> 259; 8 experts 2816 x 1280, 1254 tokens 130 -> 117.)
  int ids[GROUPED ? RB : 1];
  float weights[GROUPED ? RB : 1];
  if constexpr (GROUPED) {
#pragma unroll
    for (int mb = 0; mb < RB; ++mb) {
      const int r = 16 * mb + col16;
      ids[mb] = r < tile_rows ? p.sorted_ids[first_slot + r] : -1;
    }
#pragma unroll
    for (int mb = 0; mb < RB; ++mb) {
      if ((unsigned)ids[mb] >= (unsigned)p.rows_total) ids[mb] = -1;   // padding slot
      weights[mb] = p.mul_topk && ids[mb] >= 0 ? p.topk_weights[ids[mb]] : 1.f;
    }
  }
  // Rows leave as whole 128-byte lines, turned in the stages of A, which are nobody's any more: a wavefront's rows x 128 bytes,
  // 16-byte piece q of row r at slot q ^ (r % 8).  (8-byte pieces straight from the accumulators were 32
  // bytes a row and store: M = 8192, K = 4096, N = 28672, fp16 1442 -> 1412 us; MXFP8, M = 4000, K = 2048, N = 6016 112 -> 107; NVFP4,
  // M = 2222, K = 4096, N = 8192 148 -> 142; 32 MXFP4 experts 2880 x 2880, 2000 tokens 475 -> 462; 8 experts 1024 x 2688, AWQ, 6002
  // tokens 533 -> 513; Mixtral-8x7B shapes, 4096 tokens 2515 -> 2487.)
  const uint32_t turn = a_lds + wave * (kRows * 128);
  uint32_t turn_in[4];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
    turn_in[nb] = turn + col16 * 128 + (((2 * nb + (kb >> 1)) ^ (col16 & 7)) * 16) + 8 * (kb & 1);
#pragma unroll
  for (int mb = 0; mb < RB; ++mb) {
    // the routing weight is rounded to the activation type and the product is
    // formed and rounded in that type (marlin_template.h(moe):1893-1897)
    if (GROUPED && __builtin_amdgcn_ballot_w64(ids[mb] >= 0) == 0) continue;   // sixteen padding slots
    float row_w = 1.f;
    if constexpr (GROUPED) row_w = Dq<T>::to_float(Dq<T>::from_float(weights[mb]));
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      if (mb < kAgprBlocks) asm volatile("" : "+a"(acc[nb][mb]));   // still in its AGPRs here
      const floatx4_t v = kScaleSums ? acc[nb][mb] * sum_scale[nb] : NV ? acc[nb][mb] * gs : acc[nb][mb];
      uint16_t o[4] = {Dq<T>::from_float(v.x + bias[nb][0]), Dq<T>::from_float(v.y + bias[nb][1]),
                       Dq<T>::from_float(v.z + bias[nb][2]), Dq<T>::from_float(v.w + bias[nb][3])};
      if (GROUPED && p.mul_topk) {
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = Dq<T>::from_float(Dq<T>::to_float(o[i]) * row_w);
      }
      const uint2 packed = make_uint2((uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16));
      asm volatile("ds_write_b64 %0, %1 offset:%2" ::"v"(turn_in[nb]), "v"(packed), "i"(mb * 2048) : "memory");
      __builtin_amdgcn_sched_barrier(0);   // one accumulator at a time leaves the AGPRs
    }
  }
  const int r8 = lane >> 3;
  if constexpr (GROUPED) {
    if (p.gated != nullptr) {
      store_gated<T, RB>(p, a_lds, s_lds, wave, lane, p.gated_halves ? 2 * tile_n : strip, ids);
      return;
    }
  }
  const uint32_t turn_out = turn + r8 * 128 + (((lane & 7) ^ r8) * 16);
  uint16_t* c_strip = p.c + strip * kStripN + 8 * (lane & 7);
  const bool c_aligned = (reinterpret_cast<uintptr_t>(p.c) & 15) == 0;
#pragma unroll
  for (int i = 0; i < 2 * RB; i += 4) {
    int ids_out[4];   // of the rows that this lane stores
    if constexpr (GROUPED) {
#pragma unroll
      for (int u = 0; u < 4; ++u) ids_out[u] = __shfl(ids[(i + u) >> 1], 8 * (u & 1) + r8);
    }
    u32x4_t line[4];   // (a wavefront's LDS operations complete in order)
    asm volatile(
        "ds_read_b128 %0, %4 offset:%5\n\tds_read_b128 %1, %4 offset:%6\n\t"
        "ds_read_b128 %2, %4 offset:%7\n\tds_read_b128 %3, %4 offset:%8\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(line[0]), "=&v"(line[1]), "=&v"(line[2]), "=&v"(line[3])
        : "v"(turn_out), "i"(i * 1024), "i"(i * 1024 + 1024), "i"(i * 1024 + 2048), "i"(i * 1024 + 3072)
        : "memory");
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int row = GROUPED ? ids_out[u] : m0 + 8 * (i + u) + r8;
      if ((unsigned)row < (unsigned)(GROUPED ? p.rows_total : p.size_m)) {
        uint16_t* to = c_strip + (long)row * p.size_n;
        if (c_aligned) {
          *reinterpret_cast<u32x4_t*>(to) = line[u];
        } else {
          *reinterpret_cast<uint2*>(to) = make_uint2(line[u].x, line[u].y);
          *reinterpret_cast<uint2*>(to + 4) = make_uint2(line[u].z, line[u].w);
        }
      }
    }
  }
}

// One tile size.
template <typename T, bool HAS_ZP, bool GROUPED = false, int RB = 16, bool FP4 = false, int W8 = 0, bool G32 = FP4,
          bool NV = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void marlin_tile_wide_kernel(
    const TileParams p) {
  int tile, tile_m, tile_n, split;
  bool whole_k;
  // Grouped: the launch is sized for the most row tiles the routing could make; the tiles there are
  // (tile_table[0]) are numbered here in bands of four row tiles, so that the 32 workgroups an
  // XCD holds share 4 panels of A and 8 panels of W (of one expert where the routing is even),
  // and every XCD gets its share of them.
  // With room for partial tiles the K split is planned here too (plan_live_split).
  TileParams live = p;
  if (GROUPED) live = live_tiles(p);
  if ((GROUPED && live.tiles_m <= 0) || !tile_of_workgroup(live, tile, split, whole_k)) return;
  tile_coords(live, tile, tile_m, tile_n);
  const int first_split = whole_tiles(live), k_steps = p.size_k / kTileK;
  const int k_first = whole_k ? 0 : split * live.k_steps_per_split;
  wide_tile<T, HAS_ZP, GROUPED, RB, FP4, W8, G32, NV>(
      p, p.tile_table, p.partial, tile_m, tile_n, k_first, whole_k ? k_steps : min(k_steps, k_first + live.k_steps_per_split),
      whole_k ? -1 : split * (live.tiles_m * live.tiles_n - first_split) + tile - first_split);
}

// Both tile sizes in one launch, the 256-row tiles first: the 128-row tiles start on the compute units that the last round
// of 256-row tiles leaves idle, and there is one launch to wait for instead of two.  Us, before -> now: dense, M = 4096,
// K = 4096, N = 6144, fp16, as two launches 167 -> 161; M = 4096, K = 2880, N = 5760 (368 tiles of 256 rows), int4 with groups of
// 32 142 -> 120, MXFP4 131 -> 108; M = 4352, K = 8192, N = 4096 298 -> 229.  Mixture-of-experts layers, where two launches
// and their sums of partial tiles followed each other: 8 experts 1408 x 3712, 2000 tokens 284 -> 195; 8 experts 3072 x 6784,
// AWQ, 939 tokens 402 -> 298; 32 MXFP4 experts 2880 x 2880, 2000 tokens 543 -> 504; Mixtral-8x7B shapes, 2000 and 4096
// tokens: level.
template <typename T, bool HAS_ZP, bool GROUPED = false, bool FP4 = false, int W8 = 0, bool G32 = FP4>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void marlin_tile_wide_pair_kernel(
    const TileParams p) {
  PairTile t;
  if (!pair_tile_of_block(p, GROUPED ? p.tile_table[0] : 0, GROUPED ? p.table_small[0] : 0, blockIdx.x, t)) return;
  if (t.rows == kTileM)
    wide_tile<T, HAS_ZP, GROUPED, 16, FP4, W8, G32, false>(p, p.tile_table, p.partial, t.tile_m, t.tile_n, t.k_first, t.k_tiles,
                                                           t.partial_at);
  else
    wide_tile<T, HAS_ZP, GROUPED, 8, FP4, W8, G32, false>(p, p.table_small, p.partial_small, t.tile_m, t.tile_n, t.k_first,
                                                          t.k_tiles, t.partial_at);
}

// 128-row tiles alone, two workgroups a compute unit: while one starts or ends, the other multiplies.  A 256-row tile takes 11 to 13 us
// around its loop (first bytes, results turned and stored, the gated activation), as long as 8 to 10 steps of K, with nothing
// beside it; and the last round is finer.  Each wavefront has 256 registers, the 128 accumulators in AGPRs and at most 128 more: four
// operands of A instead of eight, one set of column constants (a column block's are replaced behind its last use), 32-bit
// offsets of A, a scale row read from one address (several groups only), and no partial tiles: K is never cut here.  The price is
// that every weight is dequantised once for 128 rows: per matrix instruction 1.7 other vector instructions in float16, 1.2 for
// MXFP4, 2.3 for integers in bfloat16.  Us, before -> now (bits equal): twin_pays and moe_twin_tiles have the figures.
template <typename T, bool HAS_ZP, bool GROUPED, bool FP4, bool G32>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void marlin_tile_twin_kernel(const TileParams p) {
  int tile, tile_m, tile_n, split;
  bool whole_k;
  TileParams live = p;
  if (GROUPED) live.tiles_m = p.tile_table[0], live.tile_band = 8;
  if ((GROUPED && live.tiles_m <= 0) || !tile_of_workgroup(live, tile, split, whole_k)) return;
  tile_coords(live, tile, tile_m, tile_n);
  wide_tile<T, HAS_ZP, GROUPED, 8, FP4, 0, G32, false, true>(p, p.tile_table, nullptr, tile_m, tile_n, 0, p.size_k / kTileK, -1);
}

// Sums the partial tiles of the split tiles of a launch in split order, adds the
// bias and writes C.  One wavefront per accumulator tile (16 rows x 16 columns).
template <typename T>
__global__ __launch_bounds__(256) void tile_reduce_kernel(const TileParams p) {
  const int lane = threadIdx.x & 63;
  const int col16 = lane & 15, kb = lane >> 4;
  const long unit = (long)blockIdx.x * 4 + (threadIdx.x >> 6);   // (tile, 1-KiB block of the partial tile)
  const int first_split = whole_tiles(p);
  const int tiles = p.tiles_m * p.tiles_n - first_split;  // split tiles
  const int blocks = p.tile_rows;                          // blocks per partial tile: 256 or 128
  if (unit >= (long)tiles * blocks) return;
  const int tile = (int)(unit / blocks);
  const int within = (int)(unit - (long)tile * blocks);
  // block = 128 (half of the rows) + 32 strip + 8 column block + row block
  const int half = within >> 7, wave = (within >> 5) & 3;
  const int nb = (within >> 3) & 3, mb = within & 7;
  int tile_m, tile_n;
  tile_coords(p, first_split + tile, tile_m, tile_n);
  const int strip = tile_n * (kTileN / kStripN) + wave;
  const int m = tile_m * p.tile_rows + 128 * half + 16 * mb + col16;
  if (strip * kStripN >= p.size_n) return;
  floatx4_t acc = floatx4_t{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < p.k_splits; ++s) {
    const float4 v = p.partial[((size_t)(s * tiles + tile) * blocks + within) * 64 + lane];
    acc += floatx4_t{v.x, v.y, v.z, v.w};
  }
  if (m >= p.size_m) return;
  if (p.global_scale) acc = acc * p.global_scale[0];
  const int nl = 16 * nb + 4 * kb;
  float bias[4] = {0.f, 0.f, 0.f, 0.f};
  if (p.bias) {
#pragma unroll
    for (int r = 0; r < 4; ++r) bias[r] = Dq<T>::to_float(p.bias[strip * kStripN + scale_slot(nl + r, false)]);
  }
  uint2 o;
  o.x = (uint32_t)Dq<T>::from_float(acc.x + bias[0]) | ((uint32_t)Dq<T>::from_float(acc.y + bias[1]) << 16);
  o.y = (uint32_t)Dq<T>::from_float(acc.z + bias[2]) | ((uint32_t)Dq<T>::from_float(acc.w + bias[3]) << 16);
  *reinterpret_cast<uint2*>(p.c + (long)m * p.size_n + strip * kStripN + nl) = o;
}

// The same for a grouped call whose kernel has split some of its tiles along K (plan_live_split):
// rows are slots of sorted_ids, bias and global scale the expert's, the routing weight applied as
// in the kernel's own epilogue.  Launched for the most tiles there can be; the rest leaves at once.
template <typename T>
__global__ __launch_bounds__(256) void moe_tile_reduce_kernel(const TileParams p) {
  const int lane = threadIdx.x & 63;
  const int col16 = lane & 15, kb = lane >> 4;
  TileParams live;
  if (p.table_small != nullptr) {   // of both tile sizes: the grid's second row adds those of the 128-row tiles
    live = pair_params(p, blockIdx.y == 1, blockIdx.y == 1 ? p.table_small[0] : p.tile_table[0]);
  } else {
    live = live_tiles(p);
  }
  if (live.tiles_m <= 0 || live.k_splits < 2) return;
  const int first_split = live.whole_tiles;
  const int tiles = live.tiles_m * live.tiles_n - first_split;
  const int blocks = live.tile_rows;   // 1-KiB blocks per partial tile: 256 or 128
  // units: (split tile, 1-KiB block of the partial tile)
  for (int unit = blockIdx.x * 4 + (threadIdx.x >> 6); unit < tiles * blocks; unit += gridDim.x * 4) {
    const int tile = unit / blocks;
    const int within = unit - tile * blocks;
    const int half = within >> 7, wave = (within >> 5) & 3;
    const int nb = (within >> 3) & 3, mb = within & 7;
    int tile_m, tile_n;
    tile_coords(live, first_split + tile, tile_m, tile_n);
    // The gated activation, where the tiles that are not cut form it too (store_gated): strips 0 and 1 of a tile are gate, 2 and 3 up,
    // whose sums are made by the lane that has the gate's.  Us a layer, against a launch of its own for calls that may cut tiles: 8 experts
    // 2816 x 1280, 1254 tokens 113.6 -> 109.8; 16 of 2048 x 1408, 2000 tokens 126.7 -> 120.7; 16 of 2048 x 768, 1000 tokens, top 4
    // 95.7 -> 90.8; 18 random-size layers 1.026 times as fast, one (16 of 4096 x 1024, 2000 tokens: one round of tiles, none cut, whose
    // ends take as long as the launch did) 183.3 -> 184.2.
    const bool halves = p.gated != nullptr && p.gated_halves;
    if (halves && wave >= 2) continue;
    const int strip = halves ? 2 * tile_n + wave : tile_n * (kTileN / kStripN) + wave;
    if (strip * kStripN >= p.size_n) continue;
    const int first_slot = live.tile_table[1 + 3 * tile_m] * 64;
    const int tile_rows = live.tile_table[2 + 3 * tile_m] * 64;
    const long expert = live.tile_table[3 + 3 * tile_m];
    const int r = 128 * half + 16 * mb + col16;
    const int id = r < tile_rows ? p.sorted_ids[first_slot + r] : p.rows_total;
    if ((unsigned)id >= (unsigned)p.rows_total) continue;   // padding slot
    const int nl = 16 * nb + 4 * kb;
    uint16_t o[4];
    // the four values of this lane in block `at` of the partial tiles, which is of strip `of`
    auto values = [&](int at, int of, uint16_t (&out)[4]) {
      floatx4_t acc = floatx4_t{0.f, 0.f, 0.f, 0.f};
      for (int s = 0; s < live.k_splits; ++s) {
        const float4 v = live.partial[((size_t)(s * tiles + tile) * blocks + at) * 64 + lane];
        acc += floatx4_t{v.x, v.y, v.z, v.w};
      }
      if (p.global_scale) acc = acc * p.global_scale[expert];
      float bias[4] = {0.f, 0.f, 0.f, 0.f};
      if (p.bias) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          bias[i] = Dq<T>::to_float(p.bias[expert * p.expert_bias_stride + of * kStripN + scale_slot(nl + i, false)]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) out[i] = Dq<T>::from_float(acc[i] + bias[i]);
      if (p.mul_topk) {
        // rounded to the activation type, the product formed and rounded in that type (as in the kernel)
        const float row_w = Dq<T>::to_float(Dq<T>::from_float(p.topk_weights[id]));
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i] = Dq<T>::from_float(Dq<T>::to_float(out[i]) * row_w);
      }
    };
    values(within, strip, o);
    if (halves) {
      uint16_t up[4];
      values(within + 2 * 32, strip + p.size_n / (2 * kStripN), up);
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = silu_times<T>(o[i], up[i]);
    } else if (p.gated != nullptr) {
      const uint32_t pair = (uint32_t)swiglu_oai<T>(o[0], o[1], p.gated_limit, p.gated_alpha) |
                            ((uint32_t)swiglu_oai<T>(o[2], o[3], p.gated_limit, p.gated_alpha) << 16);
      *reinterpret_cast<uint32_t*>(p.gated + (long)id * (p.size_n / 2) + strip * (kStripN / 2) + nl / 2) = pair;
      continue;
    }
    uint2 packed;
    packed.x = (uint32_t)o[0] | ((uint32_t)o[1] << 16);
    packed.y = (uint32_t)o[2] | ((uint32_t)o[3] << 16);
    uint16_t* row = halves ? p.gated + (long)id * (p.size_n / 2) : p.c + (long)id * p.size_n;
    *reinterpret_cast<uint2*>(row + strip * kStripN + nl) = packed;
  }
}

// Builds the row-tile table of a grouped call: runs of blocks with the same
// expert are cut into tiles of up to four blocks.  With `table_small` the one or
// two blocks a run ends in go there instead, to be computed as a 128-row tile at
// half the cost, and of the longer tiles as many are halved as makes the launch shortest
// (pair_cost).  One workgroup, a thread per block of slots: where a block's run begins comes from a
// ballot inside the wavefront and the other wavefronts' last run starts, a tile's number from counts of
// the tile heads before it.  Latency bound (one thread scanning the blocks: 16 us at 157 blocks; 4 us so).
// (1024 threads for up to 256 blocks: 3 us longer, and the code of a kernel that runs once is fetched from memory.)
// The second workgroup does the same for the layer's other GEMM (a launch of 5 to 9 us less;
// us a layer: 64 MXFP4 experts 2048 x 768, 4000 tokens, top 8 405 -> 397; 8 experts 2816 x 1280, 1254 tokens 122 -> 118; 8 of
// 1024 x 2688, AWQ, 6002 tokens 274 -> 269).
struct TableJob {
  int32_t *table, *table_small;
  int tiles_n, k_steps, may_split;   // may_split: 0, 1 (two sizes: K may be cut), or
};
constexpr int kTwinTiles = 2;        // 128-row tiles alone, in `table`

template <int kTableWaves>
__global__ __launch_bounds__(64 * kTableWaves) void moe_tile_table_kernel(const int32_t* __restrict__ expert_ids,
                                                                      const int32_t* __restrict__ num_post_pad,
                                                                      int num_blocks_max, int block_size,
                                                                      int num_experts, int max_tiles, const TableJob first,
                                                                      const TableJob second) {
  int32_t* __restrict__ table = blockIdx.x == 0 ? first.table : second.table;
  int32_t* __restrict__ table_small = blockIdx.x == 0 ? first.table_small : second.table_small;
  const int tiles_n = blockIdx.x == 0 ? first.tiles_n : second.tiles_n;
  const int k_steps = blockIdx.x == 0 ? first.k_steps : second.k_steps;
  const int may_split = blockIdx.x == 0 ? first.may_split : second.may_split;
  constexpr int kTableThreads = 64 * kTableWaves;
  const int most = may_split == kTwinTiles ? 2 : 4;   // blocks of a tile
  __shared__ int32_t last_start[kTableWaves], heads[2][kTableWaves];
  __shared__ unsigned long long best;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int blocks = min(num_post_pad[0] / block_size, num_blocks_max);
  if (threadIdx.x == 0) best = ~0ull;
  int run_carry = 0;          // where the run that reaches into this round of blocks begins
  int count[2] = {0, 0};      // tiles so far: up to four blocks, and the small ones
  struct Tile {
    int first, blocks, expert, number, small;
    bool head;
  };
  // the tile that begins at this thread's block of the round from `base` on
  auto scan = [&](int base) -> Tile {
    const int b = base + threadIdx.x;
    const int e = b < blocks ? expert_ids[b] : -1;
    const bool start = b < blocks && (b == 0 || expert_ids[b - 1] != e);
    const unsigned long long starts = __ballot(start);
    if (lane == 0) last_start[wave] = starts ? base + 64 * wave + 63 - __clzll(starts) : -1;
    __syncthreads();
    int run = run_carry;
    for (int w = 0; w < kTableWaves; ++w) {
      const int t = last_start[w];
      if (t >= 0 && w < wave) run = t;
      if (t >= 0) run_carry = t;
    }
    const unsigned long long upto = starts & (~0ull >> (63 - lane));
    if (upto) run = base + 64 * wave + 63 - __clzll(upto);
    const bool head = b < blocks && e >= 0 && e < num_experts && ((b - run) & (most - 1)) == 0;
    int n = 1;
    if (head)
      while (n < most && b + n < blocks && expert_ids[b + n] == e) ++n;
    const int small = table_small != nullptr && n <= 2;
    const unsigned long long mask[2] = {__ballot(head && !small), __ballot(head && small)};
    if (lane < 2) heads[lane][wave] = __popcll(mask[lane]);
    __syncthreads();
    int at[2] = {count[0], count[1]};
    for (int w = 0; w < kTableWaves; ++w)
      for (int i = 0; i < 2; ++i) {
        const int t = heads[i][w];
        if (w < wave) at[i] += t;
        count[i] += t;
      }
    __syncthreads();
    return Tile{b, n, e, at[small] + (int)__popcll(mask[small] & ((1ull << lane) - 1ull)), small, head};
  };
  auto put = [&](int32_t* to, int i, int first, int num, int expert) {
    if (i >= max_tiles) return;
    int32_t* t = to + 1 + 3 * i;
    t[0] = first;
    t[1] = num;
    t[2] = expert;
  };
  if (table_small == nullptr) {
    for (int base = 0; base < blocks; base += kTableThreads) {
      const Tile t = scan(base);
      if (t.head) put(table, t.number, t.first, t.blocks, t.expert);
    }
    if (threadIdx.x == 0) table[0] = min(count[0], max_tiles);
    return;
  }
  // two sizes: the tiles are counted first and written when it is known which are halved
  Tile t = {};
  for (int base = 0; base < blocks; base += kTableThreads) t = scan(base);
  __syncthreads();   // `best` is set (scan() has barriers of its own, but there may be no block)
  const int big = count[0], small = count[1], plans = pair_plans(big, may_split);
  for (int i = threadIdx.x; i < plans; i += kTableThreads) {
    const PairPlan plan = pair_plan(i, big, may_split);
    if (!pair_has_room(big, small, plan, tiles_n, k_steps)) continue;
    // (a positive float's bits order as it does)
    const float cost = pair_cost(big, small, plan, tiles_n, k_steps);
    atomicMin(&best, ((unsigned long long)__float_as_uint(cost) << 32) | (unsigned)i);
  }
  __syncthreads();
  const PairPlan plan = pair_plan((int)(unsigned)best, big, may_split);
  const int whole = big - plan.halved;
  run_carry = count[0] = count[1] = 0;
  for (int base = 0; base < blocks; base += kTableThreads) {
    if (blocks > kTableThreads) t = scan(base);
    if (!t.head) continue;
    if (t.small) {
      put(table_small, 2 * plan.halved + t.number, t.first, t.blocks, t.expert);
    } else if (t.number < whole) {
      put(table, t.number, t.first, t.blocks, t.expert);
    } else {
      put(table_small, 2 * (t.number - whole), t.first, 2, t.expert);
      put(table_small, 2 * (t.number - whole) + 1, t.first + 2, t.blocks - 2, t.expert);
    }
  }
  if (threadIdx.x == 0) {
    table[0] = pair_word(min(whole, max_tiles), plan.splits[0]);
    table_small[0] = pair_word(min(small + 2 * plan.halved, max_tiles), plan.splits[1]);
  }
}

template <typename T, bool HAS_ZP, bool GROUPED, bool FP4 = false, bool W8 = false>
int launch_tile_async(const TileParams& p, hipStream_t st) {
  constexpr int kLds = W8 ? async_lds8() : async_lds(FP4);
  static bool attr_set = false;  // raising the dynamic LDS limit is needed once per kernel
  if (!attr_set) {
    SONAR_HIP(hipFuncSetAttribute((const void*)marlin_tile_async_kernel<T, HAS_ZP, GROUPED, FP4, W8>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, kLds));
    attr_set = true;
  }
  marlin_tile_async_kernel<T, HAS_ZP, GROUPED, FP4, W8><<<tile_grid(p), kTileWaves * 64, kLds, st>>>(p);
  return SONAR_OK;
}
// groups of a multiple of 64 rows that is no power of two times 64
template <bool GROUPED>
int launch_tile_async_type(const TileParams& p, int dtype, int bits, hipStream_t st) {
  if (bits == 8)
    return dtype == SONAR_DTYPE_F16 ? launch_tile_async<_Float16, false, GROUPED, false, true>(p, st)
                                    : launch_tile_async<__bf16, false, GROUPED, false, true>(p, st);
  if (dtype == SONAR_DTYPE_F16)
    return p.zeros ? launch_tile_async<_Float16, true, GROUPED>(p, st) : launch_tile_async<_Float16, false, GROUPED>(p, st);
  return p.zeros ? launch_tile_async<__bf16, true, GROUPED>(p, st) : launch_tile_async<__bf16, false, GROUPED>(p, st);
}

// (Grouped calls: marlin_tile_wide_pair_kernel, but for NVFP4 and 8-bit codes with groups of 32 rows.)
template <typename T, bool HAS_ZP, int RB>
int launch_tile_wide_rows(const TileParams& p, hipStream_t st) {
  static bool attr_set = false;
  if (!attr_set) {
    SONAR_HIP(hipFuncSetAttribute((const void*)marlin_tile_wide_kernel<T, HAS_ZP, false, RB>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, wide_lds(RB)));
    attr_set = true;
  }
  marlin_tile_wide_kernel<T, HAS_ZP, false, RB><<<tile_grid(p), 256, wide_lds(RB), st>>>(p);
  return SONAR_OK;
}
// MXFP4: bf16, groups of 32 rows, float4_e2m1f codes
template <int RB>
int launch_tile_wide_fp4_rows(const TileParams& p, hipStream_t st) {
  static bool attr_set = false;
  if (!attr_set) {
    SONAR_HIP(hipFuncSetAttribute((const void*)marlin_tile_wide_kernel<__bf16, false, false, RB, true>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, wide_lds(RB)));
    attr_set = true;
  }
  marlin_tile_wide_kernel<__bf16, false, false, RB, true><<<tile_grid(p), 256, wide_lds(RB), st>>>(p);
  return SONAR_OK;
}
int launch_tile_wide_fp4(const TileParams& p, hipStream_t st) {
  return p.tile_rows == 128 ? launch_tile_wide_fp4_rows<8>(p, st) : launch_tile_wide_fp4_rows<16>(p, st);
}
// NVFP4: either activation type, groups of 16 rows, a global scale (one per expert when GROUPED)
template <typename T, bool GROUPED, int RB>
int launch_tile_wide_nvfp4_rows(const TileParams& p, hipStream_t st) {
  static bool attr_set = false;
  if (!attr_set) {
    SONAR_HIP(hipFuncSetAttribute((const void*)marlin_tile_wide_kernel<T, false, GROUPED, RB, true, 0, true, true>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, wide_lds(RB)));
    attr_set = true;
  }
  marlin_tile_wide_kernel<T, false, GROUPED, RB, true, 0, true, true><<<tile_grid(p), 256, wide_lds(RB), st>>>(p);
  return SONAR_OK;
}
template <typename T, bool GROUPED>
int launch_tile_wide_nvfp4(const TileParams& p, hipStream_t st) {
  if (p.tile_rows != kTileM) return fail(SONAR_E_INVALID, "internal: NVFP4 runs on 256-row tiles");
  return launch_tile_wide_nvfp4_rows<T, GROUPED, 16>(p, st);
}
// 8-bit codes: uint8b128 or float8_e4m3fn (groups of 64 * 2^i rows or one group; G32: of 32 rows, MXFP8)
inline bool wide_groups_of_32(const TileParams& p) { return p.num_groups > 1 && p.group_size == 32; }
template <typename T, bool GROUPED, int W8, bool G32, int RB = 16>
int launch_tile_wide8_groups(const TileParams& p, hipStream_t st) {
  static bool attr_set = false;
  if (!attr_set) {
    SONAR_HIP(hipFuncSetAttribute((const void*)marlin_tile_wide_kernel<T, false, GROUPED, RB, false, W8, G32>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, wide_lds(RB)));
    attr_set = true;
  }
  marlin_tile_wide_kernel<T, false, GROUPED, RB, false, W8, G32><<<tile_grid(p), 256, wide_lds(RB), st>>>(p);
  return SONAR_OK;
}
template <typename T, bool GROUPED>
int launch_tile_wide8(const TileParams& p, bool fp8, hipStream_t st) {
  const bool g32 = wide_groups_of_32(p);
  // 128-row tiles (dense calls with few tiles)
  if (p.tile_rows == 128 && g32) return fail(SONAR_E_INVALID, "internal: 8-bit codes with groups of 32 rows run on 256-row tiles");
  if (g32) return fp8 ? launch_tile_wide8_groups<T, GROUPED, 2, true>(p, st) : launch_tile_wide8_groups<T, GROUPED, 1, true>(p, st);
  if constexpr (!GROUPED) {
    if (p.tile_rows == 128)
      return fp8 ? launch_tile_wide8_groups<T, false, 2, false, 8>(p, st)
                 : launch_tile_wide8_groups<T, false, 1, false, 8>(p, st);
    return fp8 ? launch_tile_wide8_groups<T, false, 2, false>(p, st) : launch_tile_wide8_groups<T, false, 1, false>(p, st);
  }
  return fail(SONAR_E_INVALID, "internal: a grouped call of one tile size");
}
// 4-bit integer codes with groups of 32 rows
template <typename T, bool HAS_ZP, int RB>
int launch_tile_wide_g32_rows(const TileParams& p, hipStream_t st) {
  static bool attr_set = false;
  if (!attr_set) {
    SONAR_HIP(hipFuncSetAttribute((const void*)marlin_tile_wide_kernel<T, HAS_ZP, false, RB, false, 0, true>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, wide_lds(RB)));
    attr_set = true;
  }
  marlin_tile_wide_kernel<T, HAS_ZP, false, RB, false, 0, true><<<tile_grid(p), 256, wide_lds(RB), st>>>(p);
  return SONAR_OK;
}
template <typename T, bool HAS_ZP>
int launch_tile_wide(const TileParams& p, hipStream_t st) {
  if (wide_groups_of_32(p))
    return p.tile_rows == 128 ? launch_tile_wide_g32_rows<T, HAS_ZP, 8>(p, st) : launch_tile_wide_g32_rows<T, HAS_ZP, 16>(p, st);
  return p.tile_rows == 128 ? launch_tile_wide_rows<T, HAS_ZP, 8>(p, st) : launch_tile_wide_rows<T, HAS_ZP, 16>(p, st);
}

// Both tile sizes; `max_row_tiles`: grouped calls, the most row tiles there can be.
template <typename T, bool HAS_ZP, bool GROUPED, bool FP4, int W8, bool G32>
int launch_pair_form(const TileParams& p, int max_row_tiles, hipStream_t st) {
  static bool attr_set = false;
  if (!attr_set) {
    SONAR_HIP(hipFuncSetAttribute((const void*)marlin_tile_wide_pair_kernel<T, HAS_ZP, GROUPED, FP4, W8, G32>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, wide_lds(16)));
    attr_set = true;
  }
  marlin_tile_wide_pair_kernel<T, HAS_ZP, GROUPED, FP4, W8, G32><<<pair_grid(p, max_row_tiles), 256, wide_lds(16), st>>>(p);
  return SONAR_OK;
}
template <typename T, bool HAS_ZP, bool GROUPED, bool FP4, bool G32>
int launch_twin_form(const TileParams& p, hipStream_t st) {
  static bool attr_set = false;
  if (!attr_set) {
    SONAR_HIP(hipFuncSetAttribute((const void*)marlin_tile_twin_kernel<T, HAS_ZP, GROUPED, FP4, G32>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, wide_lds(8)));
    attr_set = true;
  }
  marlin_tile_twin_kernel<T, HAS_ZP, GROUPED, FP4, G32><<<tile_grid(p), 256, wide_lds(8), st>>>(p);
  return SONAR_OK;
}
template <typename T, bool GROUPED>
int launch_twin_type(const TileParams& p, bool fp4, hipStream_t st) {
  if constexpr (std::is_same<T, __bf16>::value)
    if (fp4) return launch_twin_form<T, false, GROUPED, true, true>(p, st);
  if (fp4) return fail(SONAR_E_INVALID, "internal: MXFP4 weights with float16 activations");
  if (wide_groups_of_32(p))
    return p.zeros ? launch_twin_form<T, true, GROUPED, false, true>(p, st) : launch_twin_form<T, false, GROUPED, false, true>(p, st);
  return p.zeros ? launch_twin_form<T, true, GROUPED, false, false>(p, st) : launch_twin_form<T, false, GROUPED, false, false>(p, st);
}
template <bool GROUPED>
int launch_twin(const TileParams& p, int dtype, bool fp4, hipStream_t st) {
  const int rc = dtype == SONAR_DTYPE_F16 ? launch_twin_type<_Float16, GROUPED>(p, fp4, st) : launch_twin_type<__bf16, GROUPED>(p, fp4, st);
  return rc ? rc : launch_status("marlin_tile_twin_kernel");
}

template <typename T, bool GROUPED>
int launch_pair_type(const TileParams& p, int max_row_tiles, bool fp4, int bits, bool fp8, hipStream_t st) {
  if constexpr (std::is_same<T, __bf16>::value)
    if (fp4) return launch_pair_form<T, false, GROUPED, true, 0, true>(p, max_row_tiles, st);
  if (fp4) return fail(SONAR_E_INVALID, "internal: MXFP4 weights with float16 activations");
  if (bits == 8)
    return fp8 ? launch_pair_form<T, false, GROUPED, false, 2, false>(p, max_row_tiles, st)
               : launch_pair_form<T, false, GROUPED, false, 1, false>(p, max_row_tiles, st);
  if (wide_groups_of_32(p))
    return p.zeros ? launch_pair_form<T, true, GROUPED, false, 0, true>(p, max_row_tiles, st)
                   : launch_pair_form<T, false, GROUPED, false, 0, true>(p, max_row_tiles, st);
  return p.zeros ? launch_pair_form<T, true, GROUPED, false, 0, false>(p, max_row_tiles, st)
                 : launch_pair_form<T, false, GROUPED, false, 0, false>(p, max_row_tiles, st);
}
template <bool GROUPED>
int launch_pair(const TileParams& p, int max_row_tiles, int dtype, bool fp4, int bits, bool fp8, hipStream_t st) {
  const int rc = dtype == SONAR_DTYPE_F16 ? launch_pair_type<_Float16, GROUPED>(p, max_row_tiles, fp4, bits, fp8, st)
                                          : launch_pair_type<__bf16, GROUPED>(p, max_row_tiles, fp4, bits, fp8, st);
  return rc ? rc : launch_status("marlin_tile_wide_pair_kernel");
}

template <typename T, bool HAS_ZP, bool HAS_PERM>
int launch_tile(const TileParams& p, hipStream_t st) {
  static bool attr_set = false;  // raising the dynamic LDS limit is needed once per kernel
  if (!attr_set) {
    SONAR_HIP(hipFuncSetAttribute((const void*)marlin_tile_kernel<T, HAS_ZP, HAS_PERM>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, kTileLds));
    attr_set = true;
  }
  const int grid = tile_grid(p);
  marlin_tile_kernel<T, HAS_ZP, HAS_PERM><<<grid, kTileWaves * 64, kTileLds, st>>>(p);
  return SONAR_OK;
}

}  // namespace

namespace {
// (grouped calls: 64-bit addresses)
bool wide_takes_rows(const TileParams& p) { return p.tile_table != nullptr || wide_rows_within_32_bits(p.lda); }
// The wide form: groups of 32 or 64 * 2^i rows or one group, K of any number of steps.  (Passes of the loop were whole
// before: up to three steps of zeros where that was at most a tenth of K, and eight wavefronts elsewhere.  Us, before ->
// now: int4 with groups of 32, M = 4096, K = 2880, N = 5760 204 -> 142; AWQ, M = 4000, K = 1152, N = 6144 117 -> 71; NVFP4
// bf16, M = 2048, K = 4480, N = 8192 148 -> 118; MXFP8, M = 3000, K = 2944, N = 6144 188 -> 168; int4, M = 2000, K = 2944,
// N = 7808, once padded, 81.5 -> 78.3; 2000 tokens on 32 MXFP4 experts of 2880 x 2880, the whole layer 626 -> 543.)
bool wide_applies(const TileParams& p) {
  static const bool no_wide = getenv("SONAR_MARLIN_NO_WIDE_TILE") != nullptr;   // debugging aid
  if (!wide_takes_rows(p)) return false;
  if (wide_groups_of_32(p)) return true;
  if (no_wide) return false;
  if (p.num_groups == 1) return true;
  const int per_group = p.group_size / kTileK;   // steps per group: a power of two
  return p.group_size % kTileK == 0 && (per_group & (per_group - 1)) == 0;
}
// ... and for MXFP4 and NVFP4 (groups of 32 and 16 rows, the caller has checked).  Dense MXFP4 calls whose 256-row tiles
// leave a quarter of the compute units without one stay with eight wavefronts, at the higher clock of such a launch
// the faster ones on these codes (M = 3000, K = 6656, N = 3072, 144 tiles: 127 us against 131; M = 2048, K = 4224, N = 5120,
// 160 tiles: 85.6 against 88.4; but M = 2048, K = 6400, N = 7680, 240 tiles: 148 against 145, M = 4096, K = 4224, N = 8192,
// 512 tiles: 215 against 201).
bool wide_applies_fp4(const TileParams& p) {
  static const bool no_wide = getenv("SONAR_MARLIN_NO_WIDE_TILE") != nullptr;
  if (p.tile_table != nullptr || p.global_scale != nullptr) return true;
  const bool few = p.tile_rows == kTileM && p.k_splits == 1 && p.tiles_m * p.tiles_n <= 192;
  return !no_wide && !few && wide_takes_rows(p);
}
// ... and for 8-bit codes (the same rule; floating-point ones come in groups of 32 or 128 rows or one).
bool wide_applies8(const TileParams& p, bool fp8) { return fp8 || wide_applies(p); }
}  // namespace

// The 128-row tiles of marlin_tile_twin_kernel: 4-bit integers and MXFP4 with several groups.
bool tile_twin_applies(int bits, bool nvfp4, int64_t num_groups, int group_size, int64_t a_row_stride) {
  // debugging aids: the switch of these tiles, and those that single out an older path
  static const bool off = [] {
    for (const char* name : {"SONAR_MARLIN_NO_TWIN_TILES", "SONAR_MARLIN_NO_WIDE_TILE", "SONAR_MARLIN_NO_128_ROW_TILES",
                             "SONAR_MARLIN_NO_TWO_TILE_SIZES", "SONAR_MARLIN_MAX_K_SPLITS", "SONAR_MARLIN_NO_ASYNC_TILE",
                             "SONAR_MARLIN_NO_MOE_K_SPLIT"})
      if (getenv(name) != nullptr) return true;
    return false;
  }();
  if (off || bits != 4 || nvfp4 || num_groups <= 1 || !wide_rows_within_32_bits(a_row_stride)) return false;
  const int per_group = group_size / kTileK;
  return group_size == 32 || (group_size % kTileK == 0 && (per_group & (per_group - 1)) == 0);
}

// The asynchronous tile kernel needs groups of 32 rows or a multiple of 64 and no gather of A.
bool tile_async_applies(bool has_perm, int64_t num_groups, int group_size) {
  return !has_perm && (num_groups == 1 || group_size % kTileK == 0 || group_size == 32);
}

namespace {
// What tile_gemm launches for a call the asynchronous tile kernels take: one tile size (with
// tile_reduce_kernel behind it when K is split), both sizes of the wide kernel, or 128-row tiles two at a time.
struct TileLaunches {
  bool ok, pair, twin;
  TileParams launch;
};

// `p` arrives with the shape, the pointers and one 256-row launch over the whole of K filled in.
TileLaunches plan_tile_launches(TileParams p, int64_t size_m, int64_t size_n, int64_t size_k, int64_t num_groups,
                                int group_size, void* partial, size_t partial_bytes, bool fp4, bool nvfp4, int bits,
                                bool has_perm, bool float16, bool may_twin = true) {
  TileLaunches out;
  out.ok = true;
  out.pair = out.twin = false;
  const int steps_per_group = group_size / kTileK;
  const bool wide128 = bits == 4 && !fp4 && !has_perm &&
                       (num_groups == 1 || (group_size % kTileK == 0 && (steps_per_group & (steps_per_group - 1)) == 0));
  const bool rows_97_128 = plan_rows_97_128(size_m, size_n, size_k, wide128);
  // few tiles and a call the wide kernel takes: 128-row tiles
  static const bool no_128 = getenv("SONAR_MARLIN_NO_128_ROW_TILES") != nullptr;   // debugging aid
  // (not for NVFP4 and 8-bit codes with groups of 32 rows, whose heavier dequantisation wants the 16 row blocks
  // to hide behind: M = 512, K = 4096, N = 11008: NVFP4 69.9 us against 68.7, MXFP8 91.8 against 82.2)
  const bool rows128_ok = !nvfp4 && !(bits == 8 && num_groups > 1 && group_size == 32);
  GemmPlan plan = tile_plan(size_m, size_n, size_k, rows128_ok && !no_128, rows_97_128);
  // two 128-row tiles at a time
  if (may_twin && !has_perm && tile_twin_applies(bits, nvfp4, num_groups, group_size, p.lda) &&
      twin_pays(size_m, size_n, size_k, float16, fp4, rows128_ok, rows_97_128)) {
    p.tile_rows = 128;
    p.tiles_m = (int)((size_m + 127) / 128);
    p.tile_band = 8;   // the same rows of A per band as four 256-row tiles
    out.twin = true;
    out.launch = p;
    return out;
  }
  if (plan.tile_rows == 128) {
    TileParams probe = p;
    probe.tile_rows = 128;
    probe.k_splits = plan.k_splits;
    probe.k_steps_per_split = plan.k_steps_per_split;
    if ((fp4 ? wide_applies_fp4(probe) : wide_applies(probe)) &&
        (plan.k_splits == 1 || (partial != nullptr && partial_bytes >= plan_partial_bytes(plan, size_m, size_n)))) {
      p.tile_rows = 128;
      p.tiles_m = (int)((size_m + 127) / 128);
      p.tile_band = 8;
    } else {
      plan = tile_plan(size_m, size_n, size_k, false, rows_97_128);
    }
  }
  if (plan.k_splits > 1 && partial != nullptr && partial_bytes >= plan_partial_bytes(plan, size_m, size_n)) {
    p.k_splits = plan.k_splits;
    p.k_steps_per_split = plan.k_steps_per_split;
    p.whole_tiles = (int)plan.whole_tiles;
    p.partial = static_cast<float4*>(partial);
    static const char* max_splits = getenv("SONAR_MARLIN_MAX_K_SPLITS");  // debugging aid
    if (max_splits && atoi(max_splits) >= 1 && p.k_splits > atoi(max_splits)) {
      const int k_steps = (int)(size_k / kTileK);
      p.k_splits = atoi(max_splits);
      p.k_steps_per_split = (k_steps + p.k_splits - 1) / p.k_splits;
      p.k_splits = (k_steps + p.k_steps_per_split - 1) / p.k_steps_per_split;
      if (p.k_splits == 1) p.partial = nullptr;
    }
  }
  out.launch = p;
  if (p.tile_rows != kTileM && !(fp4 ? wide_applies_fp4(p) : wide_applies(p))) {
    out.ok = false;   // 128-row tiles exist in the wide tile kernel only
    return out;
  }
  auto takes_wide = [&](const TileParams& q) {
    return fp4 ? wide_applies_fp4(q) : wide_applies(q);
  };
  // More tiles than compute units with a last round that fills half of them or less (M = 4096, N = 6144: 384 tiles of 256
  // rows = 256 + 128): the full rounds run as they are and the tiles of the last round as two 128-row tiles each, over
  // the whole of K and in the same launch: nothing goes through scratch.  Tile t of the 256-row numbering is tiles 2 t and
  // 2 t + 1 of the 128-row numbering with bands twice as high.
  static const bool no_two_sizes = getenv("SONAR_MARLIN_NO_TWO_TILE_SIZES") != nullptr;   // debugging aid
  const int tiles = p.tiles_m * p.tiles_n, last_round = tiles % 256;
  // (Where K is long enough to be cut into three ranges or more, a short last round is shorter that way.)
  if (!no_two_sizes && !no_128 && rows128_ok && p.tile_rows == kTileM && p.k_splits < 3 && tiles > 256 && last_round > 0 &&
      last_round <= 128) {
    TileParams both = p;
    both.k_splits = 1;
    both.k_steps_per_split = (int)(size_k / kTileK);
    both.partial = nullptr;
    both.big_tiles = tiles - last_round;
    if (takes_wide(both)) {
      out.pair = true;
      out.launch = both;
    }
  }
  return out;
}

// The shape of a dense call as one 256-row launch over the whole of K (no pointers).
TileParams dense_tile_shape(int64_t size_m, int64_t size_n, int64_t size_k, int64_t num_groups, int group_size) {
  TileParams p = {};
  p.size_m = (int)size_m;
  p.size_n = (int)size_n;
  p.size_k = (int)size_k;
  p.num_groups = (int)num_groups;
  p.group_size = group_size;
  p.chunks_per_strip = (int)(size_k / kChunkK);
  p.tile_rows = kTileM;
  p.tiles_m = (int)((size_m + kTileM - 1) / kTileM);
  p.tile_band = 4;
  p.tiles_n = (int)((size_n + kTileN - 1) / kTileN);
  p.k_splits = 1;
  p.whole_tiles = 0;  // read only with k_splits > 1
  p.k_steps_per_split = (int)(size_k / kTileK);
  return p;
}
}  // namespace

// Called by sonar_marlin_gemm for size_m > 64.  Shapes and pointers have been
// validated by the caller; size_k % 64 == 0 is required here.
int tile_gemm(const void* a, int64_t a_row_stride, void* c, const uint32_t* b, const void* bias,
              const void* scales, const float* global_scale, const uint32_t* zeros, const int32_t* perm, int dtype,
              int64_t size_m, int64_t size_n, int64_t size_k, int64_t num_groups, int group_size, void* partial,
              size_t partial_bytes, bool fp4, int bits, bool fp8, hipStream_t st) {
  TileParams p = dense_tile_shape(size_m, size_n, size_k, num_groups, group_size);
  p.global_scale = global_scale;
  p.a = static_cast<const uint16_t*>(a);
  p.lda = a_row_stride;
  p.c = static_cast<uint16_t*>(c);
  p.b = reinterpret_cast<const uint4*>(b);
  p.bias = static_cast<const uint16_t*>(bias);
  p.scales = static_cast<const uint16_t*>(scales);
  p.zeros = zeros;
  p.perm = perm;
  const bool zp = zeros != nullptr, pm = perm != nullptr;
  int rc;
  static const bool no_async = getenv("SONAR_MARLIN_NO_ASYNC_TILE") != nullptr;  // debugging aid
  const bool nvfp4 = fp4 && global_scale != nullptr;   // the caller has checked: groups of 16 rows
  if ((nvfp4 || tile_async_applies(pm, num_groups, group_size)) &&
      (!no_async || fp4 || bits == 8)) {   // float4 and 8-bit codes exist here only
    const TileLaunches plan = plan_tile_launches(p, size_m, size_n, size_k, num_groups, group_size, partial,
                                                 partial_bytes, fp4, nvfp4, bits, pm, dtype == SONAR_DTYPE_F16);
    if (!plan.ok)
      return fail(SONAR_E_INVALID, "internal: 128-row tiles exist in the wide tile kernel only");
    // the kernel a launch described by q takes
    auto launch = [&](const TileParams& q) -> int {
      if (nvfp4)
        return dtype == SONAR_DTYPE_F16 ? launch_tile_wide_nvfp4<_Float16, false>(q, st)
                                        : launch_tile_wide_nvfp4<__bf16, false>(q, st);
      if (fp4)   // the caller has checked: bf16, groups of 32 rows, no zero points
        return wide_applies_fp4(q) ? launch_tile_wide_fp4(q, st) : launch_tile_async<__bf16, false, false, true>(q, st);
      if (bits == 8 && wide_applies8(q, fp8))   // symmetric 8-bit codes: the caller has checked
        return dtype == SONAR_DTYPE_F16 ? launch_tile_wide8<_Float16, false>(q, fp8, st)
                                        : launch_tile_wide8<__bf16, false>(q, fp8, st);
      if (bits == 8 || !wide_applies(q)) return launch_tile_async_type<false>(q, dtype, bits, st);
      if (dtype == SONAR_DTYPE_F16) return zp ? launch_tile_wide<_Float16, true>(q, st) : launch_tile_wide<_Float16, false>(q, st);
      return zp ? launch_tile_wide<__bf16, true>(q, st) : launch_tile_wide<__bf16, false>(q, st);
    };
    p = plan.launch;
    if (plan.twin) return launch_twin<false>(p, dtype, fp4, st);
    if (plan.pair) return launch_pair<false>(p, 0, dtype, fp4, bits, fp8, st);
    rc = launch(p);
    if (rc) return rc;
    if (int rc2 = launch_status("marlin_tile_async_kernel")) return rc2;
    if (p.k_splits > 1) {
      const int blocks = (p.tiles_m * p.tiles_n - p.whole_tiles) * (p.tile_rows / 4);
      if (dtype == SONAR_DTYPE_F16) tile_reduce_kernel<_Float16><<<blocks, 256, 0, st>>>(p);
      else tile_reduce_kernel<__bf16><<<blocks, 256, 0, st>>>(p);
      return launch_status("tile_reduce_kernel");
    }
    return SONAR_OK;
  }
  if (bits == 8) return fail(SONAR_E_INVALID, "internal: 8-bit codes exist in the asynchronous tile kernel only");
  if (zp && pm) return fail(SONAR_E_INVALID, "internal: act-order with zero points");   // refused by the entry point
  if (dtype == SONAR_DTYPE_F16) {
    rc = zp ? launch_tile<_Float16, true, false>(p, st)
            : (pm ? launch_tile<_Float16, false, true>(p, st) : launch_tile<_Float16, false, false>(p, st));
  } else {
    rc = zp ? launch_tile<__bf16, true, false>(p, st)
            : (pm ? launch_tile<__bf16, false, true>(p, st) : launch_tile<__bf16, false, false>(p, st));
  }
  if (rc) return rc;
  return launch_status("marlin_tile_kernel");
}

// Row tiles a grouped call can have at most, and the bytes of its tile table.  A tile is a
// run of up to four blocks of one expert; expert_ids need not be grouped by expert (blocks of
// absent experts, -1, may sit between runs), so the bound is one tile per block: the table
// can never be short of an entry, whatever the routing.
int moe_tile_max(int64_t sorted_len, int64_t num_experts) {
  (void)num_experts;
  return (int)((sorted_len + 63) / 64);
}
// (two tables: the tiles of up to four blocks, and the one- or two-block ends of the experts' rows
// that the wide kernel computes as 128-row tiles)
static size_t moe_one_table_bytes(int64_t sorted_len) {
  return ((size_t)(1 + 3 * moe_tile_max(sorted_len, 0)) * sizeof(int32_t) + 255) & ~(size_t)255;
}
size_t moe_tile_table_bytes(int64_t sorted_len, int64_t num_experts) {
  (void)num_experts;
  return 2 * moe_one_table_bytes(sorted_len);
}
// Room for the fp32 partial tiles of a grouped call that splits some of its tiles along K on the
// device (plan_live_split): 64 MiB for the 256-row tiles and 32 MiB for the 128-row tiles where K
// allows a split, else none.
static size_t moe_partial_bytes_of(int tile_rows) { return (size_t)kLiveSplitWorkMax * tile_rows * 1024; }
size_t moe_tile_partial_bytes(int64_t size_k) {
  const int64_t k_steps = size_k / kTileK;
  if (size_k % (4 * kTileK) != 0 || k_steps < 16) return 0;
  return moe_partial_bytes_of(kTileM) + moe_partial_bytes_of(128);
}

// Two 128-row tiles at a time, which hide each other's start and end, instead: always up to 160 rows an expert, whose tiles have 128
// rows either way; with more, while the second dequantisation of the weights (integers in bf16 twice the instructions of float16 and
// MXFP4) costs less than that; not where K is long and the tiles fill half of the compute units, which K in ranges does.  Us a layer, two
// sizes -> here, over 325 random layers of 8 to 64 experts 0.91 times (0.74 to 1.04): 32 experts of 71 rows 2560 x 1152 225 -> 180; 16
// MXFP4 of 97, 2688 x 10880 404 -> 361; 16 of 632, 1280 x 2688 270 -> 233; 64 MXFP4 of 500, 2048 x 768 398 -> 342; 32 MXFP4 of 250,
// 2880 x 2880 457 -> 429.  Left out: Mixtral-8x7B shapes, bf16, 500 and 1024 rows 1267 -> 1360 and 2417 -> 2529; 16 of 453, bf16, AWQ,
// 3968 x 7040 1112 -> 1157; 8 of 200, fp16, 7168 x 7168 505 -> 518; 8 of 116, 2048 x 5888 137 -> 141.
// (The offsets of A have 32 bits: its rows are slots, at most sorted_len of them, or row ids / top_k, and a list of slots may be shorter
// than the rows that its ids reach.)
static bool moe_twin_tiles(const TileParams& q, int64_t sorted_len, int64_t num_experts, int bits, bool fp4, bool nvfp4, bool float16,
                           bool may_split) {
  const int64_t a_rows = std::max<int64_t>(sorted_len, q.rows_total);
  if (!tile_twin_applies(bits, nvfp4, q.num_groups, q.group_size, q.size_k) || a_rows * q.size_k * 2 >= (1LL << 32)) return false;
  const int64_t tiles = (q.rows_total / 128 + num_experts / 2) * q.tiles_n;
  if (may_split && tiles < 128 && q.size_k >= 2048) return false;
  return q.rows_total <= 160 * num_experts || q.size_k <= (fp4 ? 8192 : float16 ? 6144 : 3072);
}

// Called by sonar_moe_wna16_marlin_gemm for 64-slot blocks without act-order
// when group_size % 64 == 0 (or one group) and size_k % 64 == 0.
int moe_tile_gemm(const void* a, void* c, const uint32_t* b, const void* bias, const void* scales,
                  const float* global_scale, const uint32_t* zeros, const int32_t* sorted_ids, int64_t sorted_len, const int32_t* expert_ids,
                  const int32_t* num_post_pad, const float* topk_weights, int64_t top_k, int mul_topk,
                  int64_t num_experts, int32_t* table, int dtype, int64_t size_m, int64_t size_n, int64_t size_k,
                  int64_t num_groups, int group_size, int a_by_slot, bool fp4, int bits, bool fp8, void* partial,
                  size_t partial_bytes, const MoeLayerCall& layer, hipStream_t st) {
  const int max_tiles = moe_tile_max(sorted_len, num_experts);
  const int blocks_max = (int)((sorted_len + 63) / 64);
  TileParams p = {};
  p.global_scale = global_scale;   // NVFP4: one per expert
  p.a = static_cast<const uint16_t*>(a);
  p.lda = size_k;
  p.c = static_cast<uint16_t*>(c);
  p.b = reinterpret_cast<const uint4*>(b);
  p.bias = static_cast<const uint16_t*>(bias);
  p.scales = static_cast<const uint16_t*>(scales);
  p.zeros = zeros;
  p.perm = nullptr;
  p.size_m = (int)size_m;
  p.size_n = (int)size_n;
  p.size_k = (int)size_k;
  p.num_groups = (int)num_groups;
  p.group_size = group_size;
  p.chunks_per_strip = (int)(size_k / kChunkK);
  p.tile_rows = kTileM;
  p.tiles_m = max_tiles;
  p.tile_band = max_tiles > 0 ? max_tiles : 1;  // whole columns of row tiles (the wide kernel numbers its tiles itself)
  p.k_splits = 1;
  p.whole_tiles = 0;  // read only with k_splits > 1
  p.k_steps_per_split = (int)(size_k / kTileK);
  p.partial = nullptr;
  p.tiles_n = (int)((size_n + kTileN - 1) / kTileN);
  p.sorted_ids = sorted_ids;
  p.topk_weights = topk_weights;
  p.tile_table = table;
  p.rows_total = (int)(size_m * top_k);
  p.top_k = (int)top_k;
  p.mul_topk = mul_topk;
  p.a_by_slot = a_by_slot;
  p.expert_b_stride = (long)(size_k * size_n / (32 / bits) / 4);
  p.expert_s_stride = (long)(num_groups * size_n);
  p.expert_z_stride = (long)(num_groups * (size_n / 8));
  p.expert_bias_stride = (long)size_n;
  // The wide kernel splits the tiles of a short last round (or all of them when they are few) along
  // K, given room for their partial tiles; moe_tile_reduce_kernel sums them.
  static const bool no_live_split = getenv("SONAR_MARLIN_NO_MOE_K_SPLIT") != nullptr;   // debugging aid
  auto is_wide = [&](const TileParams& q) {
    return fp4 ? wide_applies_fp4(q) : (bits == 8 ? wide_applies8(q, fp8) : wide_applies(q));
  };
  const bool wide = is_wide(p);
  const size_t partial_need = moe_tile_partial_bytes(size_k);
  if (wide && !no_live_split && partial != nullptr && partial_need > 0 && partial_bytes >= partial_need &&
      ((uintptr_t)partial) % 16 == 0)
    p.partial = static_cast<float4*>(partial);
  // ... and computes the one or two blocks an expert's rows end in as a 128-row tile, and others where that makes the launch
  // shorter (marlin_tile_wide_pair_kernel; not NVFP4, and not 8-bit codes with groups of 32 rows)
  const bool nvfp4 = fp4 && global_scale != nullptr;
  auto has_two_sizes = [&](const TileParams& q) { return is_wide(q) && !nvfp4 && !(bits == 8 && wide_groups_of_32(q)); };
  const bool two_sizes = has_two_sizes(p);
  int32_t* table_small = two_sizes ? table + moe_one_table_bytes(sorted_len) / sizeof(int32_t) : nullptr;
  // tiles are cut along K only while they are few (and the second kernel is launched only where they may be): not when
  // the rows nearly fill the chip wherever they go, or, with a long K, fill it twice
  auto may_cut = [](const TileParams& q) {
    return (int64_t)(q.rows_total + 255) / 256 * q.tiles_n <= (q.size_k >= 64 * kTileK ? 512 : 192);
  };
  auto is_twin = [&](const TileParams& q, bool may_split) {
    return moe_twin_tiles(q, sorted_len, num_experts, bits, fp4, nvfp4, dtype == SONAR_DTYPE_F16, may_split);
  };
  if (two_sizes && !may_cut(p)) p.partial = nullptr;
  const bool twin = two_sizes && is_twin(p, p.partial != nullptr);
  if (twin) {
    p.partial = nullptr;
    p.tile_rows = 128;
    table_small = nullptr;   // (one table, of tiles of up to two blocks)
  } else if (two_sizes) {
    if (p.partial != nullptr)
      p.partial_small = reinterpret_cast<float4*>(static_cast<char*>(partial) + moe_partial_bytes_of(kTileM));
  }
  // The activation at the end of the tiles, or of the sums of partial tiles
  GatedOutput* gated = layer.gated;
  if (gated != nullptr && wide && ((uintptr_t)gated->out) % 16 == 0 &&
      (gated->kind == 0 ? size_n % (2 * 2 * kStripN) == 0 : gated->kind == SONAR_ACT_SWIGLUOAI && gated->limit > 0.f)) {
    p.gated = static_cast<uint16_t*>(gated->out);
    p.gated_halves = gated->kind == 0;
    p.gated_limit = gated->limit;
    p.gated_alpha = gated->alpha;
    gated->done = true;
  }
  TableJob job = {table, table_small, p.tiles_n, (int)(size_k / kTileK), twin ? kTwinTiles : p.partial != nullptr}, next_job = {};
  sonar_moe_tables* ready = layer.ready;
  if (two_sizes && ready != nullptr && ready->built && ready->expert_ids == expert_ids && ready->sorted_len == sorted_len &&
      ready->tiles_n == job.tiles_n && ready->k_steps == job.k_steps && ready->may_split == job.may_split) {
    p.tile_table = table = ready->table;
    ready->built = 0;   // (the routing may change in place before another call)
    if (!twin) table_small = table + moe_one_table_bytes(sorted_len) / sizeof(int32_t);
  } else {
    // the layer's next GEMM, if it is one for both tile sizes as well, with the room for partial tiles it would be given
    sonar_moe_tables* next = layer.next;
    if (two_sizes && next != nullptr && next->size_k % kTileK == 0 && next->num_groups > 0 &&
        next->table_bytes >= moe_tile_table_bytes(sorted_len, num_experts)) {
      TileParams q = p;
      q.size_n = (int)next->size_n, q.size_k = (int)next->size_k;
      q.num_groups = (int)next->num_groups, q.group_size = (int)(next->size_k / next->num_groups);
      q.tiles_n = (int)((next->size_n + kTileN - 1) / kTileN);
      if (has_two_sizes(q)) {
        next_job = {next->table, next->table + moe_one_table_bytes(sorted_len) / sizeof(int32_t), q.tiles_n, q.size_k / kTileK,
                    !no_live_split && moe_tile_partial_bytes(q.size_k) > 0 && may_cut(q)};
        if (is_twin(q, next_job.may_split)) next_job.table_small = nullptr, next_job.may_split = kTwinTiles;
        next->expert_ids = expert_ids, next->sorted_len = sorted_len;
        next->tiles_n = next_job.tiles_n, next->k_steps = next_job.k_steps, next->may_split = next_job.may_split;
        next->built = 1;
      }
    }
    auto build_table = [&](auto kernel, int threads) {
      kernel<<<next_job.table != nullptr ? 2 : 1, threads, 0, st>>>(expert_ids, num_post_pad, blocks_max, 64, (int)num_experts,
                                                                    max_tiles, job, next_job);
    };
    if (blocks_max <= 256) build_table(moe_tile_table_kernel<4>, 256);
    else build_table(moe_tile_table_kernel<16>, 1024);
    if (int rc = launch_status("moe_tile_table_kernel")) return rc;
  }
  auto reduce = [&](const TileParams& q) -> int {
    if (q.partial == nullptr) return SONAR_OK;
    const int64_t tiles = std::min<int64_t>((int64_t)max_tiles * q.tiles_n, kLiveSplitTilesMax);
    const dim3 blocks((unsigned)std::min<int64_t>(tiles * (q.tile_rows / 4), 1024), q.table_small != nullptr ? 2 : 1);
    if (dtype == SONAR_DTYPE_F16) moe_tile_reduce_kernel<_Float16><<<blocks, 256, 0, st>>>(q);
    else moe_tile_reduce_kernel<__bf16><<<blocks, 256, 0, st>>>(q);
    return launch_status("moe_tile_reduce_kernel");
  };
  if (twin) return launch_twin<true>(p, dtype, fp4, st);
  if (two_sizes) {
    p.table_small = table_small;
    if (int rc = launch_pair<true>(p, max_tiles, dtype, fp4, bits, fp8, st)) return rc;
    return reduce(p);
  }
  int rc;
  if (nvfp4)
    rc = dtype == SONAR_DTYPE_F16 ? launch_tile_wide_nvfp4<_Float16, true>(p, st)
                                  : launch_tile_wide_nvfp4<__bf16, true>(p, st);
  else if (wide)   // 8-bit codes with groups of 32 rows
    rc = dtype == SONAR_DTYPE_F16 ? launch_tile_wide8<_Float16, true>(p, fp8, st)
                                  : launch_tile_wide8<__bf16, true>(p, fp8, st);
  else
    rc = launch_tile_async_type<true>(p, dtype, bits, st);
  if (rc) return rc;
  if (int rc2 = launch_status("tile kernel (grouped)")) return rc2;
  return reduce(p);
}

}  // namespace sonar

// ---------------------------------------------------------------------------
// Diagnostics for host-side tests (no counterpart in the reference): which tile and which K
// steps every workgroup id of the tile kernels' launches works on, from the same planning and
// mapping code the launches and the kernels run.  One row of six int32 per workgroup that has
// work: launch, rows of a tile, row tile, column tile, first K step, end of its K steps.
namespace {
int64_t schedule_rows(const sonar::TileParams& p, const sonar::TileParams& mapped, int launch, int32_t* out,
                      int64_t out_rows, int64_t at) {
  using namespace sonar;
  const int grid = tile_grid(p);
  const int k_steps = p.size_k / kTileK;
  for (int block = 0; block < grid; ++block) {
    int tile, split, tile_m, tile_n;
    bool whole_k;
    if (!tile_of_block(mapped, block, tile, split, whole_k)) continue;
    tile_coords(mapped, tile, tile_m, tile_n);
    if (at < out_rows) {
      int32_t* row = out + 6 * at;
      row[0] = launch;
      row[1] = mapped.tile_rows;
      row[2] = tile_m;
      row[3] = tile_n;
      row[4] = whole_k ? 0 : split * mapped.k_steps_per_split;
      row[5] = whole_k ? k_steps : std::min(k_steps, row[4] + mapped.k_steps_per_split);
    }
    ++at;
  }
  return at;
}
// A launch with both tile sizes, reported as launch 0 (256-row tiles) and launch 1.
int64_t pair_schedule_rows(const sonar::TileParams& p, int big_word, int small_word, int grid, int32_t* out, int64_t out_rows) {
  using namespace sonar;
  int64_t at = 0;
  for (int block = 0; block < grid; ++block) {
    PairTile t;
    if (!pair_tile_of_block(p, big_word, small_word, block, t)) continue;
    if (at < out_rows) {
      const int32_t row[6] = {t.rows == kTileM ? 0 : 1, t.rows, t.tile_m, t.tile_n, t.k_first, t.k_tiles};
      std::copy(row, row + 6, out + 6 * at);
    }
    ++at;
  }
  return at;
}
}  // namespace

// What the choice between the mid-size and the tile kernels takes the latter's time to be, in us, for 4-bit integer codes.
extern "C" double sonar_debug_tile_estimate(int64_t size_m, int64_t size_n, int64_t size_k) {
  using namespace sonar;
  return tile_estimate(size_m, size_n, size_k, kTileStepInt4, true, plan_rows_97_128(size_m, size_n, size_k, true));
}

// A dense call that runs as 128-row tiles two at a time (`format`: 0 integers, 1 MXFP4); no rows: it runs otherwise.
extern "C" int64_t sonar_debug_twin_schedule(int64_t size_m, int64_t size_n, int64_t size_k, int64_t num_groups, int dtype, int format,
                                             int32_t* out, int64_t out_rows) {
  using namespace sonar;
  if (size_m <= 0 || size_n <= 0 || size_k <= 0 || size_k % kTileK != 0 || num_groups < 1 || size_k % num_groups != 0)
    return -1;
  const int group_size = (int)(size_k / num_groups);
  static float4 never_read;
  const TileLaunches plan = plan_tile_launches(dense_tile_shape(size_m, size_n, size_k, num_groups, group_size), size_m, size_n, size_k,
                                               num_groups, group_size, &never_read, ~(size_t)0, format == 1, false, 4, false,
                                               dtype == SONAR_DTYPE_F16);
  return plan.twin ? schedule_rows(plan.launch, plan.launch, 0, out, out_rows, 0) : 0;
}

// Whether a grouped call that the wide tile kernels take runs as 128-row tiles two at a time.
extern "C" int sonar_debug_moe_twin(int64_t rows_total, int64_t sorted_len, int64_t num_experts, int64_t size_n, int64_t size_k,
                                    int64_t num_groups, int dtype, int format, int may_split) {
  using namespace sonar;
  if (rows_total <= 0 || rows_total >= (1LL << 30) || size_n <= 0 || size_k <= 0 || size_k % kTileK != 0 || num_groups < 1 ||
      size_k % num_groups != 0)
    return -1;
  TileParams q = {};
  q.rows_total = (int)rows_total;
  q.size_k = (int)size_k;
  q.num_groups = (int)num_groups;
  q.group_size = (int)(size_k / num_groups);
  q.tiles_n = (int)((size_n + kTileN - 1) / kTileN);
  return moe_twin_tiles(q, sorted_len, num_experts, 4, format == 1, false, dtype == SONAR_DTYPE_F16, may_split != 0) ? 1 : 0;
}

// A dense call (4-bit integer codes, no act-order) with room for every partial tile, as the other tile kernels run it.
extern "C" int64_t sonar_debug_tile_schedule(int64_t size_m, int64_t size_n, int64_t size_k, int64_t num_groups,
                                             int32_t* out, int64_t out_rows) {
  using namespace sonar;
  if (size_m <= 0 || size_n <= 0 || size_k <= 0 || size_k % kTileK != 0 || num_groups < 1 || size_k % num_groups != 0)
    return -1;
  const int group_size = (int)(size_k / num_groups);
  static float4 never_read;
  const TileLaunches plan =
      plan_tile_launches(dense_tile_shape(size_m, size_n, size_k, num_groups, group_size), size_m, size_n, size_k,
                         num_groups, group_size, &never_read, ~(size_t)0, false, false, 4, false, true, false);
  if (!plan.pair) return schedule_rows(plan.launch, plan.launch, 0, out, out_rows, 0);
  return pair_schedule_rows(plan.launch, 0, 0, pair_grid(plan.launch, 0), out, out_rows);
}

// A grouped call of one tile size whose routing made `row_tiles` row tiles, launched for up to
// `max_row_tiles` of them; `with_partial`: the call has room for partial tiles.
extern "C" int64_t sonar_debug_moe_tile_schedule(int64_t row_tiles, int64_t max_row_tiles, int64_t size_n,
                                                 int64_t size_k, int with_partial, int32_t* out, int64_t out_rows) {
  using namespace sonar;
  if (row_tiles < 0 || row_tiles > max_row_tiles || size_n <= 0 || size_k <= 0 || size_k % kTileK != 0) return -1;
  static float4 never_read;
  static int32_t no_table;
  TileParams p = dense_tile_shape(max_row_tiles * kTileM, size_n, size_k, 1, (int)size_k);
  p.tiles_m = (int)max_row_tiles;
  p.tile_table = &no_table;
  if (with_partial && moe_tile_partial_bytes(size_k) > 0) p.partial = &never_read;
  return schedule_rows(p, live_tiles_of(p, (int)row_tiles), 0, out, out_rows, 0);
}

// A grouped call whose routing made `big` row tiles of three or four blocks and `small` of one or two, with both tile
// sizes in one launch, for up to `max_row_tiles` blocks.  What the device would choose comes back in `chosen`: 256-row tiles
// that are halved, K ranges of the tiles of each size.
extern "C" int64_t sonar_debug_moe_pair_schedule(int64_t big, int64_t small, int64_t max_row_tiles, int64_t size_n,
                                                 int64_t size_k, int with_partial, int32_t* chosen, int32_t* out,
                                                 int64_t out_rows) {
  using namespace sonar;
  if (big < 0 || small < 0 || 3 * big + small > max_row_tiles || size_n <= 0 || size_k <= 0 || size_k % kTileK != 0)
    return -1;
  static float4 never_read;
  static int32_t no_table;
  TileParams p = dense_tile_shape(max_row_tiles * kTileM, size_n, size_k, 1, (int)size_k);
  p.tiles_m = (int)max_row_tiles;
  p.tile_table = p.table_small = &no_table;
  const int k_steps = p.size_k / kTileK;
  if (with_partial && moe_tile_partial_bytes(size_k) > 0) p.partial = &never_read;
  const bool may_split = p.partial != nullptr;
  float best = 0.f;
  PairPlan plan = pair_plan(0, (int)big, may_split);
  for (int i = 0; i < pair_plans((int)big, may_split); ++i) {
    const PairPlan one = pair_plan(i, (int)big, may_split);
    if (!pair_has_room((int)big, (int)small, one, p.tiles_n, k_steps)) continue;
    const float cost = pair_cost((int)big, (int)small, one, p.tiles_n, k_steps);
    if (i == 0 || cost < best) best = cost, plan = one;
  }
  chosen[0] = plan.halved;
  chosen[1] = plan.splits[0];
  chosen[2] = plan.splits[1];
  return pair_schedule_rows(p, pair_word((int)big - plan.halved, plan.splits[0]),
                            pair_word((int)small + 2 * plan.halved, plan.splits[1]), pair_grid(p, (int)max_row_tiles), out, out_rows);
}
