// W4A8: 4-bit weights, 8-bit activations, on the full-rate 8-bit matrix instructions with 32 x 32 results
// (v_mfma_i32_32x32x32_i8, v_mfma_f32_32x32x64_f8f6f4), from 17 rows up.
//
// A wavefront owns 32 R rows x one 64-column strip of its range of K, and dequantises its strip's packed codes by
// itself; a workgroup is S strips x RG ranges.  Few rows: 2 strips x 4 ranges, so that a small grid still has two
// wavefronts on every SIMD; many rows: 4 strips, one range, two workgroups on a compute unit.  32 x 32 results
// because one instruction then spans a group of 32 (int8), which the 16 x 16 forms do at half their rate only, takes
// half the issue slots, and has a column per lane: the group's scale is one register.  The weight order holds a
// column's 32 rows of a chunk in four lanes; v_permlane16_swap, one per two packed words, makes it two.
//
// What bounds it: with few rows the vector instructions that dequantise (9.5 per packed word, of which 2 put the
// bytes into the order of K).  With many rows vector instructions and waits: at 2048 rows, K 4096, N 11008, int8, 10.0 other vector
// instructions go with a matrix instruction (16 multiply-adds of the group scales per tile and group, and a wavefront
// dequantises its whole strip for 128 rows), vector issue fills 57 % of the cycles, the matrix pipes 41 %, a fifth of the
// wavefronts' time is waits, and 13 % of the cycles are bank conflicts; 1.5 POP/s, where the int8 instruction alone reaches 3.15 on
// random operands.  R = 3 with 256 registers, R = 4 where the scales in flight leave room for it.
// Measured against the kernels it takes over from (us, before -> now):
//   M  153, K 1152, N 22976, fp8:  42 -> 23       M  259, K 3456, N 20032, int8: 172 -> 40
//   M  987, K 1664, N 12608, int8: 206 -> 55      M 2048, K 4096, N 11008, int8: 181 -> 137
//   M 1929, K 3072, N 25216, int8, groups of 32, zero points: 1836 -> 536
//   44 random shapes of 17 to 8192 rows: 1.69 times as fast (geometric mean; one, of 25 rows, 0.89)
// and since rows of C leave as whole lines (they were 2-byte stores from a lane's column):
//   M 1024, K 4096, N  8192, int8: 67 -> 56       M 2048, K 4096, N 11008, int8: 146 -> 124 (the same box)
//   M   64, K 4096, N 11008, int8, 64 rows a tile: 18.8 -> 17.2      M 1213, K 1152, N 6336: 39 -> 24 with the quantisation
// and since copies have a scalar base and 32-bit offsets:
//   M 2048, K 4096, N 11008, int8, with the quantisation: 118.3 -> 116.6
//
// Pipeline, per step of 128 rows of K: activations (shared by the strips of a range) and packed codes (a wavefront's
// own) go to LDS by LDS-DMA and the scales to registers, two steps ahead (three with one row block), and one
// barrier a step.  The operands of a row block replace those of the one before as its last matrix instructions issue; the
// left half of the next step's weights is dequantised behind the last tile of a step, the right half behind the first;
// a group's totals are scaled behind the matrix instructions of the next group.
#include <type_traits>

#include "common.hpp"
#include "dequant.hpp"
#include "gemm_a8_block.hpp"

namespace sonar {
namespace {

typedef int intx4_t __attribute__((ext_vector_type(4)));
typedef int intx8_t __attribute__((ext_vector_type(8)));
typedef int intx16_t __attribute__((ext_vector_type(16)));
typedef float floatx16_t __attribute__((ext_vector_type(16)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kStepK = 128;        // rows of K a step takes from each range: four chunks
constexpr int kStepBytes = 4096;   // LDS bytes of 32 rows of A, or of a strip's packed codes, of a step
constexpr int kTurnRow = 144;      // bytes between rows of results in LDS: the halves of a wavefront write to banks of their own

// Steps between asking for a stage and using it.  One row block is bound by memory and its steps are short.
constexpr int a8_ahead(int rows) { return rows == 1 ? 3 : 2; }
constexpr int a8_lds(int rows, int strips, int ranges) {
  const int stages = (ranges * (a8_ahead(rows) + 1) * rows + strips * ranges * a8_ahead(rows)) * kStepBytes;
  const int end = (ranges > 1 ? strips * ranges * 8192 : 0) + strips * 32 * kTurnRow + 32 * rows * 4;
  return stages > end ? stages : end;
}

// A chunk's word (rows 8 b .. 8 b + 7 of a column, nibbles in the order {0, 2, 4, 6, 1, 3, 5, 7}) -> eight operand
// bytes in the order of K.
struct BlockInt8 {
  typedef intx16_t acc_t;
  typedef int scalar_t;
  static constexpr bool kFp8 = false;
  static constexpr int kWide = 1;   // chunks of K per matrix instruction
  // uint4b8, channelwise: 16 (q - 8) in the byte; the factor leaves at the end
  static __device__ __forceinline__ u32x2_t shifted(uint32_t w) {
    const uint32_t x = w ^ 0x88888888u;
    const uint32_t lo = (x << 4) & 0xf0f0f0f0u, hi = x & 0xf0f0f0f0u;
    return u32x2_t{__builtin_amdgcn_perm(hi, lo, 0x06040200u), __builtin_amdgcn_perm(hi, lo, 0x07050301u)};
  }
  // q - z: (q + 0x80 - z) ^ 0x80 carries nothing between the bytes; `bias` = 0x80 - z in each
  static __device__ __forceinline__ u32x2_t word(uint32_t w, uint32_t bias) {
    const uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;
    const uint32_t n0 = __builtin_amdgcn_perm(hi, lo, 0x06040200u), n1 = __builtin_amdgcn_perm(hi, lo, 0x07050301u);
    return u32x2_t{(n0 + bias) ^ 0x80808080u, (n1 + bias) ^ 0x80808080u};
  }
  static __device__ __forceinline__ uint32_t zero_bytes(uint32_t z) {
    return 0x80808080u - __builtin_amdgcn_perm(z, z, 0);
  }
  static __device__ __forceinline__ acc_t mfma(u32x4_t a, u32x4_t b, acc_t c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(intx4_t, a), __builtin_bit_cast(intx4_t, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ int scaled(int total, int scale, int acc) { return acc + __mul24(total, scale); }
};

struct BlockFp8 {
  typedef floatx16_t acc_t;
  typedef float scalar_t;
  static constexpr bool kFp8 = true;
  static constexpr int kWide = 2;
  static __device__ __forceinline__ u32x2_t shifted(uint32_t w) { return word(w, 0); }
  // p: sign and magnitude as marlin_int4_fp8_preprocess leaves them (p < 8: p, else -((p & 7) + 1)), read as a
  // float8_e4m3fn byte with a zero exponent field; the scales carry the factor 512
  static __device__ __forceinline__ uint32_t four(uint32_t p) {
    const uint32_t s = p & 0x08080808u;
    return ((p & 0x07070707u) | (s << 4)) + (s >> 3);
  }
  static __device__ __forceinline__ u32x2_t word(uint32_t w, uint32_t) {
    const uint32_t h = w >> 4;
    return u32x2_t{four(__builtin_amdgcn_perm(h, w, 0x06040200u)), four(__builtin_amdgcn_perm(h, w, 0x07050301u))};
  }
  // with zero points: q + z >= 16 ? .. as the nibble was stored: sign and magnitude of q - z
  static __device__ __forceinline__ uint32_t four_zp(uint32_t p, uint32_t z4) {
    const uint32_t q0 = p | 0x70707070u;
    const uint32_t s = (q0 + z4) & 0x80808080u;
    return ((q0 + (s >> 7) * ((z4 & 0xffu) + 1)) & 0x0f0f0f0fu) | s;
  }
  static __device__ __forceinline__ u32x2_t word_zp(uint32_t w, uint32_t z4) {
    const uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;
    return u32x2_t{four_zp(__builtin_amdgcn_perm(hi, lo, 0x06040200u), z4),
                   four_zp(__builtin_amdgcn_perm(hi, lo, 0x07050301u), z4)};
  }
  static __device__ __forceinline__ uint32_t zero_bytes(uint32_t z) { return __builtin_amdgcn_perm(z, z, 0); }
  static __device__ __forceinline__ acc_t mfma(intx8_t a, intx8_t b, acc_t c) {
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 127, 0, 127);
  }
  static __device__ __forceinline__ float scaled(float total, float scale, float acc) { return acc + total * scale; }
};

__device__ __forceinline__ uint32_t a8_bits(int v) { return (uint32_t)v; }
__device__ __forceinline__ uint32_t a8_bits(float v) { return __float_as_uint(v); }
__device__ __forceinline__ void a8_from_bits(uint32_t b, int& v) { v = (int)b; }
__device__ __forceinline__ void a8_from_bits(uint32_t b, float& v) { v = __uint_as_float(b); }

__device__ __forceinline__ float a8_number(uint16_t bits, bool bf16) {
  return bf16 ? __uint_as_float((uint32_t)bits << 16) : (float)__builtin_bit_cast(_Float16, bits);
}

// ZP: zero points; GC: chunks per group (0: channelwise)
template <typename ACT, bool ZP, int GC, int R, int S, int RG>
__global__ __launch_bounds__(64 * S * RG) __attribute__((amdgpu_waves_per_eu(2, 2))) void marlin_a8_block(
    const A8BlockParams p) {
  typedef typename ACT::acc_t acc_t;
  typedef typename ACT::scalar_t scalar_t;
  constexpr int kWaves = S * RG;
  constexpr int kAhead = a8_ahead(R), kRing = kAhead + 1;
  constexpr int kLoadsA = 4 * R / S;                       // 1-KiB copies of a wavefront per step
  constexpr int kGroups = GC == 0 ? 0 : 4 / GC;            // groups per step
  constexpr int kOpsW = 4 + kGroups * (ZP ? 3 : 2);
  constexpr int kWide = ACT::kWide, kPerSeg = 4 / kWide;   // matrix instructions per 32 x 32 tile and step
  constexpr bool kShifted = GC == 0 && !ZP && !ACT::kFp8;
  static_assert(4 * R % S == 0 && (GC == 0 || GC >= kWide), "");
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int range = wave / S, ws = wave % S;

  // Workgroup ids congruent mod 8 run on one XCD: each takes a contiguous run of tiles, the row tiles of the same
  // columns next to each other.
  const int units = p.tiles * p.splits, per_xcd = (units + 7) / 8;
  const int unit = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || unit >= units) return;
  const int split = unit / p.tiles, tile = unit - split * p.tiles;
  const int tile_n = tile / p.tiles_m, tile_m = tile - tile_n * p.tiles_m;
  const int m0 = tile_m * 32 * R;
  const int strips = p.size_n / kStripN;
  const bool active = tile_n * S + ws < strips;   // strips past the last repeat it and are not stored
  const int strip = __builtin_amdgcn_readfirstlane(active ? tile_n * S + ws : strips - 1);

  const int first = split * p.split_steps;       // of the steps this workgroup takes
  const int all_steps = p.size_k / kStepK, steps = min(first + p.split_steps, all_steps);
  const int per_range = (steps - first + RG - 1) / RG;
  const int k_first = first + range * per_range;
  const int count = min(per_range, steps - k_first);   // of this range; the others' barriers are kept company

  // ---- sources.  Rows of A are copied 8 x 128 bytes at a time; piece q of row r sits at slot q ^ (r % 8).
  uint32_t a_off[kLoadsA];
#pragma unroll
  for (int i = 0; i < kLoadsA; ++i) {
    int row = m0 + 8 * (ws * kLoadsA + i) + (lane >> 3);
    if (row >= p.size_m) row = p.size_m - 1;   // rows past M are computed and never stored
    a_off[i] = (uint32_t)row * (uint32_t)p.lda + 16 * ((lane & 7) ^ (lane >> 3));
  }
  const char* b_base = reinterpret_cast<const char*>(p.w) + (size_t)strip * all_steps * kStepBytes;
  const uint32_t b_off = 16 * lane;
  const char* s_base = reinterpret_cast<const char*>(p.scales + (size_t)strip * kStripN);
  const uint32_t s_off = 2 * scale_slot(l32, false);
  const char* z_base = reinterpret_cast<const char*>(p.zeros + (size_t)strip * (kStripN / 8));
  const uint32_t z_off = 4 * (lane & 7);
  char* a_stage = smem + range * (kRing * R * kStepBytes);
  char* w_stage = smem + RG * kRing * R * kStepBytes + wave * (kAhead * kStepBytes);
  const uint32_t a_lds = (uint32_t)(uintptr_t)(lds_void_t*)a_stage;
  const uint32_t w_stage_lds = (uint32_t)(uintptr_t)(lds_void_t*)w_stage, w_lds = w_stage_lds + 16 * lane;

  // uint16 scales of both column halves and zero-point words of the steps in flight
  uint32_t sv[kRing][kGroups ? kGroups : 1][2], zv[kRing][kGroups ? kGroups : 1];
  auto issue_w = [&](const int ring, int wslot, int k) __attribute__((always_inline)) {
    k = min(k_first + k, steps - 1);
    const char* src = b_base + (size_t)k * kStepBytes;
    copy_4k_to_lds<false>(w_stage_lds + wslot * kStepBytes, b_off, src);
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      const char* s_src = s_base + (size_t)(k * kGroups + g) * p.size_n * 2;
      asm volatile("global_load_ushort %0, %1, %2" : "=&v"(sv[ring][g][0]) : "v"(s_off), "s"(s_src) : "memory");
      asm volatile("global_load_ushort %0, %1, %2 offset:64" : "=&v"(sv[ring][g][1]) : "v"(s_off), "s"(s_src) : "memory");
      if constexpr (ZP) {
        const char* z_src = z_base + (size_t)(k * kGroups + g) * (p.size_n / 2);
        asm volatile("global_load_dword %0, %1, %2" : "=&v"(zv[ring][g]) : "v"(z_off), "s"(z_src) : "memory");
      }
    }
  };
  auto issue_a = [&](const int ring, int k) __attribute__((always_inline)) {
    const char* src = reinterpret_cast<const char*>(p.a) + (size_t)min(k_first + k, steps - 1) * kStepK;
#pragma unroll
    for (int i = 0; i < kLoadsA; ++i)
      copy_to_lds<16>(a_lds + ring * (R * kStepBytes) + (ws * kLoadsA + i) * 1024, a_off[i], src);
  };
  // until only the `n` youngest operations are outstanding; the registers of ring position `ring` have landed
  auto landed = [&](const int ring, const int n) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(n) : "memory");
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      asm volatile("" : "+v"(sv[ring][g][0]), "+v"(sv[ring][g][1]));
      if constexpr (ZP) asm volatile("" : "+v"(zv[ring][g]));
    }
  };

  const int nibble = 8 * (lane >> 4 & 1) + 4 * (lane >> 3 & 1);   // + 16 for the right half: bits of a zero-point word
  uint32_t one_zero[2] = {0x78787878u, 0x78787878u};              // channelwise, or uint4b8: q - 8
  if constexpr (GC == 0 && ZP) {
    const uint32_t zw = p.zeros[(size_t)strip * (kStripN / 8) + (lane & 7)];
#pragma unroll
    for (int j = 0; j < 2; ++j) one_zero[j] = ACT::zero_bytes((zw >> (nibble + 16 * j)) & 15u);
  }

  acc_t acc[R][2], tmp[2];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    tmp[0][i] = tmp[1][i] = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r][0][i] = acc[r][1][i] = 0;
  }
  scalar_t pending_scale = 0;   // of the last group of the step before

  u32x4_t av[4];                 // this lane's bytes of the four chunks of a row block
  u32x2_t xw[2][4];              // packed words of a column half
  typedef typename std::conditional<ACT::kFp8, intx8_t, u32x4_t>::type operand_t;
  operand_t bq[2][kPerSeg];      // operands of a column half
  uint32_t zb[2] = {one_zero[0], one_zero[1]};

  uint32_t a_at[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) a_at[c] = a_lds + l32 * 128 + (((2 * c + half) ^ (l32 & 7)) * 16);

#define SONAR_A8_READ_A(ring, rb, c)                                                              \
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(av[c]) : "v"(a_at[c]),                      \
               "i"((ring) * (R * kStepBytes) + (rb) * kStepBytes) : "memory")
#define SONAR_A8_READ_W(j, c, at)                                                                 \
  asm volatile("ds_read_b64 %0, %1 offset:%2" : "=&v"(xw[j][c]) : "v"(at), "i"((c) * 1024 + (j) * 8) : "memory")

  // chunk c of column half j of the step in ring position `ring`, from xw
  auto dequant = [&](const int ring, const int j, const int c) __attribute__((always_inline)) {
    // lanes 16 .. 31 and 48 .. 63 hold rows 8 .. 15 and 24 .. 31 of the left sixteen columns of the half, which the
    // others hold the rows before of: swapped with the right sixteen columns, a lane has 16 rows of one column
    const auto y = __builtin_amdgcn_permlane16_swap(xw[j][c].x, xw[j][c].y, false, false);
    xw[j][c] = u32x2_t{y[0], y[1]};   // (in place: as copies they took eight instructions and registers a half)
    if constexpr (ZP && GC != 0) {
      if (c % GC == 0) zb[j] = ACT::zero_bytes((zv[ring][c / GC] >> (nibble + 16 * j)) & 15u);
    }
    u32x2_t lo, hi;
    if constexpr (kShifted) {
      lo = ACT::shifted(y[0]);
      hi = ACT::shifted(y[1]);
    } else if constexpr (ACT::kFp8 && ZP) {
      lo = ACT::word_zp(y[0], zb[j]);
      hi = ACT::word_zp(y[1], zb[j]);
    } else {
      lo = ACT::word(y[0], zb[j]);
      hi = ACT::word(y[1], zb[j]);
    }
    if constexpr (ACT::kFp8) {
      operand_t& o = bq[j][c >> 1];
      const int at = 4 * (c & 1);
      o[at] = (int)lo.x, o[at + 1] = (int)lo.y, o[at + 2] = (int)hi.x, o[at + 3] = (int)hi.y;
    } else {
      bq[j][c] = u32x4_t{lo.x, lo.y, hi.x, hi.y};
    }
  };
  auto scale_of = [&](uint32_t bits) __attribute__((always_inline)) -> scalar_t {
    if constexpr (ACT::kFp8) return a8_number((uint16_t)bits, p.bf16);
    else return (int)bits;
  };

  // One 32 x 32 tile (row block rb, column half j) of a step in ring position `ring`: its matrix instructions, and
  // behind each of them
  //  - a share of adding the group before, times its scale, to its totals;
  //  - j = 1: the read of the row block that follows, chunk by chunk into the registers just used;
  //  - last row block: the packed words of the next step, its left half's operands (whose last user was the tile
  //    before this one); first row block: its right half's.
  auto tile_step = [&](const int ring, const int rb, const int j, uint32_t w_next) __attribute__((always_inline)) {
    const int next_ring = (ring + 1) % kRing;
    constexpr int kPerGroup = GC == 0 ? 1 : GC / kWide;
#pragma unroll
    for (int m = 0; m < kPerSeg; ++m) {
      const int c0 = m * kWide, cl = c0 + kWide - 1;
      int younger = -1;   // LDS reads that may still be under way
      if (j == 0 && rb == 0) younger = 2 * (3 - cl) + (R == 1 ? c0 : 0);
      else if (j == 0) younger = (3 - cl) + (rb == R - 1 ? c0 : 0);
      else if (rb == R - 1) younger = (3 - cl) + 2 * c0;
      if (younger >= 0) {
        asm volatile("s_waitcnt lgkmcnt(%0)" ::"i"(younger) : "memory");
#pragma unroll
        for (int c = c0; c <= cl; ++c) {
          if (j == 0) asm volatile("" : "+v"(av[c]));
          if (j == 0 && rb == 0) asm volatile("" : "+v"(xw[1][c]));
          if (j == 1 && rb == R - 1) asm volatile("" : "+v"(xw[0][c]));
        }
      }
      operand_t a;
      if constexpr (ACT::kFp8) {
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = (int)av[c0][i], a[4 + i] = (int)av[cl][i];
      } else {
        a = av[c0];
      }
      const int group = GC == 0 ? 0 : (rb * 2 + j) * kGroups + c0 / (GC ? GC : 1);   // within the step
      if constexpr (GC == 0) {
        acc[rb][j] = ACT::mfma(a, bq[j][m], acc[rb][j]);
      } else {
        if (m % kPerGroup == 0) {
          acc_t zero;
#pragma unroll
          for (int i = 0; i < 16; ++i) zero[i] = 0;
          tmp[group & 1] = ACT::mfma(a, bq[j][m], zero);
        } else {
          tmp[group & 1] = ACT::mfma(a, bq[j][m], tmp[group & 1]);
        }
        const int before = group - 1;
        const int prb = group == 0 ? R - 1 : before / kGroups / 2, pj = group == 0 ? 1 : before / kGroups % 2;
        const scalar_t scale = group == 0 ? pending_scale : scale_of(sv[ring][before % kGroups][pj]);
        const int at = m % kPerGroup;
        const int from = kPerGroup == 1 ? 0 : (at == 0 ? 0 : 16 * (at - 1) / (kPerGroup - 1));
        const int to = kPerGroup == 1 ? 16 : 16 * at / (kPerGroup - 1);
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (i >= from && i < to) acc[prb][pj][i] = ACT::scaled(tmp[(group & 1) ^ 1][i], scale, acc[prb][pj][i]);
      }
#pragma unroll
      for (int c = c0; c <= cl; ++c) {
        if (rb == 0 && j == 0) dequant(ring, 1, c);
        if (rb == R - 1 && j == 1) dequant(next_ring, 0, c);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = c0; c <= cl; ++c) {
        if (rb == R - 1 && j == 0) SONAR_A8_READ_W(0, c, w_next);
        if (j == 1) {
          if (rb < R - 1) {
            SONAR_A8_READ_A(ring, rb + 1, c);
          } else {
            SONAR_A8_READ_A(next_ring, 0, c);
            SONAR_A8_READ_W(1, c, w_next);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- prologue
#pragma unroll
  for (int t = 0; t < kAhead; ++t) {
    issue_w(t, t, t);
    issue_a(t, t);
  }
  landed(0, (kAhead - 1) * (kOpsW + kLoadsA));
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int c = 0; c < 4; ++c) SONAR_A8_READ_W(0, c, w_lds);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int c = 0; c < 4; ++c) asm volatile("" : "+v"(xw[0][c]));
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    SONAR_A8_READ_A(0, 0, c);
    SONAR_A8_READ_W(1, c, w_lds);
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) dequant(0, 0, c);

  // One step.  Its only barrier is before the last row block: behind it stage t + 1 has landed for everyone and
  // nobody reads the activations of step t - 1 any more, whose place those of step t + kAhead take.
  int wslot = 0;
  auto step = [&](const int ring, int t) __attribute__((always_inline)) {
    const int next_slot = wslot == kAhead - 1 ? 0 : wslot + 1;
    const uint32_t w_next = w_lds + next_slot * kStepBytes;
    const int fill = (ring + kAhead) % kRing;
    const bool live = t < count;
    if constexpr (R > 1) {
      if (live) tile_step(ring, 0, 0, w_next);
      issue_w(fill, wslot, t + kAhead);
      if (live) {
        tile_step(ring, 0, 1, w_next);
#pragma unroll
        for (int rb = 1; rb < R - 1; ++rb) {
          tile_step(ring, rb, 0, w_next);
          tile_step(ring, rb, 1, w_next);
        }
      }
      landed((ring + 1) % kRing, kOpsW);
    } else {
      landed((ring + 1) % kRing, kOpsW + kLoadsA);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (live) tile_step(ring, R - 1, 0, w_next);
    if constexpr (R == 1) issue_w(fill, wslot, t + kAhead);
    issue_a(fill, t + kAhead);
    if (live) {
      tile_step(ring, R - 1, 1, w_next);
      if constexpr (GC != 0) pending_scale = scale_of(sv[ring][kGroups - 1][1]);
    }
    wslot = next_slot;
  };
  for (int t = 0; t < per_range; t += kRing) {
    step(0, t);
    if (t + 1 < per_range) step(1, t + 1);
    if (t + 2 < per_range) step(2, t + 2);
    if constexpr (kRing > 3)
      if (t + 3 < per_range) step(3, t + 3);
  }
  if constexpr (GC != 0) {
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[R - 1][1][i] = ACT::scaled(tmp[1][i], pending_scale, acc[R - 1][1][i]);
  }
  // copies and reads still under way must not outlive this point
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int c = 0; c < 4; ++c) asm volatile("" : "+v"(av[c]), "+v"(xw[0][c]), "+v"(xw[1][c]));
#pragma unroll
  for (int r = 0; r < kRing; ++r)
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      asm volatile("" : "+v"(sv[r][g][0]), "+v"(sv[r][g][1]));
      if constexpr (ZP) asm volatile("" : "+v"(zv[r][g]));
    }
#undef SONAR_A8_READ_A
#undef SONAR_A8_READ_W

  // ---- results.  Element i of a tile: row 8 (i / 4) + 4 half + i % 4, column l32.
  int at_end = lane;   // a register of its own: what is computed from it is not kept through the loop
  asm volatile("" : "+v"(at_end));
  const int end_l32 = at_end & 31, end_half = at_end >> 5;
  const bool bf16 = p.bf16 != 0;
  float col_scale[2] = {1.f, 1.f}, bias[2] = {0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int slot = strip * kStripN + scale_slot(32 * j + end_l32, false);
    if (GC == 0) col_scale[j] = a8_number(p.scales[slot], bf16);
    if (p.bias) bias[j] = a8_number(p.bias[slot], bf16);
  }
  auto number = [&](scalar_t total, float row_scale, int j) __attribute__((always_inline)) -> uint16_t {
    // every step rounds to fp32 as written; contraction would fuse them
#pragma clang fp contract(off)
    if constexpr (kShifted) total >>= 4;
    float f = (float)total * row_scale;
    if (GC == 0) f *= col_scale[j];
    f += bias[j];
    return bf16 ? __builtin_bit_cast(uint16_t, (__bf16)f) : __builtin_bit_cast(uint16_t, (_Float16)f);
  };
  auto store_raw = [&](scalar_t total, int row, int j) __attribute__((always_inline)) {
    if (row >= p.size_m || !active) return;
    if constexpr (kShifted) total >>= 4;
    p.partial[((size_t)split * p.size_m + row) * p.size_n + strip * kStripN + 32 * j + end_l32] = a8_bits(total);
  };
  // Rows of C leave as whole 128-byte lines, turned in LDS: 2-byte stores straight from a lane's column, each behind the
  // load of its row's scale, took 44 to 54 thousand cycles for 128 x 256 results, a third of the kernel; this takes 10.
  char* sums_end = smem + (RG > 1 ? kWaves * 8192 : 0);
  char* turn = sums_end + (RG > 1 ? ws : wave) * (32 * kTurnRow);
  float* row_scale = reinterpret_cast<float*>(sums_end + (RG > 1 ? S : kWaves) * (32 * kTurnRow));
  const bool wide = (reinterpret_cast<uintptr_t>(p.c) & 15) == 0;
  auto turn_in = [&](scalar_t total, int row, float by, int j) __attribute__((always_inline)) {
    *reinterpret_cast<uint16_t*>(turn + row * kTurnRow + 64 * j + 2 * end_l32) = number(total, by, j);
  };
  // rows 8 q .. 8 q + 7 of row block rb
  auto turn_out = [&](int rb, int q) __attribute__((always_inline)) {
    const int r = 8 * q + (at_end >> 3), row = m0 + 32 * rb + r;
    const uint4 v = *reinterpret_cast<const uint4*>(turn + r * kTurnRow + 16 * (at_end & 7));
    if (row >= p.size_m || !active) return;
    uint16_t* to = p.c + (size_t)row * p.size_n + strip * kStripN + 8 * (at_end & 7);
    if (wide) {
      *reinterpret_cast<uint4*>(to) = v;
    } else {
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) to[e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
    }
  };
  __syncthreads();   // the stages are nobody's any more
  if (p.splits == 1)
    for (int r = threadIdx.x; r < 32 * R; r += 64 * kWaves) row_scale[r] = p.a_scales[min(m0 + r, p.size_m - 1)];
  if constexpr (RG == 1) {
    if (p.splits > 1) {
#pragma unroll
      for (int rb = 0; rb < R; ++rb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) store_raw(acc[rb][j][i], m0 + 32 * rb + 8 * (i >> 2) + 4 * end_half + (i & 3), j);
      return;
    }
    __syncthreads();   // the rows' scales
#pragma unroll
    for (int rb = 0; rb < R; ++rb) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 by = *reinterpret_cast<const float4*>(row_scale + 32 * rb + 8 * q + 4 * end_half);
        const float bys[4] = {by.x, by.y, by.z, by.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) turn_in(acc[rb][j][4 * q + i], 8 * q + 4 * end_half + i, bys[i], j);
      }
      // only this wavefront writes and reads here, and its LDS operations complete in order
#pragma unroll
      for (int q = 0; q < 4; ++q) turn_out(rb, q);
    }
  } else {
    // the ranges meet in LDS, a row block at a time; a wavefront adds 1/RG of its strip's tiles
    uint4* sums = reinterpret_cast<uint4*>(smem);
#pragma unroll
    for (int rb = 0; rb < R; ++rb) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {   // four elements of tile q / 4
        const acc_t& v = acc[rb][q >> 2];
        const int i = 4 * (q & 3);
        const scalar_t v0 = v[i], v1 = v[i + 1], v2 = v[i + 2], v3 = v[i + 3];
        sums[(wave * 8 + q) * 64 + at_end] = make_uint4(a8_bits(v0), a8_bits(v1), a8_bits(v2), a8_bits(v3));
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < 8 / RG; ++u) {
        const int q = range * (8 / RG) + u;
        scalar_t total[4] = {0, 0, 0, 0};
#pragma unroll
        for (int g = 0; g < RG; ++g) {
          const uint4 s = sums[((g * S + ws) * 8 + q) * 64 + at_end];
          scalar_t v;
          a8_from_bits(s.x, v), total[0] += v;
          a8_from_bits(s.y, v), total[1] += v;
          a8_from_bits(s.z, v), total[2] += v;
          a8_from_bits(s.w, v), total[3] += v;
        }
        const int r = 8 * (q & 3) + 4 * end_half;
        if (p.splits > 1) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (q >> 2) store_raw(total[i], m0 + 32 * rb + r + i, 1);
            else store_raw(total[i], m0 + 32 * rb + r + i, 0);
          }
        } else {
          const float4 by = *reinterpret_cast<const float4*>(row_scale + 32 * rb + r);
          const float bys[4] = {by.x, by.y, by.z, by.w};
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (q >> 2) turn_in(total[i], r + i, bys[i], 1);
            else turn_in(total[i], r + i, bys[i], 0);
          }
        }
      }
      __syncthreads();   // the sums have been read, the rows of all ranges stand
      if (p.splits == 1) {
#pragma unroll
        for (int u = 0; u < 4 / RG; ++u) turn_out(rb, range * (4 / RG) + u);
      }
    }
  }
}

template <typename ACT, bool ZP, int GC, int R, int S, int RG>
int launch_a8_shape(A8BlockParams p, int splits, hipStream_t st) {
  constexpr int lds = a8_lds(R, S, RG);
  static_assert(lds <= 160 * 1024, "");
  static bool attr_set = false;   // raising the dynamic LDS limit is needed once per form
  if (!attr_set) {
    SONAR_HIP(hipFuncSetAttribute((const void*)marlin_a8_block<ACT, ZP, GC, R, S, RG>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    attr_set = true;
  }
  p.splits = splits;
  p.tiles_m = (p.size_m + 32 * R - 1) / (32 * R);
  p.tiles = p.tiles_m * ((p.size_n / kStripN + S - 1) / S);
  marlin_a8_block<ACT, ZP, GC, R, S, RG><<<(p.tiles * splits + 7) / 8 * 8, 64 * S * RG, lds, st>>>(p);
  return launch_status("marlin_a8_block");
}

template <typename ACT, bool ZP, int GC>
int launch_a8_groups(const A8BlockParams& p, A8BlockShape s, hipStream_t st) {
  constexpr int kMost = a8_max_row_blocks(ACT::kFp8, ZP, GC);
  if (s.rows == 1) return launch_a8_shape<ACT, ZP, GC, 1, 2, 4>(p, s.splits, st);
  if (s.rows == 2 || kMost == 2) return launch_a8_shape<ACT, ZP, GC, 2, 2, 4>(p, s.splits, st);
  if constexpr (kMost >= 3) {
    if (s.ranges == 2) return launch_a8_shape<ACT, ZP, GC, 3, 4, 2>(p, s.splits, st);
    if constexpr (kMost >= 4)
      if (s.rows == 4) return launch_a8_shape<ACT, ZP, GC, 4, 4, 1>(p, s.splits, st);
    return launch_a8_shape<ACT, ZP, GC, 3, 4, 1>(p, s.splits, st);
  }
  return fail(SONAR_E_INVALID, "internal: %d row blocks", s.rows);
}

template <typename ACT, bool ZP>
int launch_a8_zero(const A8BlockParams& p, A8BlockShape s, hipStream_t st) {
  switch (p.group_chunks) {
    case 0: return launch_a8_groups<ACT, ZP, 0>(p, s, st);
    case 1:
      if constexpr (!ACT::kFp8) return launch_a8_groups<ACT, ZP, 1>(p, s, st);
      return fail(SONAR_E_INVALID, "internal: fp8 activations with groups of 32 rows");
    case 2: return launch_a8_groups<ACT, ZP, 2>(p, s, st);
    default: return launch_a8_groups<ACT, ZP, 4>(p, s, st);
  }
}

}  // namespace

int a8_block_gemm(A8BlockParams p, bool fp8, A8BlockShape shape, hipStream_t st) {
  const int steps = p.size_k / kStepK;
  p.split_steps = (steps + shape.splits - 1) / shape.splits;
  if (fp8) return p.zeros ? launch_a8_zero<BlockFp8, true>(p, shape, st) : launch_a8_zero<BlockFp8, false>(p, shape, st);
  return p.zeros ? launch_a8_zero<BlockInt8, true>(p, shape, st) : launch_a8_zero<BlockInt8, false>(p, shape, st);
}

}  // namespace sonar
