// The GEMM between decode and prefill: from a few tens of rows up to where the tiles of the wide tile
// kernel (gemm_tile.hip) fill the chip.  A workgroup owns 16 MB rows x 128 columns over the whole of K, so that no
// partial tile goes through memory; where that leaves compute units idle, a part of K, and a second kernel adds the parts.
//
// Eight wavefronts: two strips of 64 columns x four ranges of K.  So every packed chunk is dequantised
// exactly once in the workgroup, a wavefront's accumulators are small (16 MB registers), two wavefronts
// share a SIMD (one's matrix instructions run beside the other's dequantisation), and the activations,
// which the two strips share, are staged in LDS at half the bytes per matrix instruction of a one-strip
// workgroup (at one strip the copies alone would need the whole 64 bytes per clock of a compute unit).  Grouped calls of
// many rounds of workgroups take four strips x two ranges (mid_moe_strips): start, end and the sum of the ranges once for twice the columns,
// and half the copies (32 experts of 42 rows, K = 1152, N = 15360: 187 -> 132 us); so do 64-row tiles of 4-bit integers in more than a
// round (M 327, K 1408, N 16704, fp16: 33.6 -> 22.6 with the host; M 110, K 3200, N 24576, bf16: 37.2 -> 31.3).
//
// What bounds it: the sum of vector and matrix instructions, which two wavefronts a SIMD overlap in part, and the start and the
// end.  (Counters at 64 to 333 rows: of the busy cycles vector issue fills 41 to 48 % and the matrix pipes 26 to 38 %; without
// start and end 55 to 70 % and 35 to 50 %.)  Measured on this chip, a v_mfma_f32_16x16x32 takes 16 cycles of the
// matrix pipe and 8 of the issue port when other vector instructions want it; those take 4.3 each (two-operand
// logic, shifts and multiplies half of that).  A chunk (32 rows of a strip) costs 52 (fp16) to 68 (bf16) instructions
// to dequantise and a few for its scales, beside 4 MB matrix instructions.  K = 4096, N = 8192, 64 rows, bf16:
// 18.0 + 1.45 (MB - 2) us, of which about 6 are launch, first bytes and the sum over the ranges at the end.
// Calls on 4-bit integers that would else run in the decode kernel's blocks of rows (one group or groups of 128 * 2^i
// rows) feed the matrix cores the integers as that kernel does (kOneGroupRaw, kUnitGroupsRaw): 36 and 28
// instructions a chunk, and per unit of 128 rows 16 (fp16) or 36 (bf16) a row block for the fold.  The error against
// 64 bits is the output's own rounding (1.00 times it in fp16 and bf16; rounding each scaled weight: 1.28 times), and
//   M   64, K 4096, N 28672, bf16: 22.6 -> 21.7      M  200, K 4096, N 6144, fp16, zero points: 20.4 -> 17.6
//   M   80, K 4096, N 11008, bf16: 23.8 -> 18.4      M   17, K 2048, N 20032, bf16: 11.4 -> 10.0
// against scaled weights or the decode kernel.  But two sets of sums end at four row blocks, so that some calls lose the single
// round of tiles of five or six that scaled weights have (fp16, scaled -> now, and the decode kernel):
//   M   80, K 4096, N 28672: 27.9 -> 36.5, 45.0       M  144, K 4096, N 11008: 22.9 -> 27.9, 29.7
// Five and six row blocks on four wavefronts with 512 registers each took 30 and 33 us in the first call with M 80 and 96, and
// 1.5 times as long as eight wavefronts elsewhere.
// (Copies of activations by asm with a scalar base, the trees before and after in turn: the first two 22.8 -> 22.5 and 18.1 -> 17.9
// with the host, where two runs of one tree differ by up to 0.1.)
// Measured against the kernels it takes over from (us, before -> now):
//   M   64, K 4096, N 28672, bf16: 29.1 -> 21.7      M  200, K 4096, N 6144, fp16, zero points: 24.6 -> 17.6
//   M  333, K 2880, N  5760, bf16, groups of 32: 40.5 -> 21.7      M  512, K 4096, N 2048, bf16: 36 -> 20
//   M  128, K 2048, N 20032, MXFP4: 47.6 -> 20.5     M   96, K 2048, N 20032, 8-bit codes: 48 -> 18.5
// and with K split over workgroups, where there are fewer tiles than compute units:
//   M  101, K 2048, N 1536, bf16, zero points: 27.8 -> 10.6      M  125, K 6528, N 4672, bf16: 44.5 -> 20.8
//   M   76, K 9088, N 1920, MXFP4: 32.4 -> 14.5                  M   84, K 9088, N 2560, 8-bit codes: 32.5 -> 16.1
// Up to 16 rows of the formats that the decode kernel does not have take one row block and one strip a workgroup: eight
// ranges of K, so that 64 columns are enough to keep a compute unit busy (two strips: 4096 x 11008 18.6 us, one: 17.3).
//   M    8, K 4096, N 11008, fp8, bf16: 19.9 -> 14.8     M    8, K 2048, N 1536, 8-bit codes: 12.3 -> 7.2
//   M    8, K 8192, N  8192, fp8, bf16: 30.5 -> 21.0     M    8, K 4096, N 28672, NVFP4: 33.3 -> 23.4
// Tried without gain there: every workgroup starting its rows of K at another place (no channel conflicts to avoid).
// Tried and slower: one strip a workgroup with eight ranges (half the dequantisation per workgroup, but twice the
// activation bytes through the copy path per matrix instruction: 200 rows above 23 us, 64 rows on N = 28672 31 us).
//
// Pipeline, per K step of 64 rows of each of the four ranges: the activations (LDS, copied by
// LDS-DMA), two chunks of weights and the scales (registers) of step t + D - 1 are asked for during the
// second half of step t, one operation behind a matrix instruction, and waited for in the middle of step
// t + D - 2.  One barrier a step, in its middle: behind it stage t + 1 has landed for everyone and nobody
// reads stage t - 1 any more, whose slot the copies of the second half fill.  The operands of the next half are
// read behind the matrix instructions of their row block in this one, and each half dequantises the
// chunk of the half after it, a pair of weights behind each matrix instruction (its last instruction one
// matrix instruction later: the conversion to bf16 may not follow the multiply-adds at once).
#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "dequant.hpp"
#include "gemm_mid.hpp"
#include "moe_activation.hpp"

namespace sonar {
namespace {

constexpr int kMidWaves = 8;
constexpr int mid_strips(int mb) { return mb == 1 ? 1 : 2; }                 // strips of a workgroup (grouped: or four)
constexpr int mid_ranges(int strips) { return kMidWaves / strips; }          // ranges of K
constexpr int kMidStepK = 64;     // rows of K a step takes from each range

// Activation stages in LDS.
constexpr int mid_stages(int mb, bool deep) { return deep ? 5 : mb > 1 && mb <= 4 ? 4 : 3; }
// Wavefronts a SIMD: two (one workgroup a compute unit), or four for a single row block with more workgroups than
// compute units, `deep` without: its loop is so short that the bytes under way have to come from two workgroups or
// a longer ring.  That ring pays from six steps a range on: K = 4096, N = 11008, fp8 (8 steps) 16.3 -> 14.8 us, K = 3072,
// N = 16384 (6) 16.3 -> 15.6, but K = 2048, N = 8192 (4) 9.6 -> 10.2, K = 1024, N = 1024 (2) 5.1 -> 6.1.
constexpr int kMidDeepSteps = 6;
constexpr int mid_waves_per_simd(int mb, bool deep) { return mb == 1 && !deep ? 4 : 2; }
constexpr int mid_stage_bytes(int mb, int strips) { return mid_ranges(strips) * mb * 2048; }
constexpr int mid_sum_rows(int mb) { return mb < 4 ? mb : 4; }   // row blocks summed at a time at the end
constexpr int mid_lds(int mb, bool deep, int strips) {
  const int stages = mid_stages(mb, deep) * mid_stage_bytes(mb, strips), sum = kMidWaves * mid_sum_rows(mb) * 4096;
  return stages > sum ? stages : sum;
}

// How the scales come: one group, groups of 64 * 2^i rows (a scale row a step), or groups of 32 rows or less (a
// scale row a chunk; NVFP4: two groups a chunk).  The last two are forms for 4-bit integers (MidParams::raw_codes): the
// codes go to the matrix cores as integers, and the scale of one group or of groups of 128 * 2^i rows (a scale row a
// unit of two steps) into the fp32 sums.
enum MidGroups { kOneGroup = 0, kStepGroups = 1, kChunkGroups = 2, kOneGroupRaw = 3, kUnitGroupsRaw = 4 };

template <typename T, int FMT>
struct MidDequant {
  static constexpr bool kF4 = FMT == kMidMxFp4 || FMT == kMidNvFp4;
  static constexpr bool k8 = FMT == kMidInt8 || FMT == kMidFp8;
  typedef typename Dq4Of<T, kF4, FMT == kMidNvFp4>::type D4;
  typedef typename Dq8Of<T, FMT == kMidFp8>::type D8;
  typedef typename std::conditional<k8, typename D8::Col, typename D4::Col>::type Col;
};

template <typename T, int FMT, int GROUPS, int MB, bool DEEP, bool GROUPED = false, int STRIPS = mid_strips(MB)>
__global__ __launch_bounds__(kMidWaves * 64) __attribute__((amdgpu_waves_per_eu(mid_waves_per_simd(MB, DEEP), mid_waves_per_simd(MB, DEEP)))) void marlin_mid_gemm(
    const typename std::conditional<GROUPED, MidMoeParams, MidParams>::type p) {
  MidMoe moe = {};
  if constexpr (GROUPED) moe = p.moe;
  typedef MidDequant<T, FMT> Fmt;
  typedef typename Fmt::D4 D4;
  typedef typename Fmt::D8 D8;
  typedef typename Fmt::Col Col;
  typedef typename Dq<T>::vec8 vec8;
  constexpr bool kZero = FMT == kMidInt4Zp;
  // 8-bit codes go to the matrix cores as they are, which halves their instructions, and their scales into the fp32
  // sums: at the end with one group; else group by group (`raw` to `acc`), which pays for a single row block only
  // and has the operands of the matrix instruction the other way round, so that a lane's sums share a column.
  // (K = 4096, N = 4096, 8 rows, fp8, one group / MXFP8: 10.6 -> 10.2 / 11.0 -> 10.6 us; K = 12288, N = 2560: 14.4 -> 14.0.)
  constexpr bool kRaw = Fmt::k8 && std::is_same<T, __bf16>::value && (GROUPS == kOneGroup || MB == 1);
  constexpr bool kFold = kRaw && GROUPS != kOneGroup;
  // 4-bit integers that way: v - z in fp16 (nine instructions a word instead of 13), in bf16 128 + v (7 instead of 17), whose
  // surplus (128 + z) * sum(a) comes off with the sum of the activations, one more matrix instruction with an operand of
  // ones per row block and chunk.  The sums of a unit of 128 rows (`unit_sum`) are folded into `acc` behind the matrix instructions
  // of the row block after them; with one group and fp16 nothing is folded and the scale waits for the end.  Both sets of
  // sums are 16 registers a row block: with four the largest form has 256.
  constexpr bool kBf16 = std::is_same<T, __bf16>::value;
  constexpr bool kCodes = GROUPS == kOneGroupRaw || GROUPS == kUnitGroupsRaw;
  constexpr bool kUnits = GROUPS == kUnitGroupsRaw || (GROUPS == kOneGroupRaw && kBf16);
  constexpr bool kSwap = kFold || kCodes;            // activations are the row operand: a lane's sums share a column
  constexpr bool kNoScales = GROUPS == kOneGroup || kCodes;   // none among the memory operations of every step
  constexpr int D = mid_stages(MB, DEEP);
  constexpr int W = D - 1;                           // ring of the packed codes and scales in registers
  constexpr int kStage = mid_stage_bytes(MB, STRIPS);
  constexpr int kMidStrips = STRIPS, kMidRanges = mid_ranges(STRIPS);
  // 8-row copies of activations per wavefront and step (three row blocks and four strips: the last wavefront's are copies 5 again)
  constexpr int kCopies = (2 * MB + kMidStrips - 1) / kMidStrips;
  constexpr bool kEvenCopies = kCopies * kMidStrips == 2 * MB;
  constexpr int kLoads = Fmt::k8 ? 4 : 2;            // 16-byte loads of packed codes per lane and step
  constexpr int kScaleRows = GROUPS == kChunkGroups ? 2 : 1;
  // memory operations per wavefront and step
  constexpr int kOps = kCopies + kLoads + (kNoScales ? 0 : kScaleRows * (kZero ? 2 : 1));
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col16 = lane & 15, kb = lane >> 4;
  const int range = wave / kMidStrips, strip_of = wave % kMidStrips;
  const uint32_t magic = magic_register(kCodes ? RawOperand<T>::kMagic : 0x64006400u);

  // Workgroup ids congruent mod 8 run on one XCD: each XCD takes a contiguous run of tiles, the row tiles
  // of a pair of strips next to each other, so the second to ask for a chunk finds it in that L2.
  // (Grouped: of the blocks that the routing has made, one after the other, so that those of an expert share its chunks.)
  const int strips = p.size_n / kStripN;
  const int tiles_m = GROUPED ? min(p.tiles_m, moe.num_post_pad[0] / moe.block_size) : p.tiles_m;
  constexpr int kOfHalf = kMidStrips > 1 ? kMidStrips / 2 : 1;
  const bool halves = GROUPED && moe.gated != nullptr && moe.gated_halves;
  const int across = halves ? strips / 2 : strips, each = halves ? kOfHalf : kMidStrips;
  const int tiles = GROUPED ? tiles_m * ((across + each - 1) / each) : p.tiles;
  const int units = tiles * p.splits, per_xcd = (units + 7) / 8;
  const int unit = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || unit >= units) return;
  const int split = unit / tiles, tile = unit - split * tiles;
  const int tile_n = tile / tiles_m, tile_m = tile - tile_n * tiles_m;
  const int m0 = tile_m * 16 * MB;
  const int expert = GROUPED ? moe.expert_ids[tile_m] : 0;
  if (GROUPED && (unsigned)expert >= (unsigned)moe.num_experts) return;
  // (the second strip of an odd last pair is the first again, and not stored)
  // (halves: the first strips are of the gate half, the others the same columns of the up half)
  const int of_tile = halves ? strip_of % kOfHalf : strip_of;
  const bool active = tile_n * each + of_tile < across;
  const int strip = __builtin_amdgcn_readfirstlane((active ? tile_n * each + of_tile : across - 1) + (halves ? strip_of / kOfHalf * across : 0));

  const int first = split * p.split_steps;   // of the steps this workgroup takes
  const int steps = min(first + p.split_steps, p.size_k / kMidStepK);
  int per_range = (steps - first + kMidRanges - 1) / kMidRanges;
  if constexpr (kUnits) per_range = (per_range + 1) & ~1;   // whole units: the host has seen to it that `first` and `steps` are even
  const int k_first = first + range * per_range;

  // ---- sources.  The activations of a range are copied by its own wavefronts, kCopies copies each of 8 rows x
  // one 128-byte line; piece q of row r sits at 16-byte slot q ^ r of the row, off the other rows' banks.
  uint32_t a_off[kCopies];
#pragma unroll
  for (int i = 0; i < kCopies; ++i) {
    int row = m0 + 8 * (kEvenCopies ? strip_of * kCopies + i : min(strip_of * kCopies + i, 2 * MB - 1)) + (lane >> 3);
    if constexpr (GROUPED) {   // (padding slots read row 0 and are not stored)
      const int id = row < moe.sorted_len ? moe.sorted_ids[row] : moe.rows_total;
      row = (unsigned)id < (unsigned)moe.rows_total ? (moe.a_by_slot ? row : id / moe.top_k) : 0;
    } else if (row >= p.size_m) {
      row = p.size_m - 1;   // rows past M are computed and never stored
    }
    a_off[i] = (uint32_t)row * (uint32_t)(p.lda * 2) + 16 * ((lane & 7) ^ (lane >> 3));
  }
  const uint16_t* scales = p.scales + (GROUPED ? expert * moe.expert_s_stride : 0) + (size_t)strip * kStripN;
  const uint32_t* zeros = p.zeros + (GROUPED ? expert * moe.expert_z_stride : 0) + (size_t)strip * (kStripN / 8);
  const char* b_base = reinterpret_cast<const char*>(p.b + (GROUPED ? expert * moe.expert_b_stride : 0)) +
                       (size_t)strip * p.chunks_per_strip * (Fmt::k8 ? 2048 : 1024);
  const uint32_t b_off = 16 * lane;
  const char* s_base = reinterpret_cast<const char*>(scales);
  const uint32_t s_off = 16 * (col16 & 7) + (FMT == kMidNvFp4 ? (kb >> 1) * (uint32_t)p.size_n * 2 : 0);
  const char* z_base = reinterpret_cast<const char*>(zeros);
  const uint32_t z_off = 4 * (col16 & 7);
  char* a_stage = smem + range * (MB * 2048);
  const uint32_t a_lds = (uint32_t)(uintptr_t)(lds_void_t*)a_stage;

  u32x4_t wq[W][kLoads];
  u32x4_t sv[W][kScaleRows];
  uint32_t zv[W][kScaleRows];
  u32x4_t unit_sv;    // kUnitGroupsRaw: scales and zero points of a unit, asked for two steps before they are used
  uint32_t unit_zv;

  // Memory operation `op` (0..kOps-1) of step k: first the codes and scales into ring position R, then the
  // activations into LDS slot `slot`.
  auto issue_one = [&](const int R, const int slot, const int k, const int op) __attribute__((always_inline)) {
    if (op < kLoads) {
      const char* b_src = b_base + (size_t)k * (kLoads * 1024);
      asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "=&v"(wq[R][op]) : "v"(b_off), "s"(b_src), "i"(op * 1024) : "memory");
    } else if (op < kOps - kCopies) {
      const int h = (op - kLoads) / (kZero ? 2 : 1);
      const int g = GROUPS == kStepGroups ? k >> p.group_shift : (FMT == kMidNvFp4 ? 2 : 1) * (2 * k + h);
      if (!kZero || (op - kLoads) % 2 == 0) {
        const char* s_src = s_base + (size_t)g * p.size_n * 2;
        asm volatile("global_load_dwordx4 %0, %1, %2" : "=&v"(sv[R][h]) : "v"(s_off), "s"(s_src) : "memory");
      } else {
        const char* z_src = z_base + (size_t)g * (p.size_n / 2);
        asm volatile("global_load_dword %0, %1, %2" : "=&v"(zv[R][h]) : "v"(z_off), "s"(z_src) : "memory");
      }
    } else {
      const int i = op - (kOps - kCopies);
      const char* a_src = reinterpret_cast<const char*>(p.a) + (size_t)k * (kMidStepK * 2);
      // (not one call with a chosen index: that costs every copy an instruction more)
      if constexpr (kEvenCopies) copy_to_lds<16>(a_lds + slot * kStage + (strip_of * kCopies + i) * 1024, a_off[i], a_src);
      else copy_to_lds<16>(a_lds + slot * kStage + min(strip_of * kCopies + i, 2 * MB - 1) * 1024, a_off[i], a_src);
    }
  };
  // Scales of the unit of step `k`, behind whose first half they are taken from the registers, and zero points, which fp16
  // needs for the unit after it.  Older than the other operations of their step.
  auto issue_unit = [&](const int k) __attribute__((always_inline)) {
    const int g = min(k, steps - 1) >> p.group_shift, gz = kBf16 ? g : min(k + 1, steps - 1) >> p.group_shift;
    const char* s_src = s_base + (size_t)g * p.size_n * 2;
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=&v"(unit_sv) : "v"(s_off), "s"(s_src) : "memory");
    if constexpr (kZero) {
      const char* z_src = z_base + (size_t)gz * (p.size_n / 2);
      asm volatile("global_load_dword %0, %1, %2" : "=&v"(unit_zv) : "v"(z_off), "s"(z_src) : "memory");
    }
  };
  auto unit_landed = [&]() __attribute__((always_inline)) {
    asm volatile("" : "+v"(unit_sv));
    if constexpr (kZero) asm volatile("" : "+v"(unit_zv));
  };
  // until only the `n` youngest operations are outstanding; the registers of ring position R are in its hands
  auto landed = [&](const int R, const int n) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(n) : "memory");
#pragma unroll
    for (int i = 0; i < kLoads; ++i) asm volatile("" : "+v"(wq[R][i]));
    if constexpr (!kNoScales) {
#pragma unroll
      for (int h = 0; h < kScaleRows; ++h) {
        asm volatile("" : "+v"(sv[R][h]));
        if constexpr (kZero) asm volatile("" : "+v"(zv[R][h]));
      }
    }
  };

  Col cols[4];
  float fold_scale[2][4];   // kFold: of the chunk or step that is multiplied and the one after it
  auto set_col = [&](int j, uint16_t scale_bits, uint32_t zero_word) __attribute__((always_inline)) {
    int z = 8;
    if (kZero) z = (int)((zero_word >> (4 * (j + 4 * (col16 >> 3)))) & 0xFu);   // zero_point_shift(16 j + col16)
    if constexpr (Fmt::k8) cols[j] = D8::make_col(scale_bits);
    else cols[j] = D4::make_col(scale_bits, z);
  };
  float unit_scale[4], unit_zero[4];   // kCodes: of the unit whose sums are folded next; bf16: z + 128 below zero
  uint32_t next_zeros = 0;             // kUnitGroupsRaw in fp16: of the unit after it
  auto zero_point = [&](int j, uint32_t word) __attribute__((always_inline)) {   // zero_point_shift(16 j + col16)
    return (int)((word >> (4 * (j + 4 * (col16 >> 3)))) & 0xFu);
  };
  auto take_unit = [&](int j) __attribute__((always_inline)) {
    const uint32_t word = j == 0 ? unit_sv.x : j == 1 ? unit_sv.y : j == 2 ? unit_sv.z : unit_sv.w;
    unit_scale[j] = Dq<T>::to_float((uint16_t)((col16 & 8) ? word >> 16 : word));   // the slots of make_col
    if constexpr (kZero && kBf16) unit_zero[j] = -RawOperand<T>::kBase - (float)zero_point(j, unit_zv);
    if constexpr (kZero && !kBf16)
      if (j == 3) asm volatile("v_mov_b32 %0, %1" : "=v"(next_zeros) : "v"(unit_zv));   // (a register of its own: unit_zv is loaded again)
  };
  // the constants of column block j from ring position R (chunk h of the step)
  auto make_col = [&](const int R, const int h, const int j) __attribute__((always_inline)) {
    if constexpr (!kNoScales) {
      const u32x4_t& v = sv[R][GROUPS == kChunkGroups ? h : 0];
      const uint32_t word = j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w;
      // column 16 j + col16 is slot 2 j + col16 / 8 of the lane's eight
      const uint32_t bits = (col16 & 8) ? word >> 16 : word & 0xFFFFu;
      if constexpr (kFold) fold_scale[GROUPS == kChunkGroups ? h : R % 2][j] = Raw8<FMT == kMidFp8>::column_scale((uint16_t)bits);
      else set_col(j, (uint16_t)bits, kZero ? zv[R][GROUPS == kChunkGroups ? h : 0] : 0);
    }
  };
  if constexpr (GROUPS == kOneGroup && !kRaw) {
    uint32_t zword = 0;
    if (kZero) zword = zeros[col16 & 7];
#pragma unroll
    for (int j = 0; j < 4; ++j) set_col(j, scales[scale_slot(16 * j + col16, false)], zword);
  }

  uint16_t one_scale[4];   // kOneGroupRaw: as they were loaded, used when the first step has landed or later
  uint32_t one_zeros = 0;
  if constexpr (GROUPS == kOneGroupRaw) {
#pragma unroll
    for (int j = 0; j < 4; ++j) one_scale[j] = scales[scale_slot(16 * j + col16, false)];
    if (kZero) one_zeros = zeros[col16 & 7];
  }

  u32x4_t av[MB];
  uint32_t wv[2][4][4];    // dequantised chunk of either half: four operand blocks of 16 columns
  floatx4_t acc[4][MB];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < MB; ++i) acc[j][i] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  floatx4_t raw[4];
  floatx4_t unit_sum[kUnits ? 4 : 1][kUnits ? MB : 1], a_sum[kUnits ? MB : 1];   // of codes times activations, of activations
  u32x4_t ones = u32x4_t{RawOperand<T>::kOnes, RawOperand<T>::kOnes, RawOperand<T>::kOnes, RawOperand<T>::kOnes};
  if constexpr (kCodes && kBf16) asm("" : "+v"(ones));

  // Piece `q` (0..15) of dequantising chunk h of ring position R into wv[h].  A pair of 4-bit integer codes is
  // finished by the piece after it (q = 16 finishes the last).
  typename Dq<T>::Mid mid;
  // (`odd`: the chunk's step is the second of its unit)
  auto piece = [&](const int R, const int h, const bool odd, const int q) __attribute__((always_inline)) {
    const int j = q >> 2, part = q & 3;
    if constexpr (kCodes) {
      if (q == 16) return;
      const u32x4_t& v = wq[R][h];
      const uint32_t word = j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w;
      if constexpr (GROUPS == kUnitGroupsRaw)
        if (part == 0 && odd && h == 1) take_unit(j);
      if constexpr (kBf16) {
        wv[h][j][part] = and_or(part ? word >> (4 * part) : word, 0x000f000fu, magic);
      } else {
        if constexpr (GROUPS == kUnitGroupsRaw && kZero)
          if (part == 0 && !odd && h == 0) cols[j] = D4::make_col(0, zero_point(j, next_zeros));
        wv[h][j][part] = __builtin_bit_cast(uint32_t, D4::stage2(D4::stage1(part < 2 ? word : word >> 8, part, magic), cols[j], part));
      }
      return;
    }
    if constexpr (!Fmt::k8 && !Fmt::kF4) {
      if (q > 0) wv[h][(q - 1) >> 2][(q - 1) & 3] = D4::stage3(mid, cols[(q - 1) >> 2]);
    }
    if (q == 16) return;
    if (part == 0 && (GROUPS == kChunkGroups || h == 0)) make_col(R, h, j);
    if constexpr (Fmt::k8) {
      if (part & 1) return;
      const u32x4_t& v = wq[R][2 * h + (part >> 1)];   // the low, then the high four of a lane's eight rows
      const uint32_t word = j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w;
      uint2 w;
      if constexpr (kRaw) w = Raw8<FMT == kMidFp8>::word4(word);
      else w = D8::word4(word, cols[j], magic);
      wv[h][j][part] = w.x;
      wv[h][j][part + 1] = w.y;
    } else {
      const u32x4_t& v = wq[R][h];
      const uint32_t word = j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w;
      if constexpr (Fmt::kF4) {
        if (part != 0) return;
        const u32x4_t w = __builtin_bit_cast(u32x4_t, D4::word(word, cols[j], magic));
        wv[h][j][0] = w.x, wv[h][j][1] = w.y, wv[h][j][2] = w.z, wv[h][j][3] = w.w;
      } else {
        mid = D4::stage2(D4::stage1(part < 2 ? word : word >> 8, part, magic), cols[j], part);
      }
    }
  };
  // operand lane (kb, col16) of row block 0, chunk h: piece 4 h + kb of row col16
  uint32_t a_at[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    a_at[h] = a_lds + (col16 >> 3) * 1024 + (col16 & 7) * 128 + (((4 * h + kb) ^ (col16 & 7)) * 16);
#define SONAR_MID_READ(dst, base, off) \
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(dst) : "v"(base), "i"(off) : "memory")
  // One half of a step: 4 MB matrix instructions on chunk H of the step in ring position R, LDS slot `slot`.
  // Behind each, a share of the next half's dequantisation and (H = 1) of the memory operations of step `k_copy`;
  // behind a row block's four, the read of its operand of the next half.
  auto fold = [&](const int R, const int H, const int j) __attribute__((always_inline)) {
    const float s = fold_scale[GROUPS == kChunkGroups ? H : R % 2][j];
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[j][0][r] = __builtin_fmaf(raw[j][r], s, acc[j][0][r]);
  };
  // the sums of row block i, column block j of a unit
  float surplus[4];
  auto fold_unit = [&](const int i, const int j) __attribute__((always_inline)) {
    if constexpr (kUnits) {
      if constexpr (kBf16 && !kZero) {
        if (j == 0) {
#pragma unroll
          for (int r = 0; r < 4; ++r) surplus[r] = (RawOperand<T>::kBase + 8.f) * a_sum[i][r];
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float x = unit_sum[j][i][r];
        if constexpr (kBf16 && kZero) x = __builtin_fmaf(unit_zero[j], a_sum[i][r], x);
        else if constexpr (kBf16) x -= surplus[r];
        if constexpr (GROUPS == kUnitGroupsRaw) acc[j][i][r] = __builtin_fmaf(x, unit_scale[j], acc[j][i][r]);
        else acc[j][i][r] += x;
      }
    }
  };
  // (`odd`: the second step of a unit)
  auto half_step = [&](const int R, const int H, const bool odd, const int slot, const int next_slot, const int fill,
                       const int k_copy, const int k_unit) __attribute__((always_inline)) {
    const int NR = H ? (R + 1) % W : R, NH = H ^ 1;
    const bool next_odd = odd != (H == 1), begins = !odd && H == 0, ends = odd && H == 1;   // of the unit
    const uint32_t a_next = a_at[NH] + (H ? next_slot : slot) * kStage;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      // the operands of this half are the oldest reads, MB are outstanding at every row block
      asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(av[i]) : "i"(MB - 1) : "memory");
      if constexpr (kUnits && kBf16)
        a_sum[i] = Dq<T>::mfma(__builtin_bit_cast(vec8, av[i]), __builtin_bit_cast(vec8, ones),
                               begins ? floatx4_t{0.f, 0.f, 0.f, 0.f} : a_sum[i]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const vec8 w = __builtin_bit_cast(vec8, u32x4_t{wv[H][j][0], wv[H][j][1], wv[H][j][2], wv[H][j][3]});
        if constexpr (kUnits)
          unit_sum[j][i] = Dq<T>::mfma(__builtin_bit_cast(vec8, av[i]), w,
                                       begins ? floatx4_t{0.f, 0.f, 0.f, 0.f} : unit_sum[j][i]);
        else if constexpr (kCodes)
          acc[j][i] = Dq<T>::mfma(__builtin_bit_cast(vec8, av[i]), w, acc[j][i]);
        else if constexpr (kFold)
          raw[j] = Dq<T>::mfma(__builtin_bit_cast(vec8, av[i]), w,
                               GROUPS == kChunkGroups || H == 0 ? floatx4_t{0.f, 0.f, 0.f, 0.f} : raw[j]);
        else
          acc[j][i] = Dq<T>::mfma(w, __builtin_bit_cast(vec8, av[i]), acc[j][i]);
        const int at = 4 * i + j;
        if (kFold && j > 0 && (GROUPS == kChunkGroups || H == 1)) fold(R, H, j - 1);   // (one matrix instruction later)
        if (kUnits && ends && i > 0) fold_unit(i - 1, j);
#pragma unroll
        for (int q = 0; q < 16; ++q)
          if (q >= 16 * at / (4 * MB) && q < 16 * (at + 1) / (4 * MB)) piece(NR, NH, next_odd, q);
        if constexpr (GROUPS == kUnitGroupsRaw)
          if (ends && at == 0) issue_unit(k_unit);
        if (H) {
#pragma unroll
          for (int o = 0; o < kOps; ++o)
            if (o >= kOps * at / (4 * MB) && o < kOps * (at + 1) / (4 * MB)) issue_one(R, fill, k_copy, o);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      SONAR_MID_READ(av[i], a_next, i * 2048);
      __builtin_amdgcn_sched_barrier(0);
    }
    piece(NR, NH, next_odd, 16);
    if (kUnits && ends) {
#pragma unroll
      for (int j = 0; j < 4; ++j) fold_unit(MB - 1, j);
    }
    if (kFold && (GROUPS == kChunkGroups || H == 1)) fold(R, H, 3);
  };

  // ---- prologue: D - 1 steps asked for, the first one here
  if constexpr (GROUPS == kUnitGroupsRaw) {
    if constexpr (kZero && !kBf16) {   // (the zero points of the first unit)
      const char* z_src = z_base + (size_t)(min(k_first, steps - 1) >> p.group_shift) * (p.size_n / 2);
      asm volatile("global_load_dword %0, %1, %2" : "=&v"(next_zeros) : "v"(z_off), "s"(z_src) : "memory");
    }
    issue_unit(k_first + 1);
  }
#pragma unroll
  for (int r = 0; r < W; ++r)
#pragma unroll
    for (int o = 0; o < kOps; ++o) issue_one(r, r, min(k_first + r, steps - 1), o);
  landed(0, (W - 1) * kOps);
  if constexpr (GROUPS == kUnitGroupsRaw) {
    unit_landed();
    asm volatile("" : "+v"(next_zeros));
  }
  if constexpr (kCodes && !kBf16 && !(GROUPS == kUnitGroupsRaw && kZero)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) cols[j] = D4::make_col(0, kZero ? zero_point(j, one_zeros) : 8);
  }
  if constexpr (GROUPS == kOneGroupRaw && kBf16 && kZero) {
#pragma unroll
    for (int j = 0; j < 4; ++j) unit_zero[j] = -RawOperand<T>::kBase - (float)zero_point(j, one_zeros);
  }
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < MB; ++i) SONAR_MID_READ(av[i], a_at[0], i * 2048);
#pragma unroll
  for (int q = 0; q <= 16; ++q) piece(0, 0, false, q);

  int slot = 0, fill = W;   // LDS slot of step t, and the one step t + D - 1 goes to
  auto step = [&](const int R, const bool odd, int t) __attribute__((always_inline)) {
    const bool live = k_first + t < steps;   // uniform; past the end of K only the copies are left to do
    const int next_slot = slot == D - 1 ? 0 : slot + 1;
    const int k_copy = min(k_first + t + W, steps - 1);
    if (live) half_step(R, 0, odd, slot, next_slot, 0, 0, 0);
    landed((R + 1) % W, (W - 2) * kOps);
    if constexpr (GROUPS == kUnitGroupsRaw)
      if (!odd) unit_landed();
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (live) {
      half_step(R, 1, odd, slot, next_slot, fill, k_copy, k_first + t + 2);
    } else {
      if constexpr (GROUPS == kUnitGroupsRaw)
        if (odd) issue_unit(k_first + t + 2);
#pragma unroll
      for (int o = 0; o < kOps; ++o) issue_one(R, fill, k_copy, o);
    }
    slot = next_slot;
    fill = fill == D - 1 ? 0 : fill + 1;
  };
  if constexpr (kUnits) {   // units of two steps through a ring of three
    static_assert(W == 3);
    for (int t = 0; t < per_range; t += 6) {
      step(0, false, t);
      step(1, true, t + 1);
      if (t + 2 < per_range) {
        step(2, false, t + 2);
        step(0, true, t + 3);
      }
      if (t + 4 < per_range) {
        step(1, false, t + 4);
        step(2, true, t + 5);
      }
    }
  } else {
    for (int t = 0; t < per_range; t += W) {
      step(0, false, t);
      if (t + 1 < per_range) step(1, false, t + 1);
      if constexpr (W > 2)
        if (t + 2 < per_range) step(2, false, t + 2);
      if constexpr (W > 3)
        if (t + 3 < per_range) step(3, false, t + 3);
    }
  }
  // copies and reads still under way must not outlive this point: LDS is used for the sums from here on
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < MB; ++i) asm volatile("" : "+v"(av[i]));
#pragma unroll
  for (int r = 0; r < W; ++r) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) asm volatile("" : "+v"(wq[r][i]));
    if constexpr (!kNoScales) {
#pragma unroll
      for (int h = 0; h < kScaleRows; ++h) {
        asm volatile("" : "+v"(sv[r][h]));
        if constexpr (kZero) asm volatile("" : "+v"(zv[r][h]));
      }
    }
  }
#undef SONAR_MID_READ
  if constexpr (GROUPS == kUnitGroupsRaw) unit_landed();
  __builtin_amdgcn_s_barrier();
  if constexpr (GROUPS == kOneGroupRaw) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[j][i][r] *= Dq<T>::to_float(one_scale[j]);
  }

  // ---- the ranges meet in LDS, mid_sum_rows(MB) row blocks at a time; a wavefront adds its share (a quarter of four ranges) of
  // its strip's accumulator tiles, in the order of the ranges
  constexpr int kSum = mid_sum_rows(MB);
  float4* sums = reinterpret_cast<float4*>(smem);
  const float gs = FMT == kMidNvFp4 && p.global_scale ? p.global_scale[0] : 1.f;
  // Row and first of four columns of a tile that a lane adds.  With kSwap a lane holds rows 4 kb .. + 3 of column col16 and
  // stores them so that four columns of a row lie together; rows change places between the kb, off each other's banks.
  const int tile_row = kSwap ? 4 * kb + ((col16 >> 2) ^ kb) : col16, tile_col = 4 * (kSwap ? lane & 3 : kb);
  // The gated activation of a column of the gate half and the same of the up half, rounded as the results would be: the wavefronts of a
  // pair of strips share its tiles.  (Against a launch of 5 to 8 us that reads and writes C: 185 layers 2.5 % less time, 32 experts of
  // 42 rows, 1152 x 7680 207 -> 202 us, 8 of 52, 2560 x 3968 80.6 -> 77.6.)
  auto finish_halves = [&](const int round) __attribute__((always_inline)) {
    const int worker = 2 * range + strip_of / kOfHalf, first_tile = tile_n * kOfHalf + of_tile;
    if (!active) return;
    for (int q = worker; q < 4 * kSum; q += 2 * kMidRanges) {
      const int i = round + (q >> 2), j = q & 3;
      const int slot = m0 + 16 * i + tile_row;
      int row = i < MB && slot < moe.sorted_len ? moe.sorted_ids[slot] : moe.rows_total;
      if ((unsigned)row >= (unsigned)moe.rows_total) continue;   // padding slot
      const float row_w = moe.mul_topk ? Dq<T>::to_float(Dq<T>::from_float(moe.topk_weights[row])) : 1.f;
      const int nl = 16 * j + tile_col;
      uint16_t n[2][4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        floatx4_t v = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int g = 0; g < kMidRanges; ++g) {
          const float4 s = sums[(((kMidStrips * g + h * kOfHalf + of_tile) * kSum + (q >> 2)) * 4 + j) * 64 + lane];
          v += floatx4_t{s.x, s.y, s.z, s.w};
        }
        const uint16_t* bias_row = p.bias ? p.bias + expert * moe.expert_bias_stride + (first_tile + h * across) * kStripN : nullptr;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          n[h][r] = Dq<T>::from_float(v[r] + (bias_row ? Dq<T>::to_float(bias_row[scale_slot(nl + r, false)]) : 0.f));
          if (moe.mul_topk) n[h][r] = Dq<T>::from_float(Dq<T>::to_float(n[h][r]) * row_w);
        }
      }
      uint16_t o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = silu_times<T>(n[0][r], n[1][r]);
      *reinterpret_cast<uint2*>(moe.gated + (size_t)row * (p.size_n / 2) + first_tile * kStripN + nl) =
          make_uint2((uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16));
    }
  };
#pragma unroll
  for (int round = 0; round < MB; round += kSum) {
    if (round > 0) __syncthreads();
#pragma unroll
    for (int i = 0; i < kSum; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (round + i < MB) {
          const floatx4_t v = acc[j][round + i < MB ? round + i : 0];
          const int at = ((wave * kSum + i) * 4 + j) * 64;
          if constexpr (kSwap) {
#pragma unroll
            for (int r = 0; r < 4; ++r) reinterpret_cast<float*>(sums)[4 * at + 64 * kb + 16 * (r ^ kb) + col16] = v[r];
          } else {
            sums[at + lane] = make_float4(v.x, v.y, v.z, v.w);
          }
        }
    __syncthreads();
    if constexpr (GROUPED) {
      if (halves) {
        finish_halves(round);
        continue;
      }
    }
#pragma unroll
    for (int u = 0; u < (kMidRanges == 2 ? 2 * kSum : kSum); ++u) {
      constexpr int kEach = kSum * 4 / kMidRanges;   // accumulator tiles a wavefront adds
      if (kEach > 0 ? u >= kEach : range >= 4 * kSum) continue;
      const int q = kEach > 0 ? range * kEach + u : range;
      const int i = round + (q >> 2), j = q & 3;
      int row = m0 + 16 * i + tile_row;
      if (i >= MB || !active) continue;
      float row_w = 1.f;
      if constexpr (GROUPED) {
        row = row < moe.sorted_len ? moe.sorted_ids[row] : moe.rows_total;
        if ((unsigned)row >= (unsigned)moe.rows_total) row = moe.rows_total;   // padding slot
        // the routing weight is rounded to the activation type and the product is formed and rounded in that type
        // (marlin_template.h(moe):1893-1897)
        if (moe.mul_topk && row < moe.rows_total) row_w = Dq<T>::to_float(Dq<T>::from_float(moe.topk_weights[row]));
      }
      floatx4_t v = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int g = 0; g < kMidRanges; ++g) {
        const float4 s = sums[(((kMidStrips * g + strip_of) * kSum + (q >> 2)) * 4 + j) * 64 + lane];
        v += floatx4_t{s.x, s.y, s.z, s.w};
      }
      if (row >= (GROUPED ? moe.rows_total : p.size_m)) continue;
      const int nl = 16 * j + tile_col;
      if constexpr (kRaw && !kFold) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] *= Raw8<FMT == kMidFp8>::column_scale(scales[scale_slot(nl + r, false)]);
      }
      if (!GROUPED && p.splits > 1) {
        p.partial[(((size_t)split * p.size_m + row) * p.size_n + strip * kStripN + nl) / 4] = make_float4(v.x, v.y, v.z, v.w);
        continue;
      }
      if (FMT == kMidNvFp4) v = v * gs;
      float bias[4] = {0.f, 0.f, 0.f, 0.f};
      if (p.bias) {
        const uint16_t* bias_row = p.bias + (GROUPED ? expert * moe.expert_bias_stride : 0) + strip * kStripN;
#pragma unroll
        for (int r = 0; r < 4; ++r) bias[r] = Dq<T>::to_float(bias_row[scale_slot(nl + r, false)]);
      }
      uint16_t n[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        n[r] = Dq<T>::from_float(v[r] + bias[r]);
        if (GROUPED && moe.mul_topk) n[r] = Dq<T>::from_float(Dq<T>::to_float(n[r]) * row_w);
      }
      if constexpr (GROUPED) {
        if (moe.gated != nullptr) {
          *reinterpret_cast<uint32_t*>(moe.gated + (size_t)row * (p.size_n / 2) + (strip * kStripN + nl) / 2) =
              (uint32_t)swiglu_oai<T>(n[0], n[1], moe.gated_limit, moe.gated_alpha) |
              ((uint32_t)swiglu_oai<T>(n[2], n[3], moe.gated_limit, moe.gated_alpha) << 16);
          continue;
        }
      }
      const uint2 o = make_uint2((uint32_t)n[0] | ((uint32_t)n[1] << 16), (uint32_t)n[2] | ((uint32_t)n[3] << 16));
      *reinterpret_cast<uint2*>(p.c + (size_t)row * p.size_n + strip * kStripN + nl) = o;
    }
  }
}

// Adds the totals of up to kMost K splits, four columns a thread, in the order of K.  (All loads are asked for before the
// first is waited for: one after the other, seven splits took 5 us longer than two.)
template <typename T, int kMost>
__global__ __launch_bounds__(256) void marlin_mid_sum(const MidParams p) {
  const size_t quads = (size_t)p.size_m * p.size_n / 4;
  const float gs = p.global_scale ? p.global_scale[0] : 1.f;
  for (size_t q = (size_t)blockIdx.x * 256 + threadIdx.x; q < quads; q += (size_t)gridDim.x * 256) {
    float4 w[kMost];
#pragma unroll
    for (int s = 0; s < kMost; ++s) w[s] = p.partial[(s < p.splits ? s : 0) * quads + q];
    float4 v = w[0];
#pragma unroll
    for (int s = 1; s < kMost; ++s)
      if (s < p.splits) v.x += w[s].x, v.y += w[s].y, v.z += w[s].z, v.w += w[s].w;
    const int col = (int)(4 * q % p.size_n), nl = col & (kStripN - 1);
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (p.bias) {
#pragma unroll
      for (int r = 0; r < 4; ++r) bias[r] = Dq<T>::to_float(p.bias[col - nl + scale_slot(nl + r, false)]);
    }
    uint2 o;
    o.x = (uint32_t)Dq<T>::from_float(v.x * gs + bias[0]) | ((uint32_t)Dq<T>::from_float(v.y * gs + bias[1]) << 16);
    o.y = (uint32_t)Dq<T>::from_float(v.z * gs + bias[2]) | ((uint32_t)Dq<T>::from_float(v.w * gs + bias[3]) << 16);
    reinterpret_cast<uint2*>(p.c)[q] = o;
  }
}

template <typename T, int FMT, int GROUPS, int MB, bool DEEP = false, bool GROUPED = false, int STRIPS = mid_strips(MB)>
int launch_mid_rows(const typename std::conditional<GROUPED, MidMoeParams, MidParams>::type& p, hipStream_t st) {
  static bool attr_set = false;   // raising the dynamic LDS limit is needed once per form
  if (!attr_set) {
    SONAR_HIP(hipFuncSetAttribute((const void*)marlin_mid_gemm<T, FMT, GROUPS, MB, DEEP, GROUPED, STRIPS>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, mid_lds(MB, DEEP, STRIPS)));
    attr_set = true;
  }
  marlin_mid_gemm<T, FMT, GROUPS, MB, DEEP, GROUPED, STRIPS>
      <<<(p.tiles * p.splits + 7) / 8 * 8, kMidWaves * 64, mid_lds(MB, DEEP, STRIPS), st>>>(p);
  return launch_status("marlin_mid_gemm");
}

template <typename T, int FMT, int GROUPS>
int launch_mid_raw(const MidParams& p, int row_blocks, int strips, hipStream_t st) {
  switch (row_blocks) {
    case 2: return launch_mid_rows<T, FMT, GROUPS, 2>(p, st);
    case 3: return launch_mid_rows<T, FMT, GROUPS, 3>(p, st);
    default:
      if (strips == 4) return launch_mid_rows<T, FMT, GROUPS, kMidMostRawRows, false, false, 4>(p, st);
      return launch_mid_rows<T, FMT, GROUPS, kMidMostRawRows>(p, st);
  }
}

template <typename T, int FMT, int GROUPS>
int launch_mid(const MidParams& p, int row_blocks, hipStream_t st) {
  switch (row_blocks) {
    case 1:
      if constexpr (FMT == kMidInt8 || FMT == kMidFp8 || FMT == kMidNvFp4) {
        if (p.tiles * p.splits <= p.cus && p.split_steps >= kMidDeepSteps * mid_ranges(mid_strips(1))) return launch_mid_rows<T, FMT, GROUPS, 1, true>(p, st);
        return launch_mid_rows<T, FMT, GROUPS, 1>(p, st);
      }
    case 2: return launch_mid_rows<T, FMT, GROUPS, 2>(p, st);
    case 3: return launch_mid_rows<T, FMT, GROUPS, 3>(p, st);
    case 4: return launch_mid_rows<T, FMT, GROUPS, 4>(p, st);
    case 5: return launch_mid_rows<T, FMT, GROUPS, 5>(p, st);
    default: return launch_mid_rows<T, FMT, GROUPS, 6>(p, st);
  }
}

template <typename T, int FMT>
int launch_mid_groups(const MidParams& p, int row_blocks, int strips, hipStream_t st) {
  if constexpr (FMT == kMidMxFp4 || FMT == kMidNvFp4) {
    return launch_mid<T, FMT, kChunkGroups>(p, row_blocks, st);
  } else {
    if constexpr (FMT == kMidInt4 || FMT == kMidInt4Zp) {
      if (p.raw_codes)
        return p.num_groups == 1 ? launch_mid_raw<T, FMT, kOneGroupRaw>(p, row_blocks, strips, st)
                                 : launch_mid_raw<T, FMT, kUnitGroupsRaw>(p, row_blocks, strips, st);
    }
    if (p.num_groups == 1) return launch_mid<T, FMT, kOneGroup>(p, row_blocks, st);
    if (p.group_shift >= 0) return launch_mid<T, FMT, kStepGroups>(p, row_blocks, st);
    return launch_mid<T, FMT, kChunkGroups>(p, row_blocks, st);
  }
}

template <typename T>
int launch_mid_format(const MidParams& p, int format, int row_blocks, int strips, hipStream_t st) {
  switch (format) {
    case kMidInt4: return launch_mid_groups<T, kMidInt4>(p, row_blocks, strips, st);
    case kMidInt4Zp: return launch_mid_groups<T, kMidInt4Zp>(p, row_blocks, strips, st);
    case kMidInt8: return launch_mid_groups<T, kMidInt8>(p, row_blocks, strips, st);
    case kMidFp8: return launch_mid_groups<T, kMidFp8>(p, row_blocks, strips, st);
    case kMidNvFp4: return launch_mid_groups<T, kMidNvFp4>(p, row_blocks, strips, st);
    default:   // MXFP4: bf16 only, which the caller has checked
      if constexpr (std::is_same<T, __bf16>::value) return launch_mid_groups<T, kMidMxFp4>(p, row_blocks, strips, st);
      return fail(SONAR_E_INVALID, "internal: MXFP4 weights with float16 activations");
  }
}

template <typename T, int FMT, int GROUPS>
int launch_mid_moe(const MidMoeParams& p, hipStream_t st) {
  const bool four = p.strips_each == 4;
  switch (p.moe.block_size) {
    case 32: return four ? launch_mid_rows<T, FMT, GROUPS, 2, false, true, 4>(p, st) : launch_mid_rows<T, FMT, GROUPS, 2, false, true>(p, st);
    case 48: return four ? launch_mid_rows<T, FMT, GROUPS, 3, false, true, 4>(p, st) : launch_mid_rows<T, FMT, GROUPS, 3, false, true>(p, st);
    case 64: return four ? launch_mid_rows<T, FMT, GROUPS, 4, false, true, 4>(p, st) : launch_mid_rows<T, FMT, GROUPS, 4, false, true>(p, st);
    default: return fail(SONAR_E_INVALID, "internal: blocks of %d slots", p.moe.block_size);
  }
}

template <typename T>
int launch_mid_moe_format(const MidMoeParams& p, int format, hipStream_t st) {
  if (format == kMidInt4)
    return p.num_groups == 1 ? launch_mid_moe<T, kMidInt4, kOneGroupRaw>(p, st) : launch_mid_moe<T, kMidInt4, kUnitGroupsRaw>(p, st);
  if (format == kMidInt4Zp)
    return p.num_groups == 1 ? launch_mid_moe<T, kMidInt4Zp, kOneGroupRaw>(p, st) : launch_mid_moe<T, kMidInt4Zp, kUnitGroupsRaw>(p, st);
  if constexpr (std::is_same<T, __bf16>::value)
    if (format == kMidMxFp4) return launch_mid_moe<T, kMidMxFp4, kChunkGroups>(p, st);
  return fail(SONAR_E_INVALID, "internal: format %d of expert weights", format);
}

}  // namespace

thread_local int g_last_mid_strips = 0;

int mid_moe_gemm(MidMoeParams p, int dtype, int format, int blocks, hipStream_t st) {
  p.splits = 1;
  p.tiles_m = blocks;
  p.strips_each = mid_moe_strips(p.moe.block_size, p.moe.rows_total / p.moe.num_experts, p.moe.num_experts, p.size_n, p.size_k, p.raw_codes, p.cus);
  g_last_mid_strips = p.strips_each;
  const int halves = p.moe.gated != nullptr && p.moe.gated_halves ? 2 : 1, across = p.size_n / kStripN / halves, each = p.strips_each / halves;
  p.tiles = blocks * ((across + each - 1) / each);
  p.split_steps = p.size_k / kMidStepK;
  return dtype == SONAR_DTYPE_F16 ? launch_mid_moe_format<_Float16>(p, format, st) : launch_mid_moe_format<__bf16>(p, format, st);
}

int mid_gemm(MidParams p, int dtype, int format, int row_blocks, hipStream_t st) {
  const int strips = p.size_n / kStripN;
  // a single row block is built for the formats that the decode kernel does not have
  if (row_blocks < 2 && (format == kMidInt4 || format == kMidInt4Zp || format == kMidMxFp4)) row_blocks = 2;
  if (p.raw_codes) row_blocks = std::min(row_blocks, kMidMostRawRows);
  p.tiles_m = (p.size_m + 16 * row_blocks - 1) / (16 * row_blocks);
  const bool by_rounds = p.raw_codes && row_blocks == kMidMostRawRows && p.splits == 1;
  const int each = by_rounds ? mid_strips_by_rounds(p.tiles_m, 0.0, p.size_n, p.size_k, true, p.cus) : mid_strips(row_blocks);
  p.tiles = p.tiles_m * ((strips + each - 1) / each);
  g_last_mid_strips = each;
  const int steps = p.size_k / kMidStepK;
  p.split_steps = (steps + p.splits - 1) / p.splits;
  if (p.raw_codes) p.split_steps = (p.split_steps + 1) & ~1;   // whole units of 128 rows
  p.splits = (steps + p.split_steps - 1) / p.split_steps;
  const int rc = dtype == SONAR_DTYPE_F16 ? launch_mid_format<_Float16>(p, format, row_blocks, each, st)
                                          : launch_mid_format<__bf16>(p, format, row_blocks, each, st);
  if (rc || p.splits == 1) return rc;
  const int blocks = (int)std::min<int64_t>(((int64_t)p.size_m * p.size_n / 4 + 255) / 256, 2048);
  if (p.splits > kMidMostSplits) return fail(SONAR_E_INVALID, "internal: %d K splits", p.splits);
  if (dtype == SONAR_DTYPE_F16) {
    if (p.splits <= 4) marlin_mid_sum<_Float16, 4><<<blocks, 256, 0, st>>>(p);
    else marlin_mid_sum<_Float16, kMidMostSplits><<<blocks, 256, 0, st>>>(p);
  } else {
    if (p.splits <= 4) marlin_mid_sum<__bf16, 4><<<blocks, 256, 0, st>>>(p);
    else marlin_mid_sum<__bf16, kMidMostSplits><<<blocks, 256, 0, st>>>(p);
  }
  return launch_status("marlin_mid_sum");
}

}  // namespace sonar

extern "C" int sonar_marlin_last_mid_strips() { return sonar::g_last_mid_strips; }
