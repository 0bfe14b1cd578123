// Weight re-ordering kernels: checkpoint packings -> Marlin tile order, and
// Marlin tile order <-> the gfx950 streaming order.  Pure integer work; the
// stores of a wavefront are one contiguous run.
#include "common.hpp"

namespace sonar {

thread_local char g_last_error[512] = "";
char* last_error_buffer() { return g_last_error; }

namespace {

// Four words from or to a caller's buffer, which need only be aligned as words (a view of a larger tensor): the loads and
// stores of this chip take that, and the type makes the compiler choose instructions that do.
typedef uint32_t words4_t __attribute__((ext_vector_type(4), aligned(4)));

// Position of a weight inside a Marlin tile (16-bit activations, 4-bit
// weights).  Word w = lane*4 + j of the tile; lane = 4*c + h, c = column % 8
// inside the 16-column sub-tile j, h = (row % 8) / 2.  Nibble slot s of the
// word holds row 2h + (s >> 2) + 8*(s & 1), column c + 8*((s >> 1) & 1).
__device__ __forceinline__ void marlin_word_sources(int word, int slot, int& row, int& col) {
  const int lane = word >> 2;
  const int j = word & 3;
  const int c = lane >> 2;
  const int h = lane & 3;
  row = 2 * h + (slot >> 2) + 8 * (slot & 1);
  col = 16 * j + c + 8 * ((slot >> 1) & 1);
}

// GPTQ / AWQ words -> Marlin words, for one matrix or a stack of them (`tiles_each` tiles of one
// matrix, `in_each` its source words; the matrices follow each other in memory).  Bound by HBM:
// every source word is read once and every output word written once.  Half a wavefront owns a
// 16 x 64 tile: each lane fetches 16 bytes of it (32 lanes: two 256-byte rows of GPTQ words or
// sixteen 32-byte rows of AWQ words), the tile meets in LDS and each lane assembles the 16 bytes of
// Marlin lane `l`.  One thread per output word gathering its eight nibbles from global memory, as
// this kernel was first written, issued eight 4-byte loads per word stored and ran at 2.2 TB/s
// (117 MB moved for a 4096 x 28672 matrix in 53 us; 23 us = 5.1 TB/s this way).
// kRepackTiles tiles a workgroup.
constexpr int kRepackTiles = 8;
constexpr int kRepackLdsStride = 136;   // words between the tiles of a wavefront: neighbours on other banks

// Marlin word of the low and high nibbles of four source bytes: nibble slots 0..3 are the low nibbles
// of b0, b1, b2, b3, slots 4..7 the high ones.
__device__ __forceinline__ uint32_t interleave_nibbles(uint32_t b0, uint32_t b1, uint32_t b2, uint32_t b3) {
  const uint32_t x = b0 | (b2 << 8);   // slots 0 and 2
  const uint32_t y = b1 | (b3 << 8);   // slots 1 and 3
  const uint32_t lo = (x & 0x0F0Fu) | ((y & 0x0F0Fu) << 4);
  const uint32_t hi = ((x >> 4) & 0x0F0Fu) | (y & 0xF0F0u);
  return lo | (hi << 16);
}

// With HAS_PERM (act-order) the sixteen rows of a tile come from sixteen words of different rows: a
// half wavefront reads each as 256 bytes and leaves the selected nibbles in LDS in the source's own packing.
template <bool HAS_PERM>
__device__ __forceinline__ void gptq_tiles(uint32_t* lds, const uint32_t block, const uint32_t* __restrict__ in,
                                           const int32_t* __restrict__ perm, uint32_t* __restrict__ out, int size_k,
                                           int size_n, uint32_t tiles_each, long in_each, uint32_t total_tiles) {
  const uint32_t n_tiles = size_n / kMarlinTileN;
  const int sub = threadIdx.x >> 5, l = threadIdx.x & 31;
  const uint32_t tile = block * kRepackTiles + sub;
  const bool live = tile < total_tiles;
  uint32_t* mine = lds + sub * kRepackLdsStride;
  if (live) {
    const uint32_t matrix = tile / tiles_each, t = tile - matrix * tiles_each;
    const int kt = (int)(t / n_tiles), nt = (int)(t - kt * n_tiles);
    const uint32_t* src = in + matrix * in_each + nt * kMarlinTileN;
    const int half = l >> 4, col = 4 * (l & 15);   // which eight rows of the tile, first of four columns
    u32x4_t v;
    if constexpr (HAS_PERM) {
      const int32_t* rows = perm + (long)matrix * size_k + kt * kMarlinTileK + 8 * half;
      v = u32x4_t{0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int k = rows[r];
        const u32x4_t w = *reinterpret_cast<const words4_t*>(src + (long)(k >> 3) * size_n + col);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] |= ((w[i] >> (4 * (k & 7))) & 0xFu) << (4 * r);
      }
    } else {
      v = *reinterpret_cast<const words4_t*>(src + (long)(2 * kt + half) * size_n + col);
    }
    *reinterpret_cast<u32x4_t*>(mine + half * kMarlinTileN + col) = v;
  }
  __syncthreads();
  if (!live) return;
  const int c = l >> 2, h = l & 3;
  u32x4_t o;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    // byte h of a source word: rows 2h (low nibble) and 2h + 1 of its column
    const uint32_t* w = mine + 16 * j + c;
    o[j] = interleave_nibbles((w[0] >> (8 * h)) & 0xFFu, (w[kMarlinTileN] >> (8 * h)) & 0xFFu,
                              (w[8] >> (8 * h)) & 0xFFu, (w[kMarlinTileN + 8] >> (8 * h)) & 0xFFu);
  }
  *reinterpret_cast<words4_t*>(out + (long)tile * kMarlinTileWords + 4 * l) = o;
}
template <bool HAS_PERM>
__global__ __launch_bounds__(256) void gptq_to_marlin_kernel(
    const uint32_t* __restrict__ in, const int32_t* __restrict__ perm, uint32_t* __restrict__ out, int size_k,
    int size_n, uint32_t tiles_each, long in_each, uint32_t total_tiles) {
  __shared__ alignas(16) uint32_t lds[kRepackTiles * kRepackLdsStride];
  gptq_tiles<HAS_PERM>(lds, blockIdx.x, in, perm, out, size_k, size_n, tiles_each, in_each, total_tiles);
}

__global__ __launch_bounds__(256) void awq_to_marlin_kernel(
    const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int size_n, uint32_t tiles_each, long in_each,
    uint32_t total_tiles) {
  __shared__ alignas(16) uint32_t lds[kRepackTiles * kRepackLdsStride];
  const uint32_t n_tiles = size_n / kMarlinTileN;
  const int sub = threadIdx.x >> 5, l = threadIdx.x & 31;
  const uint32_t tile = blockIdx.x * kRepackTiles + sub;
  const bool live = tile < total_tiles;
  uint32_t* mine = lds + sub * kRepackLdsStride;
  if (live) {
    const uint32_t matrix = tile / tiles_each, t = tile - matrix * tiles_each;
    const int kt = (int)(t / n_tiles), nt = (int)(t - kt * n_tiles);
    const uint32_t* src = in + matrix * in_each + (long)(kt * kMarlinTileK + (l >> 1)) * (size_n / 8) +
                          nt * (kMarlinTileN / 8) + 4 * (l & 1);
    *reinterpret_cast<u32x4_t*>(mine + 4 * l) = *reinterpret_cast<const words4_t*>(src);   // row l / 2 of the tile: 8 words
  }
  __syncthreads();
  if (!live) return;
  const int c = l >> 2, h = l & 3;
  const int shift = 4 * ((c >> 1) + 4 * (c & 1));   // column n % 8 = c sits at nibble c / 2 + 4 (c % 2)
  u32x4_t o;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t* w = mine + 2 * h * 8 + 2 * j;   // rows 2h, 2h + 1 and eight further down; words 2j (columns 16j..) and 2j + 1
    uint32_t b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t* at = w + (i & 1) * 64 + (i >> 1);
      b[i] = ((at[0] >> shift) & 0xFu) | (((at[8] >> shift) & 0xFu) << 4);
    }
    o[j] = interleave_nibbles(b[0], b[1], b[2], b[3]);
  }
  *reinterpret_cast<words4_t*>(out + (long)tile * kMarlinTileWords + 4 * l) = o;
}

// One thread per gfx950 word.  Word j of lane L of chunk c of strip s holds
// column 64s + 16j + L%16, rows 32c + 8*(L/16) + t (t = 0..7) with row t at
// nibble slot t/2 + 4*(t%2).  Those eight rows live in Marlin k-tile
// 2c + (L/32) at tile rows 8*((L/16)%2) + t, i.e. in the four Marlin words
// lane_m*4 + j with lane_m = 4*(col%8) + t/2.
__global__ __launch_bounds__(256) void marlin_to_gfx950_kernel(
    const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int size_k,
    int size_n, long total_words) {
  const int n_tiles = size_n / kMarlinTileN;
  const int chunks = size_k / kChunkK;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total_words;
       idx += (long)gridDim.x * blockDim.x) {
    const int j = (int)(idx & 3);
    const int lane = (int)((idx >> 2) & 63);
    const long chunk_id = idx >> 8;
    const int c = (int)(chunk_id % chunks);
    const int s = (int)(chunk_id / chunks);
    const int col16 = lane & 15;
    const int kb = lane >> 4;
    const int kt = 2 * c + (kb >> 1);
    const int hb = kb & 1;  // upper half of the 16-row tile?
    const uint32_t* tile = in + ((long)kt * n_tiles + s) * kMarlinTileWords;
    // Marlin slot of (tile row 8*hb + t, column col16): hb + 2*(col16/8) + 4*(t%2)
    const int slot_even = hb + 2 * (col16 >> 3);
    uint32_t packed = 0;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const uint32_t w = tile[(4 * (col16 & 7) + h) * 4 + j];
      const uint32_t even = (w >> (4 * slot_even)) & 0xFu;        // row t = 2h
      const uint32_t odd = (w >> (4 * (slot_even + 4))) & 0xFu;   // row t = 2h+1
      packed |= (even << (4 * h)) | (odd << (4 * (h + 4)));
    }
    out[idx] = packed;
  }
}

// Inverse of the above: one thread per Marlin word.
__global__ __launch_bounds__(256) void gfx950_to_marlin_kernel(
    const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int size_k,
    int size_n, long total_words) {
  const int n_tiles = size_n / kMarlinTileN;
  const int chunks = size_k / kChunkK;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total_words;
       idx += (long)gridDim.x * blockDim.x) {
    const long tile = idx / kMarlinTileWords;
    const int word = (int)(idx % kMarlinTileWords);
    const int kt = (int)(tile / n_tiles);
    const int nt = (int)(tile % n_tiles);
    uint32_t packed = 0;
#pragma unroll
    for (int slot = 0; slot < 8; ++slot) {
      int row, col;
      marlin_word_sources(word, slot, row, col);
      const int k = kt * kMarlinTileK + row;
      const int c = k / kChunkK;
      const int kb = (k % kChunkK) >> 3;
      const int t = k & 7;
      const int lane = 16 * kb + (col & 15);
      const int j = col >> 4;
      const uint32_t src = in[(((long)nt * chunks + c) * 64 + lane) * 4 + j];
      const int src_slot = (t >> 1) + 4 * (t & 1);
      packed |= ((src >> (4 * src_slot)) & 0xFu) << (4 * slot);
    }
    out[idx] = packed;
  }
}

// ---- 8-bit codes (uint8b128): the same 16 x 64 tile in 256 words.  Word
// lane*8 + 2j + half of the tile; lane = 4*c + h as above; byte s of the word
// holds row 2h + (s >> 1) + 8*(s & 1), column 16j + c + 8*half
// (gptq_marlin_repack.cu:216-236).
constexpr int kMarlinTileWords8 = 256;

__device__ __forceinline__ void marlin8_word_sources(int word, int byte, int& row, int& col) {
  const int lane = word >> 3;
  const int j = (word >> 1) & 3;
  const int half = word & 1;
  row = 2 * (lane & 3) + (byte >> 1) + 8 * (byte & 1);
  col = 16 * j + (lane >> 2) + 8 * half;
}

// GPTQ (K/4, N) int32, byte k % 4 of word [k / 4][n] -> Marlin 8-bit order.
template <bool HAS_PERM>
__global__ __launch_bounds__(256) void gptq8_to_marlin_kernel(
    const uint32_t* __restrict__ in, const int32_t* __restrict__ perm,
    uint32_t* __restrict__ out, int size_k, int size_n, long total_words) {
  const int n_tiles = size_n / kMarlinTileN;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total_words;
       idx += (long)gridDim.x * blockDim.x) {
    const long tile = idx / kMarlinTileWords8;
    const int word = (int)(idx % kMarlinTileWords8);
    const int kt = (int)(tile / n_tiles);
    const int nt = (int)(tile % n_tiles);
    uint32_t packed = 0;
#pragma unroll
    for (int byte = 0; byte < 4; ++byte) {
      int row, col;
      marlin8_word_sources(word, byte, row, col);
      int k = kt * kMarlinTileK + row;
      if (HAS_PERM) k = perm[k];
      const int n = nt * kMarlinTileN + col;
      const uint32_t src = in[(long)(k >> 2) * size_n + n];
      packed |= ((src >> (8 * (k & 3))) & 0xFFu) << (8 * byte);
    }
    out[idx] = packed;
  }
}

// Position of W[k][n] in the Marlin 8-bit order: word index and byte.
__device__ __forceinline__ long marlin8_position(int k, int n, int n_tiles, int& byte) {
  const int kt = k / kMarlinTileK, row = k % kMarlinTileK;
  const int nt = n / kMarlinTileN, col = n % kMarlinTileN;
  const int c16 = col & 15;
  const int lane = 4 * (c16 & 7) + ((row & 7) >> 1);
  byte = ((row & 1) << 1) | (row >> 3);
  return ((long)kt * n_tiles + nt) * kMarlinTileWords8 + lane * 8 + 2 * (col >> 4) + (c16 >> 3);
}

// The gfx950 order for 8-bit codes: per strip a stream of 1-KiB blocks of 16
// rows, block 2c + h in chunk c; word j of lane L: column 64s + 16j + L%16,
// rows 32c + 8*(L/16) + 4h + t, row t at byte {0, 2, 1, 3}[t].
__device__ __forceinline__ long gfx950_8_position(int k, int n, int chunks, int& byte) {
  const int s = n / kStripN, j = (n % kStripN) >> 4, l16 = n & 15;
  const int c = k / kChunkK, r = k % kChunkK;
  const int kb = r >> 3, h = (r >> 2) & 1, t = r & 3;
  byte = ((t & 1) << 1) | (t >> 1);
  return ((((long)s * chunks + c) * 2 + h) * 64 + 16 * kb + l16) * 4 + j;
}

// One thread per output word; TO_GFX950 selects the direction.
template <bool TO_GFX950>
__global__ __launch_bounds__(256) void marlin8_gfx950_kernel(const uint32_t* __restrict__ in,
                                                            uint32_t* __restrict__ out, int size_k, int size_n,
                                                            long total_words) {
  const int n_tiles = size_n / kMarlinTileN;
  const int chunks = size_k / kChunkK;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total_words;
       idx += (long)gridDim.x * blockDim.x) {
    uint32_t packed = 0;
#pragma unroll
    for (int byte = 0; byte < 4; ++byte) {
      int k, n;
      if (TO_GFX950) {  // which (k, n) does byte `byte` of gfx950 word idx hold?
        const int j = (int)(idx & 3);
        const int lane = (int)((idx >> 2) & 63);
        const long block = idx >> 8;
        const int h = (int)(block & 1);
        const int c = (int)((block >> 1) % chunks);
        const int s = (int)((block >> 1) / chunks);
        const int t = ((byte & 1) << 1) | (byte >> 1);
        k = c * kChunkK + 8 * (lane >> 4) + 4 * h + t;
        n = s * kStripN + 16 * j + (lane & 15);
      } else {
        const long tile = idx / kMarlinTileWords8;
        int row, col;
        marlin8_word_sources((int)(idx % kMarlinTileWords8), byte, row, col);
        k = (int)(tile / n_tiles) * kMarlinTileK + row;
        n = (int)(tile % n_tiles) * kMarlinTileN + col;
      }
      int src_byte;
      const long src = TO_GFX950 ? marlin8_position(k, n, n_tiles, src_byte)
                                 : gfx950_8_position(k, n, chunks, src_byte);
      packed |= ((in[src] >> (8 * src_byte)) & 0xFFu) << (8 * byte);
    }
    out[idx] = packed;
  }
}

// ---- 4-bit codes for 8-bit activations (is_a_8bit): tiles of 32 (k) x 32 (n),
// 128 words each, tile (kt, nt) at (kt * (N / 32) + nt) * 128.  Word lane*4 + w:
// column 8w + lane/4; nibble slot s holds row 4*(lane%4) + s/2 + 16*(s%2)
// (gptq_marlin_repack.cu:129-141,176-216).
constexpr int kA8Tile = 32;

__device__ __forceinline__ void a8_word_sources(int word, int slot, int& row, int& col) {
  const int lane = word >> 2;
  row = 4 * (lane & 3) + (slot >> 1) + 16 * (slot & 1);
  col = 8 * (word & 3) + (lane >> 2);
}

// Word index and nibble slot of W[k][n] in that order.
__device__ __forceinline__ long a8_position(int k, int n, int n_tiles, int& slot) {
  const int r = k % kA8Tile, c = n % kA8Tile;
  slot = 2 * (r & 3) + (r >> 4);
  return ((long)(k / kA8Tile) * n_tiles + n / kA8Tile) * kMarlinTileWords + (4 * (c & 7) + ((r & 15) >> 2)) * 4 +
         (c >> 3);
}

// SOURCE 0: GPTQ (K/8, N) words; 1: AWQ (K, N/8) words; 2: the gfx950 order.
template <int SOURCE>
__global__ __launch_bounds__(256) void to_marlin_a8_kernel(const uint32_t* __restrict__ in,
                                                          uint32_t* __restrict__ out, int size_k, int size_n,
                                                          long total_words) {
  const int n_tiles = size_n / kA8Tile;
  const int chunks = size_k / kChunkK;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total_words;
       idx += (long)gridDim.x * blockDim.x) {
    const long tile = idx / kMarlinTileWords;
    const int word = (int)(idx % kMarlinTileWords);
    uint32_t packed = 0;
#pragma unroll
    for (int slot = 0; slot < 8; ++slot) {
      int row, col;
      a8_word_sources(word, slot, row, col);
      const int k = (int)(tile / n_tiles) * kA8Tile + row;
      const int n = (int)(tile % n_tiles) * kA8Tile + col;
      uint32_t code;
      if (SOURCE == 0) {
        code = in[(long)(k >> 3) * size_n + n] >> (4 * (k & 7));
      } else if (SOURCE == 1) {
        const int p = ((n & 7) >> 1) + 4 * (n & 1);
        code = in[(long)k * (size_n / 8) + (n >> 3)] >> (4 * p);
      } else {
        const int t = k & 7;
        const int lane = 16 * ((k % kChunkK) >> 3) + (n & 15);
        code = in[(((long)(n / kStripN) * chunks + k / kChunkK) * 64 + lane) * 4 + ((n % kStripN) >> 4)] >>
               (4 * ((t >> 1) + 4 * (t & 1)));
      }
      packed |= (code & 0xFu) << (4 * slot);
    }
    out[idx] = packed;
  }
}

// 8-bit codes in that order (gptq_marlin_repack.cu:216-236 with is_a_8bit): a 32 x 32 tile is 256
// words; word lane*8 + 2*w + h: column 8w + lane/4, rows 4*(lane%4) + {0..3} + 16h at bytes 0..3.
// No GEMM takes it (the reference has no 8-bit weights with 8-bit activations either); the
// repack op produces it.  Source: GPTQ (K/4, N) words.
__global__ __launch_bounds__(256) void gptq8_to_marlin_a8_kernel(const uint32_t* __restrict__ in,
                                                                uint32_t* __restrict__ out, int size_k, int size_n,
                                                                long total_words) {
  const int n_tiles = size_n / kA8Tile;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total_words;
       idx += (long)gridDim.x * blockDim.x) {
    const long tile = idx / 256;
    const int word = (int)(idx % 256);
    const int lane = word >> 3, w = (word >> 1) & 3, h = word & 1;
    const int n = (int)(tile % n_tiles) * kA8Tile + 8 * w + (lane >> 2);
    const int k0 = (int)(tile / n_tiles) * kA8Tile + 4 * (lane & 3) + 16 * h;   // a multiple of 4: one source word
    out[idx] = in[(long)(k0 >> 2) * size_n + n];
  }
}

// One thread per gfx950 word (rows 32c + 8*(L/16) + t of column 64s + 16j + L%16).
__global__ __launch_bounds__(256) void marlin_a8_to_gfx950_kernel(const uint32_t* __restrict__ in,
                                                                 uint32_t* __restrict__ out, int size_k,
                                                                 int size_n, long total_words) {
  const int n_tiles = size_n / kA8Tile;
  const int chunks = size_k / kChunkK;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total_words;
       idx += (long)gridDim.x * blockDim.x) {
    const int j = (int)(idx & 3);
    const int lane = (int)((idx >> 2) & 63);
    const long chunk_id = idx >> 8;
    const int n = (int)(chunk_id / chunks) * kStripN + 16 * j + (lane & 15);
    const int k0 = (int)(chunk_id % chunks) * kChunkK + 8 * (lane >> 4);
    uint32_t packed = 0;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      int slot;
      const long src = a8_position(k0 + t, n, n_tiles, slot);
      packed |= ((in[src] >> (4 * slot)) & 0xFu) << (4 * ((t >> 1) + 4 * (t & 1)));
    }
    out[idx] = packed;
  }
}

// marlin_int4_fp8_preprocess.cu:13-66: nibble by nibble, code -> sign and
// magnitude of code - z (z = 8 without zero points): q >= z ? q - z : 15 - q.
__global__ __launch_bounds__(256) void int4_fp8_preprocess_kernel(const uint32_t* __restrict__ in,
                                                                 const uint32_t* __restrict__ zeros,
                                                                 uint32_t* __restrict__ out, long words_per_row,
                                                                 int group_size, long total_words) {
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total_words;
       idx += (long)gridDim.x * blockDim.x) {
    uint32_t val = in[idx];
    uint32_t zero = zeros ? zeros[(idx / words_per_row) / group_size * words_per_row + idx % words_per_row]
                          : 0x88888888u;
    uint32_t res = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t q = (val >> (4 * i)) & 0xFu, z = (zero >> (4 * i)) & 0xFu;
      res |= (q >= z ? q - z : 15u - q) << (4 * i);
    }
    out[idx] = res;
  }
}

// ---- checkpoint tensors around the codes -----------------------------------
// marlin_permute_scales / marlin_permute_bias on 16-bit elements: inside every 64 columns
// out[8 i + j] = in[i + 8 j] (groups along K), or inside every 32 columns
// out[8 i + j] = in[2 i + {0, 1, 8, 9, 16, 17, 24, 25}[j]] (one group, bias).  A thread stores 16
// bytes; its loads stay inside one 128-byte line.
template <bool GROUPS>
__device__ __forceinline__ void permute_scale_vector(const uint16_t* __restrict__ in, uint16_t* __restrict__ out,
                                                     const long v) {
  uint32_t o[4];
  if constexpr (GROUPS) {
    const uint16_t* src = in + (v >> 3) * 64 + (v & 7);
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = (uint32_t)src[16 * j] | ((uint32_t)src[16 * j + 8] << 16);
  } else {
    const uint16_t* src = in + (v >> 2) * 32 + 2 * (v & 3);
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = (uint32_t)src[8 * j] | ((uint32_t)src[8 * j + 1] << 16);
  }
  *reinterpret_cast<uint4*>(out + 8 * v) = make_uint4(o[0], o[1], o[2], o[3]);
}
template <bool GROUPS>
__global__ __launch_bounds__(256) void permute_scale_columns(const uint16_t* __restrict__ in,
                                                             uint16_t* __restrict__ out, long vectors) {
  const long v = (long)blockIdx.x * 256 + threadIdx.x;
  if (v < vectors) permute_scale_vector<GROUPS>(in, out, v);
}

// Packed zero points -> Marlin zero points, (rows, N/8) words.  Nibble e of output word w is the code
// of column 64 (w / 8) + w % 8 + 8 * i(e), i = {0, 2, 4, 6, 1, 3, 5, 7} (the column interleave of the
// 16-bit dequantiser; the identity for 8-bit activations), i.e. always nibble w % 8 of a source word,
// or nibble (w % 8) / 2 + 4 (w % 2) where the source has the AWQ order.
__device__ __forceinline__ void pack_zero_word(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, const long idx,
                                               int words, long row_stride, long word_stride, bool awq_order, bool a8) {
  const long row = idx / words;
  const int w = (int)(idx - row * words);
  const int shift = 4 * (awq_order ? ((w & 7) >> 1) + 4 * (w & 1) : w & 7);
  const uint32_t* src = in + row * row_stride + (long)(w & ~7) * word_stride;
  uint32_t packed = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int from = a8 ? e : (e < 4 ? 2 * e : 2 * e - 7);
    packed |= ((src[from * word_stride] >> shift) & 0xFu) << (4 * e);
  }
  out[idx] = packed;
}
__global__ __launch_bounds__(256) void pack_zero_points(const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
                                                        int words, long total, long row_stride, long word_stride,
                                                        bool awq_order, bool a8) {
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx < total) pack_zero_word(in, out, idx, words, row_stride, word_stride, awq_order, a8);
}

// A GPTQ-like projection as one launch: codes, scales, zero points (when it has any) and the tickets of its workspace, which
// start at zero.  A workgroup's number says which of the four it works on; each is the body of the kernel that does it
// alone.  Up to about 40 MB of codes a load is bound by the host, which made three or four operator calls with a launch
// each; one call takes 4096x4096 from 31 us to 18 (a copy of its bytes: 3), the same with AWQ's conversion before it from
// 46 to 27, and 14336x28672, where the three launches followed one another, from 76 to 71 (its bytes: 82 at the rate of a
// large copy, part of them in the memory-side cache).
struct LoadLinear {
  const uint32_t* codes;
  uint32_t* codes_out;
  int size_k, size_n;
  uint32_t tiles, code_blocks;
  const uint16_t* scales;
  uint16_t* scales_out;
  long vectors;
  uint32_t scale_blocks;
  const uint32_t* zeros;
  uint32_t* zeros_out;
  long zero_words, zero_row_stride, zero_word_stride;
  uint32_t zero_blocks;
  uint32_t* workspace;
  int workspace_words;
  const int32_t* perm;   // act-order: the rows in the order of their groups
};
template <bool GROUPS, bool HAS_PERM>
__global__ __launch_bounds__(256) void load_linear_kernel(const LoadLinear p) {
  __shared__ alignas(16) uint32_t lds[kRepackTiles * kRepackLdsStride];
  uint32_t block = blockIdx.x;
  if (block < p.code_blocks) {
    gptq_tiles<HAS_PERM>(lds, block, p.codes, p.perm, p.codes_out, p.size_k, p.size_n, p.tiles, 0, p.tiles);
    return;
  }
  block -= p.code_blocks;
  if (block < p.scale_blocks) {
    const long v = (long)block * 256 + threadIdx.x;
    if (v < p.vectors) permute_scale_vector<GROUPS>(p.scales, p.scales_out, v);
    return;
  }
  block -= p.scale_blocks;
  if (block < p.zero_blocks) {
    const long w = (long)block * 256 + threadIdx.x;
    if (w < p.zero_words)
      pack_zero_word(p.zeros, p.zeros_out, w, p.size_n / 8, p.zero_row_stride, p.zero_word_stride, false, false);
    return;
  }
  for (int i = threadIdx.x; i < p.workspace_words; i += 256) p.workspace[i] = 0;
}

// AutoAWQ codes (K, N/8) -> the GPTQ packing (K/8, N): a thread transposes the 8 x 8 nibbles of eight
// rows of one word, three rounds of block swaps, and stores the eight columns side by side.
__device__ __forceinline__ void awq_codes_word(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int words, long idx) {
  const long r = idx / words;
  const int w = (int)(idx - r * words);
  uint32_t x[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) x[t] = in[(8 * r + t) * words + w];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t a = x[i], b = x[i + 4];
    x[i] = (a & 0xFFFFu) | (b << 16);
    x[i + 4] = (a >> 16) | (b & 0xFFFF0000u);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int i = (q >> 1) * 4 + (q & 1);
    const uint32_t a = x[i], b = x[i + 2];
    x[i] = (a & 0x00FF00FFu) | ((b & 0x00FF00FFu) << 8);
    x[i + 2] = ((a >> 8) & 0x00FF00FFu) | (b & 0xFF00FF00u);
  }
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    const uint32_t a = x[i], b = x[i + 1];
    x[i] = (a & 0x0F0F0F0Fu) | ((b & 0x0F0F0F0Fu) << 4);
    x[i + 1] = ((a >> 4) & 0x0F0F0F0Fu) | (b & 0xF0F0F0F0u);
  }
  // x[p] now holds nibble p of every row; column c sits at nibble c / 2 + 4 (c % 2)
  uint32_t* dst = out + r * (8L * words) + 8 * w;
  *reinterpret_cast<words4_t*>(dst) = words4_t{x[0], x[4], x[1], x[5]};
  *reinterpret_cast<words4_t*>(dst + 4) = words4_t{x[2], x[6], x[3], x[7]};
}

// AutoAWQ zero points (G, N/8) -> plain column order, transposed: (N/8, G).
__device__ __forceinline__ void awq_zeros_word(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, int groups, int words,
                                               long idx) {
  const long w = idx / groups;
  const uint32_t z = in[(idx - w * groups) * words + w];
  uint32_t packed = 0;
#pragma unroll
  for (int c = 0; c < 8; ++c) packed |= ((z >> (4 * ((c >> 1) + 4 * (c & 1)))) & 0xFu) << (4 * c);
  out[idx] = packed;
}

// Codes and zero points of a projection as one launch: bound by the host, it takes two of the 26.6 us off a load of 1024 x 4096.
struct AwqToPlain {
  const uint32_t* codes;
  uint32_t* codes_out;
  const uint32_t* zeros;
  uint32_t* zeros_out;
  int words, groups;         // words of a row (N / 8)
  long code_words, zero_words;
  uint32_t code_blocks;
};
__global__ __launch_bounds__(256) void awq_to_plain_kernel(const AwqToPlain p) {
  if (blockIdx.x < p.code_blocks) {
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx < p.code_words) awq_codes_word(p.codes, p.codes_out, p.words, idx);
  } else {
    const long idx = (long)(blockIdx.x - p.code_blocks) * 256 + threadIdx.x;
    if (idx < p.zero_words) awq_zeros_word(p.zeros, p.zeros_out, p.groups, p.words, idx);
  }
}

// The groups of the rows of an act-order projection in ascending order, and the rows in that order, those of a group as they came
// (torch.argsort and two gathers of the reference, marlin_utils.py: marlin_sort_g_idx).  The rank of a row is the number of smaller
// groups and of equal ones before it; a workgroup finds it for 64 rows.  Groups below kSortBins, all that a checkpoint holds, are
// counted in LDS, over all rows and over those before the workgroup's, and the counts summed up; for any other value the 16
// wavefronts compare each row with a sixteenth of all rows, which come as scalars, two vector instructions a pair.  Calls
// in a row: K = 1024 6 us, 14336 8 (compared 22), 32768 16 (compared 73); a library's sort and gathers, launches of their own, 34 to 51.
constexpr int kSortWaves = 16, kSortBins = 64 * kSortWaves;
__global__ __launch_bounds__(64 * kSortWaves) void sort_group_indices(const int32_t* __restrict__ g, int32_t* __restrict__ sorted,
                                                                      int32_t* __restrict__ order, int n) {
  __shared__ int32_t counts[kSortWaves][64];   // by wavefront and row; or of the rows before the workgroup's, by group
  __shared__ int32_t all[kSortBins], totals[kSortWaves];
  int32_t* before = &counts[0][0];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int first = 64 * blockIdx.x, i = first + lane;
  const int32_t mine = i < n ? g[i] : 0;
  all[threadIdx.x] = 0;
  before[threadIdx.x] = 0;
  __syncthreads();
  int other = 0;
#pragma unroll 4
  for (int j = threadIdx.x; j < n; j += kSortBins) {
    const int32_t group = g[j];
    if ((uint32_t)group < (uint32_t)kSortBins) {
      atomicAdd(&all[group], 1);
      if (j < first) atomicAdd(&before[group], 1);
    } else {
      other = 1;
    }
  }
  int rank = 0;
  if (!__syncthreads_or(other)) {
    int sum = all[threadIdx.x];   // up to and with this group
    const int own = sum;
#pragma unroll
    for (int step = 1; step < 64; step *= 2) {
      const int below = __shfl_up(sum, step);
      sum += lane >= step ? below : 0;
    }
    if (lane == 63) totals[wave] = sum;
    __syncthreads();
    for (int w = 0; w < wave; ++w) sum += totals[w];
    all[threadIdx.x] = sum - own;
    __syncthreads();
    if (wave > 0) return;
    for (int l = 0; l < 64; ++l) rank += l < lane && __builtin_amdgcn_readlane(mine, l) == mine ? 1 : 0;
    rank += all[mine] + before[mine];
  } else {
    const int share = (n + kSortWaves - 1) / kSortWaves, from = wave * share, to = min(n, from + share);
    int count = 0;
#pragma unroll 16
    for (int j = from; j < min(to, first); ++j) count += g[j] <= mine ? 1 : 0;
    for (int j = max(from, first); j < min(to, first + 64); ++j) count += g[j] < mine || (g[j] == mine && j < i) ? 1 : 0;
#pragma unroll 16
    for (int j = max(from, first + 64); j < to; ++j) count += g[j] < mine ? 1 : 0;
    counts[wave][lane] = count;
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) rank += counts[w][lane];
  }
  if (i >= n) return;
  sorted[rank] = mine;
  order[rank] = i;
}

int grid_for(long total_words) {
  long blocks = (total_words + 255) / 256;
  if (blocks > 256L * 32) blocks = 256L * 32;
  if (blocks < 1) blocks = 1;
  return (int)blocks;
}

int launch_awq_to_plain(AwqToPlain p, hipStream_t st) {
  p.code_blocks = (uint32_t)((p.code_words + 255) / 256);
  const int64_t blocks = (int64_t)p.code_blocks + (p.zero_words + 255) / 256;
  SONAR_REQUIRE(blocks < (1LL << 31), "weight too large");
  awq_to_plain_kernel<<<(int)blocks, 256, 0, st>>>(p);
  return launch_status("awq_to_plain_kernel");
}

int check_repack_shape(int64_t size_k, int64_t size_n, int num_bits) {
  SONAR_REQUIRE(num_bits == 4 || num_bits == 8, "num_bits must be 4 or 8. Got = %d", num_bits);
  SONAR_REQUIRE(size_k > 0 && size_n > 0, "size_k = %ld and size_n = %ld must be positive",
                (long)size_k, (long)size_n);
  SONAR_REQUIRE(size_k % kMarlinTileK == 0, "size_k = %ld is not divisible by tile_k_size = %d",
                (long)size_k, kMarlinTileK);
  SONAR_REQUIRE(size_n % kMarlinTileN == 0, "size_n = %ld is not divisible by tile_n_size = %d",
                (long)size_n, kMarlinTileN);
  SONAR_REQUIRE(size_k * size_n / 8 < (1LL << 37), "weight too large");   // half a terabyte of packed codes
  SONAR_REQUIRE(size_k < (1LL << 30) && size_n < (1LL << 30), "size_k / size_n too large");
  return SONAR_OK;
}

int check_experts(int64_t experts, int64_t size_k, int64_t size_n) {
  SONAR_REQUIRE(experts >= 1 && experts * (size_k / kMarlinTileK) * (size_n / kMarlinTileN) < (1LL << 31),
                "experts = %ld out of range", (long)experts);
  return SONAR_OK;
}

int launch_gptq_to_marlin(const uint32_t* in, const int32_t* perm, uint32_t* out, int64_t experts, int64_t size_k,
                          int64_t size_n, hipStream_t st) {
  const long each = (size_k / kMarlinTileK) * (size_n / kMarlinTileN), total = experts * each;
  const int blocks = (int)((total + kRepackTiles - 1) / kRepackTiles);
  auto* kernel = perm ? gptq_to_marlin_kernel<true> : gptq_to_marlin_kernel<false>;
  kernel<<<blocks, 256, 0, st>>>(in, perm, out, (int)size_k, (int)size_n, (uint32_t)each, size_k * size_n / 8,
                                (uint32_t)total);
  return launch_status("gptq_to_marlin_kernel");
}

int launch_awq_to_marlin(const uint32_t* in, uint32_t* out, int64_t experts, int64_t size_k, int64_t size_n,
                         hipStream_t st) {
  const long each = (size_k / kMarlinTileK) * (size_n / kMarlinTileN), total = experts * each;
  const int blocks = (int)((total + kRepackTiles - 1) / kRepackTiles);
  awq_to_marlin_kernel<<<blocks, 256, 0, st>>>(in, out, (int)size_n, (uint32_t)each, size_k * size_n / 8,
                                              (uint32_t)total);
  return launch_status("awq_to_marlin_kernel");
}

}  // namespace
}  // namespace sonar

using namespace sonar;

extern "C" const char* sonar_marlin_last_error(void) { return last_error_buffer(); }
extern "C" const char* sonar_marlin_version(void) { return "sonar-marlin-gfx950 0.1"; }

extern "C" int sonar_gptq_marlin_repack(const uint32_t* b_q_weight, const int32_t* perm,
                                        uint32_t* out, int64_t size_k, int64_t size_n,
                                        int num_bits, void* stream) {
  if (int rc = check_repack_shape(size_k, size_n, num_bits)) return rc;
  SONAR_REQUIRE(b_q_weight && out, "b_q_weight and out must not be NULL");
  hipStream_t st = (hipStream_t)stream;
  if (num_bits == 8) {
    const long words = size_k * size_n / 4;
    if (perm)
      gptq8_to_marlin_kernel<true><<<grid_for(words), 256, 0, st>>>(b_q_weight, perm, out, (int)size_k,
                                                                   (int)size_n, words);
    else
      gptq8_to_marlin_kernel<false><<<grid_for(words), 256, 0, st>>>(b_q_weight, nullptr, out, (int)size_k,
                                                                    (int)size_n, words);
    return launch_status("gptq8_to_marlin_kernel");
  }
  return launch_gptq_to_marlin(b_q_weight, perm, out, 1, size_k, size_n, st);
}

extern "C" int sonar_awq_marlin_repack(const uint32_t* b_q_weight, uint32_t* out, int64_t size_k,
                                       int64_t size_n, int num_bits, void* stream) {
  if (int rc = check_repack_shape(size_k, size_n, num_bits)) return rc;
  if (num_bits != 4) return fail(SONAR_E_UNSUPPORTED, "awq_marlin_repack: 8-bit AWQ weights are not built");
  SONAR_REQUIRE(b_q_weight && out, "b_q_weight and out must not be NULL");
  return launch_awq_to_marlin(b_q_weight, out, 1, size_k, size_n, (hipStream_t)stream);
}

// The stacked forms: matrix e at b_q_weight + e * K * N / 8 words (perm + e * K), one launch for all of them.
extern "C" int sonar_gptq_marlin_moe_repack(const uint32_t* b_q_weight, const int32_t* perm, uint32_t* out,
                                            int64_t experts, int64_t size_k, int64_t size_n, void* stream) {
  if (int rc = check_repack_shape(size_k, size_n, 4)) return rc;
  if (int rc = check_experts(experts, size_k, size_n)) return rc;
  SONAR_REQUIRE(b_q_weight && out, "b_q_weight and out must not be NULL");
  return launch_gptq_to_marlin(b_q_weight, perm, out, experts, size_k, size_n, (hipStream_t)stream);
}

extern "C" int sonar_awq_marlin_moe_repack(const uint32_t* b_q_weight, uint32_t* out, int64_t experts,
                                           int64_t size_k, int64_t size_n, void* stream) {
  if (int rc = check_repack_shape(size_k, size_n, 4)) return rc;
  if (int rc = check_experts(experts, size_k, size_n)) return rc;
  SONAR_REQUIRE(b_q_weight && out, "b_q_weight and out must not be NULL");
  return launch_awq_to_marlin(b_q_weight, out, experts, size_k, size_n, (hipStream_t)stream);
}

extern "C" int sonar_marlin_to_gfx950(const uint32_t* marlin, uint32_t* out, int64_t size_k,
                                      int64_t size_n, void* stream) {
  if (int rc = check_repack_shape(size_k, size_n, 4)) return rc;
  SONAR_REQUIRE(size_k % kChunkK == 0, "size_k = %ld is not divisible by %d", (long)size_k, kChunkK);
  SONAR_REQUIRE(marlin && out && marlin != out, "marlin and out must be distinct non-NULL buffers");
  const long total = size_k * size_n / 8;
  marlin_to_gfx950_kernel<<<grid_for(total), 256, 0, (hipStream_t)stream>>>(marlin, out, (int)size_k,
                                                                           (int)size_n, total);
  return launch_status("marlin_to_gfx950_kernel");
}

extern "C" int sonar_gfx950_to_marlin(const uint32_t* gfx950, uint32_t* out, int64_t size_k,
                                      int64_t size_n, void* stream) {
  if (int rc = check_repack_shape(size_k, size_n, 4)) return rc;
  SONAR_REQUIRE(size_k % kChunkK == 0, "size_k = %ld is not divisible by %d", (long)size_k, kChunkK);
  SONAR_REQUIRE(gfx950 && out && gfx950 != out, "gfx950 and out must be distinct non-NULL buffers");
  const long total = size_k * size_n / 8;
  gfx950_to_marlin_kernel<<<grid_for(total), 256, 0, (hipStream_t)stream>>>(gfx950, out, (int)size_k,
                                                                           (int)size_n, total);
  return launch_status("gfx950_to_marlin_kernel");
}

extern "C" int sonar_marlin8_to_gfx950(const uint32_t* marlin, uint32_t* out, int64_t size_k,
                                       int64_t size_n, void* stream) {
  if (int rc = check_repack_shape(size_k, size_n, 8)) return rc;
  SONAR_REQUIRE(size_k % kChunkK == 0, "size_k = %ld is not divisible by %d", (long)size_k, kChunkK);
  SONAR_REQUIRE(marlin && out && marlin != out, "marlin and out must be distinct non-NULL buffers");
  const long total = size_k * size_n / 4;
  marlin8_gfx950_kernel<true><<<grid_for(total), 256, 0, (hipStream_t)stream>>>(marlin, out, (int)size_k,
                                                                               (int)size_n, total);
  return launch_status("marlin8_gfx950_kernel");
}

extern "C" int sonar_gfx950_to_marlin8(const uint32_t* gfx950, uint32_t* out, int64_t size_k,
                                       int64_t size_n, void* stream) {
  if (int rc = check_repack_shape(size_k, size_n, 8)) return rc;
  SONAR_REQUIRE(size_k % kChunkK == 0, "size_k = %ld is not divisible by %d", (long)size_k, kChunkK);
  SONAR_REQUIRE(gfx950 && out && gfx950 != out, "gfx950 and out must be distinct non-NULL buffers");
  const long total = size_k * size_n / 4;
  marlin8_gfx950_kernel<false><<<grid_for(total), 256, 0, (hipStream_t)stream>>>(gfx950, out, (int)size_k,
                                                                                (int)size_n, total);
  return launch_status("marlin8_gfx950_kernel");
}

// ---- the weight order for 8-bit activations --------------------------------
namespace {
int check_a8_shape(int64_t size_k, int64_t size_n, int num_bits) {
  if (int rc = check_repack_shape(size_k, size_n, num_bits)) return rc;
  SONAR_REQUIRE(size_k % kA8Tile == 0, "size_k = %ld is not divisible by %d (the tile of 8-bit activations)",
                (long)size_k, kA8Tile);
  return SONAR_OK;
}
}  // namespace

extern "C" int sonar_gptq_marlin_repack_a8(const uint32_t* b_q_weight, uint32_t* out, int64_t size_k,
                                           int64_t size_n, int num_bits, void* stream) {
  if (int rc = check_a8_shape(size_k, size_n, num_bits)) return rc;
  SONAR_REQUIRE(b_q_weight && out, "b_q_weight and out must not be NULL");
  if (num_bits == 8) {
    const long words = size_k * size_n / 4;
    gptq8_to_marlin_a8_kernel<<<grid_for(words), 256, 0, (hipStream_t)stream>>>(b_q_weight, out, (int)size_k,
                                                                               (int)size_n, words);
    return launch_status("gptq8_to_marlin_a8_kernel");
  }
  const long total = size_k * size_n / 8;
  to_marlin_a8_kernel<0><<<grid_for(total), 256, 0, (hipStream_t)stream>>>(b_q_weight, out, (int)size_k,
                                                                          (int)size_n, total);
  return launch_status("to_marlin_a8_kernel");
}

extern "C" int sonar_awq_marlin_repack_a8(const uint32_t* b_q_weight, uint32_t* out, int64_t size_k,
                                          int64_t size_n, int num_bits, void* stream) {
  if (int rc = check_a8_shape(size_k, size_n, num_bits)) return rc;
  if (num_bits != 4) return fail(SONAR_E_UNSUPPORTED, "awq_marlin_repack: 8-bit AWQ weights are not built");
  SONAR_REQUIRE(b_q_weight && out, "b_q_weight and out must not be NULL");
  const long total = size_k * size_n / 8;
  to_marlin_a8_kernel<1><<<grid_for(total), 256, 0, (hipStream_t)stream>>>(b_q_weight, out, (int)size_k,
                                                                          (int)size_n, total);
  return launch_status("to_marlin_a8_kernel");
}

extern "C" int sonar_marlin_a8_to_gfx950(const uint32_t* marlin, uint32_t* out, int64_t size_k, int64_t size_n,
                                         void* stream) {
  if (int rc = check_a8_shape(size_k, size_n, 4)) return rc;
  SONAR_REQUIRE(marlin && out && marlin != out, "marlin and out must be distinct non-NULL buffers");
  const long total = size_k * size_n / 8;
  marlin_a8_to_gfx950_kernel<<<grid_for(total), 256, 0, (hipStream_t)stream>>>(marlin, out, (int)size_k,
                                                                              (int)size_n, total);
  return launch_status("marlin_a8_to_gfx950_kernel");
}

extern "C" int sonar_gfx950_to_marlin_a8(const uint32_t* gfx950, uint32_t* out, int64_t size_k, int64_t size_n,
                                         void* stream) {
  if (int rc = check_a8_shape(size_k, size_n, 4)) return rc;
  SONAR_REQUIRE(gfx950 && out && gfx950 != out, "gfx950 and out must be distinct non-NULL buffers");
  const long total = size_k * size_n / 8;
  to_marlin_a8_kernel<2><<<grid_for(total), 256, 0, (hipStream_t)stream>>>(gfx950, out, (int)size_k,
                                                                          (int)size_n, total);
  return launch_status("to_marlin_a8_kernel");
}

extern "C" int sonar_marlin_int4_fp8_preprocess(const uint32_t* qweight, const uint32_t* qzeros, uint32_t* out,
                                                int64_t rows, int64_t words_per_row, int64_t group_size,
                                                void* stream) {
  SONAR_REQUIRE(qweight && out, "qweight and out must not be NULL");
  SONAR_REQUIRE(rows > 0 && words_per_row > 0, "rows = %ld and words_per_row = %ld must be positive", (long)rows,
                (long)words_per_row);
  if (qzeros) {
    SONAR_REQUIRE(rows % 32 == 0, "size_k % 32 != 0");
    SONAR_REQUIRE(group_size > 0 && rows % group_size == 0, "qweight.size(0) % qzeros.size(0) != 0");
    SONAR_REQUIRE(group_size % 8 == 0, "group_size % 8 != 0");
  } else {
    SONAR_REQUIRE(rows * words_per_row * 8 % 256 == 0, "qweight.numel() * 8 % 256 != 0");
    group_size = 1;
  }
  const long total = rows * words_per_row;
  int4_fp8_preprocess_kernel<<<grid_for(total), 256, 0, (hipStream_t)stream>>>(qweight, qzeros, out, words_per_row,
                                                                              (int)group_size, total);
  return launch_status("int4_fp8_preprocess_kernel");
}

// ---- checkpoint tensors around the codes -----------------------------------
namespace {
int blocks_of(int64_t items) { return (int)((items + 255) / 256); }
}  // namespace

extern "C" int sonar_marlin_permute_scales(const void* in, void* out, int64_t numel, int grouped, void* stream) {
  SONAR_REQUIRE(numel >= 0 && numel % (grouped ? 64 : 32) == 0 && numel < (1LL << 38),
                "the number of scales = %ld must be a multiple of %d", (long)numel, grouped ? 64 : 32);
  if (numel == 0) return SONAR_OK;
  SONAR_REQUIRE(in && out && in != out, "in and out must be distinct non-NULL buffers");
  SONAR_REQUIRE((uintptr_t)out % 16 == 0, "out must be 16-byte aligned");
  auto* kernel = grouped ? permute_scale_columns<true> : permute_scale_columns<false>;
  kernel<<<blocks_of(numel / 8), 256, 0, (hipStream_t)stream>>>(static_cast<const uint16_t*>(in),
                                                               static_cast<uint16_t*>(out), numel / 8);
  return launch_status("permute_scale_columns");
}

extern "C" int sonar_marlin_pack_zero_points(const uint32_t* in, uint32_t* out, int64_t rows, int64_t size_n,
                                             int64_t row_stride, int64_t word_stride, int awq_order, int is_a_8bit,
                                             void* stream) {
  SONAR_REQUIRE(rows >= 0 && size_n > 0 && size_n % 64 == 0 && size_n < (1LL << 30),
                "size_n = %ld is not a positive multiple of 64", (long)size_n);
  const int64_t total = rows * (size_n / 8);
  SONAR_REQUIRE(total < (1LL << 38), "too many zero points");
  if (total == 0) return SONAR_OK;
  SONAR_REQUIRE(in && out && in != out, "in and out must be distinct non-NULL buffers");
  pack_zero_points<<<blocks_of(total), 256, 0, (hipStream_t)stream>>>(in, out, (int)(size_n / 8), total, row_stride,
                                                                     word_stride, awq_order != 0, is_a_8bit != 0);
  return launch_status("pack_zero_points");
}

static int load_linear(const uint32_t* codes, uint32_t* codes_out, const void* scales, void* scales_out, const uint32_t* zeros,
                       uint32_t* zeros_out, uint32_t* workspace, int64_t workspace_words, int64_t size_k, int64_t size_n,
                       int64_t groups, int grouped, int zeros_transposed, const int32_t* perm, void* stream) {
  if (int rc = check_repack_shape(size_k, size_n, 4)) return rc;
  if (int rc = check_experts(1, size_k, size_n)) return rc;
  SONAR_REQUIRE(groups >= 1 && groups * size_n < (1LL << 38), "num_groups = %ld out of range", (long)groups);
  SONAR_REQUIRE(codes && codes_out && codes != codes_out && scales && scales_out && scales != scales_out,
                "codes, scales and their outputs must be distinct non-NULL buffers");
  SONAR_REQUIRE((zeros == nullptr) == (zeros_out == nullptr) && (zeros == nullptr || zeros != zeros_out),
                "zero points and their output must be given together, as distinct buffers");
  SONAR_REQUIRE(workspace_words >= 0 && workspace_words < (1LL << 20) && (workspace || workspace_words == 0),
                "workspace of %ld words is out of range", (long)workspace_words);
  SONAR_REQUIRE((uintptr_t)scales_out % 16 == 0, "out must be 16-byte aligned");
  LoadLinear p = {};
  p.codes = codes;
  p.codes_out = codes_out;
  p.size_k = (int)size_k;
  p.size_n = (int)size_n;
  p.tiles = (uint32_t)((size_k / kMarlinTileK) * (size_n / kMarlinTileN));
  p.code_blocks = (p.tiles + kRepackTiles - 1) / kRepackTiles;
  p.scales = static_cast<const uint16_t*>(scales);
  p.scales_out = static_cast<uint16_t*>(scales_out);
  p.vectors = groups * size_n / 8;
  p.scale_blocks = (uint32_t)((p.vectors + 255) / 256);
  if (zeros) {
    p.zeros = zeros;
    p.zeros_out = zeros_out;
    p.zero_words = groups * (size_n / 8);
    p.zero_row_stride = zeros_transposed ? 1 : size_n / 8;
    p.zero_word_stride = zeros_transposed ? groups : 1;
    p.zero_blocks = (uint32_t)((p.zero_words + 255) / 256);
  }
  p.workspace = workspace;
  p.workspace_words = (int)workspace_words;
  const int64_t blocks = (int64_t)p.code_blocks + p.scale_blocks + p.zero_blocks + (workspace_words > 0);
  SONAR_REQUIRE(blocks < (1LL << 31), "weight too large");
  p.perm = perm;
  auto* kernel = perm ? (grouped ? load_linear_kernel<true, true> : load_linear_kernel<false, true>)
                      : (grouped ? load_linear_kernel<true, false> : load_linear_kernel<false, false>);
  kernel<<<(int)blocks, 256, 0, (hipStream_t)stream>>>(p);
  return launch_status("load_linear_kernel");
}

extern "C" int sonar_load_gptq_linear(const uint32_t* codes, uint32_t* codes_out, const void* scales, void* scales_out,
                                      const uint32_t* zeros, uint32_t* zeros_out, uint32_t* workspace,
                                      int64_t workspace_words, int64_t size_k, int64_t size_n, int64_t groups, int grouped,
                                      int zeros_transposed, void* stream) {
  return load_linear(codes, codes_out, scales, scales_out, zeros, zeros_out, workspace, workspace_words, size_k, size_n, groups, grouped,
                     zeros_transposed, nullptr, stream);
}

extern "C" int sonar_sort_g_idx(const int32_t* g_idx, int32_t* sorted, int32_t* order, int64_t size_k, void* stream) {
  SONAR_REQUIRE(size_k >= 0 && size_k <= (1 << 20), "size_k = %ld out of range", (long)size_k);
  if (size_k == 0) return SONAR_OK;
  SONAR_REQUIRE(g_idx && sorted && order && g_idx != sorted && g_idx != order && sorted != order,
                "g_idx and its outputs must be distinct non-NULL buffers");
  sort_group_indices<<<(int)((size_k + 63) / 64), 64 * kSortWaves, 0, (hipStream_t)stream>>>(g_idx, sorted, order, (int)size_k);
  return launch_status("sort_group_indices");
}

extern "C" int sonar_load_gptq_act_order(const uint32_t* codes, uint32_t* codes_out, const void* scales, void* scales_out,
                                         const int32_t* g_idx, int32_t* g_idx_out, int32_t* order, uint32_t* workspace,
                                         int64_t workspace_words, int64_t size_k, int64_t size_n, int64_t groups, int grouped,
                                         void* stream) {
  if (int rc = check_repack_shape(size_k, size_n, 4)) return rc;
  if (int rc = sonar_sort_g_idx(g_idx, g_idx_out, order, size_k, stream)) return rc;
  return load_linear(codes, codes_out, scales, scales_out, nullptr, nullptr, workspace, workspace_words, size_k, size_n, groups, grouped, 0,
                     order, stream);
}

extern "C" int sonar_awq_to_gptq(const uint32_t* in, uint32_t* out, int64_t size_k, int64_t size_n, void* stream) {
  SONAR_REQUIRE(size_k >= 0 && size_n > 0 && size_k % 8 == 0 && size_n % 8 == 0 && size_n < (1LL << 30) &&
                    size_k < (1LL << 30), "size_k = %ld and size_n = %ld must be multiples of 8", (long)size_k, (long)size_n);
  const int64_t total = size_k / 8 * (size_n / 8);
  SONAR_REQUIRE(total < (1LL << 38), "weight too large");
  if (total == 0) return SONAR_OK;
  SONAR_REQUIRE(in && out && in != out, "in and out must be distinct non-NULL buffers");
  return launch_awq_to_plain({in, out, nullptr, nullptr, (int)(size_n / 8), 0, total, 0, 0}, (hipStream_t)stream);
}

extern "C" int sonar_awq_to_standard(const uint32_t* codes, uint32_t* codes_out, const uint32_t* zeros, uint32_t* zeros_out,
                                     int64_t size_k, int64_t size_n, int64_t groups, void* stream) {
  SONAR_REQUIRE(size_k >= 0 && size_n > 0 && size_k % 8 == 0 && size_n % 8 == 0 && size_n < (1LL << 30) && size_k < (1LL << 30) &&
                    groups >= 0 && groups < (1LL << 30), "size_k = %ld and size_n = %ld must be multiples of 8", (long)size_k, (long)size_n);
  const int64_t code_words = size_k / 8 * (size_n / 8), zero_words = groups * (size_n / 8);
  SONAR_REQUIRE(code_words < (1LL << 38) && zero_words < (1LL << 38), "weight too large");
  SONAR_REQUIRE((code_words == 0 || (codes && codes_out && codes != codes_out)) &&
                    (zero_words == 0 || (zeros && zeros_out && zeros != zeros_out)), "inputs and outputs must be distinct non-NULL buffers");
  if (code_words + zero_words == 0) return SONAR_OK;
  return launch_awq_to_plain({codes, codes_out, zeros, zeros_out, (int)(size_n / 8), (int)groups, code_words, zero_words, 0},
                             (hipStream_t)stream);
}

extern "C" int sonar_awq_zeros_to_plain(const uint32_t* in, uint32_t* out, int64_t groups, int64_t size_n,
                                        void* stream) {
  SONAR_REQUIRE(groups >= 0 && size_n > 0 && size_n % 8 == 0 && size_n < (1LL << 30) && groups < (1LL << 30),
                "size_n = %ld must be a positive multiple of 8", (long)size_n);
  const int64_t total = groups * (size_n / 8);
  SONAR_REQUIRE(total < (1LL << 38), "too many zero points");
  if (total == 0) return SONAR_OK;
  SONAR_REQUIRE(in && out && in != out, "in and out must be distinct non-NULL buffers");
  return launch_awq_to_plain({nullptr, nullptr, in, out, (int)(size_n / 8), (int)groups, 0, total, 0}, (hipStream_t)stream);
}
