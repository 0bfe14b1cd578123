// Per-token (per-row) quantisation of the activations for the W4A8 GEMM: one
// fp32 scale per row and int8 or float8_e4m3fn codes.  The int8 kernel follows
// aphrodite/model_executor/layers/quantization/utils/int8_utils.py:70-93, the
// fp8 one QuantFP8(False, GroupShape.PER_TOKEN)
// (layers/quantization/input_quant_fp8.py:188-204).  One workgroup per row:
// the maximum magnitude first, then the codes.  Every step rounds to fp32 as
// written.  Bound by the bytes of the rows, or, for a few rows, by the latency of
// a load, the maximum over the workgroup and two divisions.
#include "common.hpp"

namespace sonar {
namespace {

template <typename T>
__device__ __forceinline__ float load_as_float(const T* p, long i) { return (float)p[i]; }

__device__ __forceinline__ float block_max(float v) {
  __shared__ float part[4];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  return fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
}

// One fp32 value -> its code, rounded as the references do.
template <bool FP8>
__device__ __forceinline__ float scaled_value(float x, float by) {
#pragma clang fp contract(off)
  const float y = x * by;
  return FP8 ? fminf(fmaxf(y, -448.0f), 448.0f) : copysignf(floorf(fabsf(y) + 0.5f), y);   // halves away from zero
}

// Eight columns from one aligned address.
template <typename T>
struct Eight {
  static constexpr int kVecs = sizeof(T) / 2;   // 16-byte loads
  uint4 v[kVecs];
  __device__ __forceinline__ void load(const T* p) {
#pragma unroll
    for (int i = 0; i < kVecs; ++i) v[i] = reinterpret_cast<const uint4*>(p)[i];
  }
  __device__ __forceinline__ float at(int i) const {
    typedef T eight_t __attribute__((ext_vector_type(8)));
    return (float)__builtin_bit_cast(eight_t, *this)[i];
  }
};

// `vec`: rows and codes are aligned for eight columns at a time; a thread then asks for all its parts of the row at
// once (up to eight: 16384 columns of 16-bit numbers) and keeps them for the second pass.  Element by element -> now,
// int8 codes of fp16 rows: 1 x 4096 4.5 -> 2.5 us, 1 x 14336 11.8 -> 3.9, 2048 x 4096 8.6 -> 6.1, 8192 x 8192
// 71.9 -> 31.7 (6.3 TB/s).
template <typename T, bool FP8>
__global__ __launch_bounds__(256) void per_token_quant_kernel(const T* __restrict__ x, long row_stride,
                                                             uint8_t* __restrict__ q, float* __restrict__ scales,
                                                             const float* __restrict__ factor, int cols, bool vec) {
#pragma clang fp contract(off)
  constexpr int kKept = 8 / Eight<T>::kVecs;
  const T* row = x + (long)blockIdx.x * row_stride;
  uint8_t* out = q + (long)blockIdx.x * cols;
  const int step = 256 * 8, first = threadIdx.x * 8;
  Eight<T> kept[kKept];
  float m = 0.0f;
  if (vec) {
#pragma unroll
    for (int i = 0; i < kKept; ++i)
      if (first + i * step < cols) kept[i].load(row + first + i * step);
#pragma unroll
    for (int i = 0; i < kKept; ++i)
      if (first + i * step < cols) {
#pragma unroll
        for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(kept[i].at(e)));
      }
    for (int c = first + kKept * step; c < cols; c += step) {
      Eight<T> v;
      v.load(row + c);
#pragma unroll
      for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(v.at(e)));
    }
  } else {
    for (int i = threadIdx.x; i < cols; i += 256) m = fmaxf(m, fabsf(load_as_float(row, i)));
  }
  m = block_max(m);
  float by;
  if (FP8) {
    const float scale = fmaxf(m / 448.0f, 1.0f / (448.0f * 512.0f));
    by = 1.0f / scale;
    if (threadIdx.x == 0) scales[blockIdx.x] = factor ? scale * factor[0] : scale;
  } else {
    const float absmax = fmaxf(m, 1e-10f);
    by = 127.0f / absmax;
    const float scale = absmax / 127.0f;
    if (threadIdx.x == 0) scales[blockIdx.x] = factor ? scale * factor[0] : scale;
  }
  if (!vec) {
    for (int i = threadIdx.x; i < cols; i += 256) {
      const float y = scaled_value<FP8>(load_as_float(row, i), by);
      out[i] = FP8 ? (uint8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(y, 0.0f, 0, false) & 0xff) : (uint8_t)(int8_t)(int)y;
    }
    return;
  }
  auto store = [&](const Eight<T>& v, int c) {
    uint32_t word[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = scaled_value<FP8>(v.at(4 * h + e), by);
      if (FP8) {
        const int low = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false);
        word[h] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], low, true);
      } else {
        word[h] = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) word[h] |= (uint32_t)((int)y[e] & 0xff) << (8 * e);
      }
    }
    *reinterpret_cast<uint2*>(out + c) = make_uint2(word[0], word[1]);
  };
#pragma unroll
  for (int i = 0; i < kKept; ++i)
    if (first + i * step < cols) store(kept[i], first + i * step);
  for (int c = first + kKept * step; c < cols; c += step) {
    Eight<T> v;
    v.load(row + c);
    store(v, c);
  }
}

template <bool FP8>
int launch_quant(const void* x, int dtype, int64_t row_stride, uint8_t* q, float* scales, const float* factor,
                 int64_t rows, int64_t cols, void* stream) {
  SONAR_REQUIRE(rows >= 0 && cols > 0 && cols < (1LL << 31) && rows < (1LL << 31), "rows = %ld, cols = %ld",
                (long)rows, (long)cols);
  SONAR_REQUIRE(row_stride >= cols, "row_stride = %ld is smaller than cols = %ld", (long)row_stride, (long)cols);
  if (rows == 0) return SONAR_OK;
  SONAR_REQUIRE(x && q && scales, "x, q and scales must not be NULL");
  hipStream_t st = (hipStream_t)stream;
  const int64_t bytes = dtype == SONAR_DTYPE_F32 ? 4 : 2;
  const bool vec = cols % 8 == 0 && (uintptr_t)x % 16 == 0 && row_stride * bytes % 16 == 0 && (uintptr_t)q % 8 == 0;
  if (dtype == SONAR_DTYPE_F16)
    per_token_quant_kernel<_Float16, FP8><<<(int)rows, 256, 0, st>>>((const _Float16*)x, row_stride, q, scales, factor, (int)cols, vec);
  else if (dtype == SONAR_DTYPE_BF16)
    per_token_quant_kernel<__bf16, FP8><<<(int)rows, 256, 0, st>>>((const __bf16*)x, row_stride, q, scales, factor, (int)cols, vec);
  else if (dtype == SONAR_DTYPE_F32)
    per_token_quant_kernel<float, FP8><<<(int)rows, 256, 0, st>>>((const float*)x, row_stride, q, scales, factor, (int)cols, vec);
  else
    return fail(SONAR_E_INVALID, "unknown dtype = %d", dtype);
  return launch_status("per_token_quant_kernel");
}

}  // namespace
}  // namespace sonar

using namespace sonar;

extern "C" int sonar_per_token_quant_int8(const void* x, int dtype, int64_t row_stride, int8_t* q, float* scales,
                                          int64_t rows, int64_t cols, void* stream) {
  return launch_quant<false>(x, dtype, row_stride, (uint8_t*)q, scales, nullptr, rows, cols, stream);
}

extern "C" int sonar_per_token_quant_int8_scaled(const void* x, int dtype, int64_t row_stride, int8_t* q,
                                                 float* scales, const float* factor, int64_t rows, int64_t cols,
                                                 void* stream) {
  return launch_quant<false>(x, dtype, row_stride, (uint8_t*)q, scales, factor, rows, cols, stream);
}

extern "C" int sonar_per_token_quant_fp8(const void* x, int dtype, int64_t row_stride, uint8_t* q, float* scales,
                                         int64_t rows, int64_t cols, void* stream) {
  return launch_quant<true>(x, dtype, row_stride, q, scales, nullptr, rows, cols, stream);
}
