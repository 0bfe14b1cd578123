// The gated activations that both moe_aux.hip's kernels and the epilogue of the grouped tile kernels form: of the 16-bit
// bits of a gate and an up value, with the roundings of the reference's kernels.
#pragma once

#include "common.hpp"

namespace sonar {

template <typename T>
__device__ __forceinline__ float to_f32(uint16_t b);
template <>
__device__ __forceinline__ float to_f32<_Float16>(uint16_t b) { return (float)__builtin_bit_cast(_Float16, b); }
template <>
__device__ __forceinline__ float to_f32<__bf16>(uint16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }
template <typename T>
__device__ __forceinline__ uint16_t from_f32(float f) { return __builtin_bit_cast(uint16_t, (T)f); }

// n / (1 + e) for e in [0, inf]: what the division of two floats gives, in 6 instructions instead of 11, because the denominator
// needs no scaling of its own (a quarter of both keeps its reciprocal a normal number).  Infinities and NaN as in the division.
__device__ __forceinline__ float over_one_plus(float n, float e) {
  const float d = __builtin_fmaf(e, 0.25f, 0.25f), m = n * 0.25f;
  const float r = __builtin_amdgcn_rcpf(d), q = m * r;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-d, q, m), r, q), d, m);
}

// silu_and_mul: T(T(silu(gate)) * up)
template <typename T>
__device__ __forceinline__ uint16_t silu_times(uint16_t gate_bits, uint16_t up_bits) {
  const float x = to_f32<T>(gate_bits);
  const float s = to_f32<T>(from_f32<T>(over_one_plus(x, __expf(-x))));
  return from_f32<T>(s * to_f32<T>(up_bits));
}

// swigluoai_and_mul: T((u + 1) g / (1 + exp(-alpha g))), g = min(gate, limit), u = clamp(up, -limit, limit).  The power of two
// takes -alpha log2(e) g with what its rounding leaves, so that the exponential is as close as expf's (which spends twice the
// instructions).  Against expf and a division: 51 -> 39 instructions a result in the kernel of moe_aux.hip; the same relative error
// against 64 bits (fp16 2.07e-4, bf16 1.66e-3), 8 of 1048576 results in a tie rounded the other way.
template <typename T>
__device__ __forceinline__ uint16_t swiglu_oai(uint16_t gate_bits, uint16_t up_bits, float limit, float alpha) {
  constexpr float kLog2e = 1.44269504f, kLog2eRest = 1.92596303e-8f, kLn2 = 0.693147181f;
  const float hi = -alpha * kLog2e, lo = __builtin_fmaf(-alpha, kLog2e, -hi) - alpha * kLog2eRest;   // (a launch's constants)
  const float g = fminf(to_f32<T>(gate_bits), limit);
  const float u = fmaxf(fminf(to_f32<T>(up_bits), limit), -limit);
  const float t = g * hi;
  const float rest = __builtin_fmaf(g, lo, __builtin_fmaf(g, hi, -t));
  // (Where the power of two is 0 or infinite it is the exponential; `rest` is no small number there, but large, infinite or NaN:
  // the minimum and the absolute value keep the product 0 or infinite.)
  const float correction = fminf(__builtin_fmaf(rest, kLn2, 1.0f), 2.0f);
  return from_f32<T>(over_one_plus((u + 1.0f) * g, fabsf(__builtin_amdgcn_exp2f(t) * correction)));
}

// Where a grouped GEMM may leave its activation instead of its result.
struct GatedOutput {
  void* out;             // (rows, size_n / 2) of the 16-bit type
  int kind;              // 0: silu_and_mul (gate half, up half); SONAR_ACT_SWIGLUOAI (gate and up alternate)
  float limit, alpha;    // of SONAR_ACT_SWIGLUOAI
  bool done;             // set by a call that wrote `out`, which then left c as it was
};
// Whether a kernel whose workgroups have whole strips of 64 columns can form it: rows of 8-byte stores, as many strips of the gate half
// as of the up half.
inline bool gated_by_strips(const GatedOutput* g, int64_t size_n) {
  return g != nullptr && ((uintptr_t)g->out) % 8 == 0 &&
         (g->kind == 0 ? size_n % 128 == 0 : g->kind == SONAR_ACT_SWIGLUOAI && g->limit > 0.f);
}

// What one grouped GEMM of a layer may do for another one of the same routing, or have had done for it.
struct MoeLayerCall {
  GatedOutput* gated = nullptr;
  sonar_moe_tables* next = nullptr;          // build the row tiles of that GEMM in this call's launch
  sonar_moe_tables* ready = nullptr;         // this GEMM's, if an earlier call has built them
  const int32_t* topk_ids = nullptr;         // the expert of every row of C, in place of the sorted slots
};

}  // namespace sonar
