// The small kernels that bracket the two grouped GEMMs of a mixture-of-experts
// layer: routing of (token, k) slots into per-expert blocks, the gated
// activation, and the sum over a token's experts.  They restate
// csrc/libtorch_stable/moe/moe_align_sum_kernels.cu:626-725,759+ and the
// silu_and_mul of csrc/libtorch_stable/activation_kernels.cu for fp16 / bf16.
#include <algorithm>

#include "common.hpp"
#include "moe_activation.hpp"

namespace sonar {
namespace {

constexpr int kAlignThreads = 1024;
constexpr int kAlignWaves = kAlignThreads / 64;
// Experts up to which one launch counts and places: a workgroup's wavefronts keep a histogram each (54 KiB of LDS with two more).
constexpr int kAlignOneLaunchExperts = 768;
// Workgroups of a launch: one up to 5000 slots (counting the other segments costs one more round trip; us, one workgroup against
// one for every 1024 slots, back to back: 2508 slots, 8 experts 5.5 / 6.9, 4000 6.1 / 6.9, 8192 8.8 / 7.3, 8000 on 32 9.2 / 7.3, 32000
// on 64 31.6 / 9.5, 65536 on 256 67.6 / 12.7), and up to 64, after which they take longer segments (131072 on 64: 114 -> 20).
constexpr int kAlignOneWorkgroup = 5000, kAlignMost = 64;

// Inclusive sum over the lanes of a wavefront.
__device__ __forceinline__ int wave_inclusive_sum(int v) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(v, d, 64);
    if ((int)(threadIdx.x & 63) >= d) v += up;
  }
  return v;
}

// Per-expert counts, padded offsets, expert id of every block, the padded total and
// the sentinels of sorted_token_ids.  With `place` it also places the slots: every wavefront owns
// a contiguous share of its workgroup's and a histogram row; the rows' prefix sums give each wavefront its first
// position per expert, and inside 64 slots a lane's rank among the lanes of the same expert comes from
// one ballot per bit of the expert number, so the slots of an expert keep ascending order.  Without it
// (more experts than the histograms have room for) offsets[e] is left for the placement kernel.
// Several workgroups take a segment of the slots each and count all of them: two more rows hold what lies before and behind the
// segment, so that nobody waits for another, and placing, whose scattered stores one compute unit takes long for, is spread.
// Latency bound with few slots, which one workgroup takes (kAlignOneWorkgroup); with many by their counting.  8000 slots on 32
// experts: 9 + 42 us as two launches whose second walked all slots once per expert, 9.2 in one workgroup (eight rounds of slots
// read at a time and, up to 8192 slots, once), 7.3 like this; a layer of 4000 tokens on 64 experts, top 8 427 -> 404.
__host__ __device__ __forceinline__ int align_share(int numel, int workgroups) {   // slots of a wavefront
  const int per_wave = (int)(((long)numel + (long)workgroups * kAlignWaves - 1) / ((long)workgroups * kAlignWaves));
  return (per_wave + 63) / 64 * 64;
}
template <int kBatch>
__global__ __launch_bounds__(kAlignThreads) void moe_align_count_kernel(
    const int32_t* __restrict__ topk_ids, int numel, int num_experts, int block_size,
    int32_t* __restrict__ sorted_ids, int sorted_len, int32_t* __restrict__ expert_ids, int expert_len,
    int32_t* __restrict__ num_post_pad, const int32_t* __restrict__ expert_map, int32_t* __restrict__ offsets,
    bool place) {
  extern __shared__ int32_t lds[];     // begin[num_experts + 1], stop[num_experts], wave totals, the histogram rows
  int32_t* begin = lds;
  int32_t* stop = begin + num_experts + 1;   // where an expert's slots end and its padding begins
  int32_t* wave_sum = stop + num_experts;
  int32_t* hist = wave_sum + kAlignWaves;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int many = gridDim.x > 1 ? 1 : 0;   // rows of the histogram: slots before the segment, the wavefronts' shares, slots behind
  const int rows = place ? kAlignWaves + 2 * many : 1;
  for (int i = tid; i < rows * num_experts; i += kAlignThreads) hist[i] = 0;
  __syncthreads();
  // The experts (-1: none) of up to kBatch rounds of 64 slots from `base` on, all asked for before the first is waited for.
  int held[kBatch];
  auto fetch = [&](int base, int end) {
#pragma unroll
    for (int r = 0; r < kBatch; ++r) {
      held[r] = -1;
      if (base + 64 * r < end && base + 64 * r + lane < end) held[r] = topk_ids[base + 64 * r + lane];
    }
#pragma unroll
    for (int r = 0; r < kBatch; ++r) {
      if (base + 64 * r >= end) break;
      if (held[r] < 0 || held[r] >= num_experts) held[r] = -1;
      else if (expert_map) held[r] = expert_map[held[r]];
      if (held[r] >= num_experts) held[r] = -1;   // (and none of a map's negative ones)
    }
  };
  // a wavefront's share of the segment: whole rounds of 64 slots
  const int share = align_share(numel, gridDim.x);
  const int segment = min(numel, (int)blockIdx.x * kAlignWaves * share), segment_end = min(numel, segment + kAlignWaves * share);
  const int from = min(segment_end, segment + wave * share), to = min(segment_end, from + share);
  int32_t* mine = hist + (place ? (many + wave) * num_experts : 0);
  if (many) {
    // the other slots, in any order, four a load where topk_ids lies so
    const bool vectors = (reinterpret_cast<uintptr_t>(topk_ids) & 15) == 0;
    auto count_others = [&](int lo, int hi, int32_t* row) {
      for (int base = lo; base < hi; base += 16 * kAlignThreads) {
        int4 v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int at = base + 4 * (kAlignThreads * r + tid);
          if (vectors && at + 4 <= hi) {
            v[r] = *reinterpret_cast<const int4*>(topk_ids + at);
          } else {
            v[r].x = at < hi ? topk_ids[at] : -1;
            v[r].y = at + 1 < hi ? topk_ids[at + 1] : -1;
            v[r].z = at + 2 < hi ? topk_ids[at + 2] : -1;
            v[r].w = at + 3 < hi ? topk_ids[at + 3] : -1;
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int e4[4] = {v[r].x, v[r].y, v[r].z, v[r].w};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            int e = e4[j];
            if (e < 0 || e >= num_experts) continue;
            if (expert_map) e = expert_map[e];
            if (e >= 0 && e < num_experts) atomicAdd(&row[e], 1);
          }
        }
      }
    };
    count_others(0, segment, hist);
    count_others(segment_end, numel, hist + (kAlignWaves + 1) * num_experts);
  }
  for (int base = from; base < to; base += 64 * kBatch) {
    fetch(base, to);
#pragma unroll
    for (int r = 0; r < kBatch; ++r) {
      if (base + 64 * r >= to) break;
      if (held[r] >= 0) atomicAdd(&mine[held[r]], 1);
    }
  }
  __syncthreads();
  // padded run of every expert -> where it begins
  int carry = 0;
  for (int base = 0; base < num_experts; base += kAlignThreads) {
    const int e = base + tid;
    int count = 0, padded = 0;
    if (e < num_experts) {
      for (int r = 0; r < rows; ++r) {
        const int c = hist[r * num_experts + e];
        hist[r * num_experts + e] = count;   // slots of this expert in earlier shares
        count += c;
      }
      padded = (count + block_size - 1) / block_size * block_size;
    }
    const int incl = wave_inclusive_sum(padded);
    if (lane == 63) wave_sum[wave] = incl;
    __syncthreads();
    int before = carry;
    for (int w = 0; w < kAlignWaves; ++w) {
      const int t = wave_sum[w];
      if (w < wave) before += t;
      carry += t;
    }
    if (e < num_experts) {
      begin[e] = before + incl - padded;
      stop[e] = begin[e] + count;
    }
    __syncthreads();
  }
  const int total = carry;
  if (tid == 0) {
    begin[num_experts] = total;
    if (blockIdx.x == 0) num_post_pad[0] = total;
  }
  __syncthreads();
  // sentinels: behind every expert's slots and behind the last run (each workgroup some of them, and of the blocks)
  const int all_waves = gridDim.x * kAlignWaves, all_threads = gridDim.x * kAlignThreads;
  for (int e = blockIdx.x * kAlignWaves + wave; e < num_experts; e += all_waves)
    for (int i = stop[e] + lane; i < begin[e + 1]; i += 64) sorted_ids[i] = numel;
  for (int i = total + blockIdx.x * kAlignThreads + tid; i < sorted_len; i += all_threads) sorted_ids[i] = numel;
  if (!place)
    for (int e = tid; e < num_experts; e += kAlignThreads) offsets[e] = begin[e];
  for (int b = blockIdx.x * kAlignThreads + tid; b < expert_len; b += all_threads) {
    const int start = b * block_size;
    int e = -1;
    if (start < total) {
      // last expert whose run begins at or before `start` and is not empty there
      int lo = 0, hi = num_experts - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (begin[mid] <= start) lo = mid; else hi = mid - 1;
      }
      e = lo;
    }
    expert_ids[b] = e;
  }
  if (!place) return;
  const int bits = 32 - __clz(num_experts);   // the number of experts itself stands for "none"
  for (int base = from; base < to; base += 64 * kBatch) {
    if (to - from > 64 * kBatch) fetch(base, to);   // else still held from the counting
#pragma unroll
    for (int r = 0; r < kBatch; ++r) {
      if (base + 64 * r >= to) break;
      const int i = base + 64 * r + lane;
      const int e = held[r] < 0 ? num_experts : held[r];
      unsigned long long same = ~0ull;
      for (int bit = 0; bit < bits; ++bit) {
        const bool set = (e >> bit) & 1;
        const unsigned long long m = __ballot(set);
        same &= set ? m : ~m;
      }
      if (e < num_experts) {
        const int at = mine[e];   // read by every lane of the expert before its last one moves it on
        sorted_ids[begin[e] + at + __popcll(same & ((1ull << lane) - 1ull))] = i;
        if ((same >> lane) == 1ull) mine[e] = at + __popcll(same);
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// One wavefront per expert walks the slots in order; a ballot gives every
// matching lane its rank, so the slots of an expert keep ascending order.
__global__ __launch_bounds__(256) void moe_align_place_kernel(const int32_t* __restrict__ topk_ids, int numel,
                                                             int num_experts,
                                                             int32_t* __restrict__ sorted_ids,
                                                             const int32_t* __restrict__ expert_map,
                                                             const int32_t* __restrict__ offsets) {
  const int lane = threadIdx.x & 63;
  const int expert = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (expert >= num_experts) return;
  int at = offsets[expert];
  for (int base = 0; base < numel; base += 64) {
    const int i = base + lane;
    int e = -1;
    if (i < numel) {
      e = topk_ids[i];
      if (e >= 0 && e < num_experts && expert_map) e = expert_map[e];
    }
    const bool mine = e == expert;
    const unsigned long long mask = __ballot(mine);
    if (mine) sorted_ids[at + __popcll(mask & ((1ull << lane) - 1ull))] = i;
    at += __popcll(mask);
  }
}

// out[r][c] = T(T(silu(x[r][c])) * x[r][d + c]): the activation is rounded to
// the tensor type before the product, as act_and_mul does.
template <typename T>
__global__ __launch_bounds__(256) void silu_and_mul_kernel(uint16_t* __restrict__ out,
                                                          const uint16_t* __restrict__ in, long rows, int d) {
  const long vec_per_row = d / 8;
  const long total = rows * vec_per_row;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const long r = i / vec_per_row;
    const int c = (int)(i - r * vec_per_row) * 8;
    const uint4 g = *reinterpret_cast<const uint4*>(in + r * 2 * d + c);
    const uint4 u = *reinterpret_cast<const uint4*>(in + r * 2 * d + d + c);
    const uint32_t gw[4] = {g.x, g.y, g.z, g.w}, uw[4] = {u.x, u.y, u.z, u.w};
    uint32_t ow[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      uint32_t o = 0;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        o |= (uint32_t)silu_times<T>((uint16_t)(gw[w] >> (16 * h)), (uint16_t)(uw[w] >> (16 * h))) << (16 * h);
      }
      ow[w] = o;
    }
    *reinterpret_cast<uint4*>(out + r * d + c) = make_uint4(ow[0], ow[1], ow[2], ow[3]);
  }
}

// The gated activations of the fused mixture-of-experts layer other than plain SiLU
// (aphrodite/model_executor/layers/fused_moe/activation.py:128-205 of the reference; the
// arithmetic of csrc/libtorch_stable/activation_kernels.cu:28-95,154-215,412-423,489-510 and of
// the Triton kernel aphrodite/model_executor/layers/activation.py:27-52), one (gate, up) pair
// -> one output, every intermediate rounding where the reference has one:
//   kClampSilu  silu_and_mul_with_clamp: g = T(min(gate, limit)), u = clamp(up, -limit, limit);
//               T(float(T(g / (1 + exp(-alpha g)))) * (u + beta))
//   kGelu       T(float(T(0.5 g (1 + erf(g / sqrt 2)))) * up);  kGeluTanh: the tanh form
//   kSwigluOai  gate / up interleaved in the input: g = min(gate, limit), u = clamp(up, +-limit);
//               T((u + 1) * g / (1 + exp(-alpha g)))
//   kSitu       T(beta tanh(gate / beta) / (1 + exp(-gate)) * (linear_beta > 0 ? linear_beta tanh(up / linear_beta) : up))
//               (beta in `alpha`, linear_beta in `beta`)
//   kSwigluStep T(min(gate * sigmoid(gate), limit) * clamp(up, -limit, limit))
enum MoeActivation { kClampSilu = 1, kGelu = 2, kGeluTanh = 3, kSwigluOai = 4, kSitu = 5, kSwigluStep = 6 };

template <typename T, int KIND>
__device__ __forceinline__ uint16_t gated_activation(uint16_t gate_bits, uint16_t up_bits, float limit, float alpha,
                                                     float beta) {
  const float gate = to_f32<T>(gate_bits), up = to_f32<T>(up_bits);
  if constexpr (KIND == kClampSilu) {
    const float g = to_f32<T>(from_f32<T>(fminf(gate, limit)));
    const float u = fmaxf(fminf(up, limit), -limit);
    const float act = to_f32<T>(from_f32<T>(g / (1.0f + expf(-g * alpha))));
    return from_f32<T>(act * (u + beta));
  } else if constexpr (KIND == kGelu) {
    const float act = to_f32<T>(from_f32<T>(gate * 0.5f * (1.0f + erff(gate * 0.70710678118654752440f))));
    return from_f32<T>(act * up);
  } else if constexpr (KIND == kGeluTanh) {
    const float inner = 0.79788456080286535588f * (gate + 0.044715f * (gate * gate * gate));
    const float act = to_f32<T>(from_f32<T>(0.5f * gate * (1.0f + tanhf(inner))));
    return from_f32<T>(act * up);
  } else if constexpr (KIND == kSwigluOai) {
    return swiglu_oai<T>(gate_bits, up_bits, limit, alpha);
  } else if constexpr (KIND == kSitu) {
    const float gate_out = alpha * tanhf(gate * (1.0f / alpha)) / (1.0f + expf(-gate));
    const float up_out = beta > 0.0f ? beta * tanhf(up * (1.0f / beta)) : up;
    return from_f32<T>(gate_out * up_out);
  } else {
    const float silu = gate / (1.0f + expf(-gate));
    return from_f32<T>(fminf(silu, limit) * fmaxf(fminf(up, limit), -limit));
  }
}

// in: rows x 2d (gate half then up half; kSwigluOai: gate and up alternate), out: rows x d.
template <typename T, int KIND>
__global__ __launch_bounds__(256) void moe_activation_kernel(uint16_t* __restrict__ out,
                                                            const uint16_t* __restrict__ in, long rows, int d,
                                                            float limit, float alpha, float beta) {
  const long vec_per_row = d / 8;
  const long total = rows * vec_per_row;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const long r = i / vec_per_row;
    const int c = (int)(i - r * vec_per_row) * 8;
    uint4 g, u;
    if constexpr (KIND == kSwigluOai) {   // sixteen values: eight pairs
      g = *reinterpret_cast<const uint4*>(in + r * 2 * d + 2 * c);
      u = *reinterpret_cast<const uint4*>(in + r * 2 * d + 2 * c + 8);
    } else {
      g = *reinterpret_cast<const uint4*>(in + r * 2 * d + c);
      u = *reinterpret_cast<const uint4*>(in + r * 2 * d + d + c);
    }
    const uint32_t gw[4] = {g.x, g.y, g.z, g.w}, uw[4] = {u.x, u.y, u.z, u.w};
    uint32_t ow[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      uint32_t o = 0;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint16_t gb, ub;
        if constexpr (KIND == kSwigluOai) {   // output 2 w + h of these eight: the pair in word 2 w + h of g | u
          const int pair = 2 * w + h;
          const uint32_t word = pair < 4 ? gw[pair] : uw[pair - 4];
          gb = (uint16_t)word;
          ub = (uint16_t)(word >> 16);
        } else {
          gb = (uint16_t)(gw[w] >> (16 * h));
          ub = (uint16_t)(uw[w] >> (16 * h));
        }
        o |= (uint32_t)gated_activation<T, KIND>(gb, ub, limit, alpha, beta) << (16 * h);
      }
      ow[w] = o;
    }
    *reinterpret_cast<uint4*>(out + r * d + c) = make_uint4(ow[0], ow[1], ow[2], ow[3]);
  }
}

// out[t][c] = T(sum_k in[t][k][c]), summed in fp32.
template <typename T>
__global__ __launch_bounds__(256) void moe_sum_kernel(uint16_t* __restrict__ out, const uint16_t* __restrict__ in,
                                                     long tokens, int topk, int d) {
  const long vec_per_row = d / 8;
  const long total = tokens * vec_per_row;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const long t = i / vec_per_row;
    const int c = (int)(i - t * vec_per_row) * 8;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < topk; ++k) {
      const uint4 v = *reinterpret_cast<const uint4*>(in + (t * topk + k) * d + c);
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc[2 * j] += to_f32<T>((uint16_t)w[j]);
        acc[2 * j + 1] += to_f32<T>((uint16_t)(w[j] >> 16));
      }
    }
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      o[j] = (uint32_t)from_f32<T>(acc[2 * j]) | ((uint32_t)from_f32<T>(acc[2 * j + 1]) << 16);
    *reinterpret_cast<uint4*>(out + t * d + c) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

inline int blocks_for(long items) {
  const long b = (items + 255) / 256;
  return (int)(b < 1 ? 1 : (b > 8192 ? 8192 : b));
}

}  // namespace
}  // namespace sonar

using namespace sonar;

extern "C" int sonar_moe_align_block_size(const int32_t* topk_ids, int64_t numel, int64_t num_experts,
                                          int64_t block_size, int32_t* sorted_token_ids, int64_t sorted_len,
                                          int32_t* expert_ids, int64_t expert_len,
                                          int32_t* num_tokens_post_pad, const int32_t* expert_map,
                                          int32_t* offsets_scratch, void* stream) {
  SONAR_REQUIRE(numel >= 0 && numel < (1LL << 30), "topk_ids.numel = %ld out of range", (long)numel);
  SONAR_REQUIRE(num_experts >= 1 && num_experts <= 8192, "num_experts = %ld out of range", (long)num_experts);
  SONAR_REQUIRE(block_size >= 1, "block_size = %ld must be positive", (long)block_size);
  SONAR_REQUIRE(sorted_len >= 0 && sorted_len < (1LL << 30) && expert_len >= 0, "output lengths out of range");
  SONAR_REQUIRE(expert_len * block_size >= sorted_len, "expert_ids holds %ld blocks, fewer than ceil(%ld / %ld)",
                (long)expert_len, (long)sorted_len, (long)block_size);
  // every expert may need block_size - 1 padding slots
  const int64_t worst = numel + num_experts * (block_size - 1);
  SONAR_REQUIRE(sorted_len >= (numel < num_experts ? (numel * block_size < worst ? numel * block_size : worst)
                                                    : worst),
                "sorted_token_ids.numel = %ld is too small", (long)sorted_len);
  SONAR_REQUIRE(sorted_token_ids && expert_ids && num_tokens_post_pad && offsets_scratch && (topk_ids || numel == 0),
                "moe_align_block_size: NULL argument");
  hipStream_t st = (hipStream_t)stream;
  const bool place = num_experts <= kAlignOneLaunchExperts;
  // a workgroup for every 1024 slots: a round of 64 a wavefront
  const int workgroups =
      place && numel > kAlignOneWorkgroup ? (int)std::min<int64_t>((numel + kAlignThreads - 1) / kAlignThreads, kAlignMost) : 1;
  const size_t lds = (size_t)(2 * num_experts + 1 + kAlignWaves +
                              (place ? kAlignWaves + (workgroups > 1 ? 2 : 0) : 1) * num_experts) * sizeof(int32_t);
  // (eight rounds at a time: 0.4 us longer where a wavefront has one)
  auto* count = align_share((int)numel, workgroups) > 64 ? moe_align_count_kernel<8> : moe_align_count_kernel<1>;
  if (lds > 64 * 1024)   // from 5456 experts on (8192: 98372 bytes); HIP promises no more unasked, though ROCm 7.2 gives it
    SONAR_HIP(hipFuncSetAttribute((const void*)count, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  count<<<workgroups, kAlignThreads, lds, st>>>(topk_ids, (int)numel, (int)num_experts, (int)block_size, sorted_token_ids,
                                       (int)sorted_len, expert_ids, (int)expert_len, num_tokens_post_pad, expert_map,
                                       offsets_scratch, place);
  if (int rc = launch_status("moe_align_count_kernel")) return rc;
  if (numel > 0 && !place) {
    moe_align_place_kernel<<<(int)((num_experts + 3) / 4), 256, 0, st>>>(topk_ids, (int)numel, (int)num_experts,
                                                                         sorted_token_ids, expert_map,
                                                                         offsets_scratch);
    if (int rc = launch_status("moe_align_place_kernel")) return rc;
  }
  return SONAR_OK;
}

extern "C" int sonar_silu_and_mul(void* out, const void* in, int64_t rows, int64_t d, int dtype, void* stream) {
  SONAR_REQUIRE(dtype == SONAR_DTYPE_F16 || dtype == SONAR_DTYPE_BF16, "unsupported dtype");
  SONAR_REQUIRE(rows >= 0 && d > 0 && d % 8 == 0, "silu_and_mul: d = %ld must be a positive multiple of 8", (long)d);
  if (rows == 0) return SONAR_OK;
  SONAR_REQUIRE(out && in && ((uintptr_t)out) % 16 == 0 && ((uintptr_t)in) % 16 == 0,
                "silu_and_mul: pointers must be 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  const int blocks = blocks_for(rows * (d / 8));
  if (dtype == SONAR_DTYPE_F16)
    silu_and_mul_kernel<_Float16><<<blocks, 256, 0, st>>>(static_cast<uint16_t*>(out),
                                                          static_cast<const uint16_t*>(in), rows, (int)d);
  else
    silu_and_mul_kernel<__bf16><<<blocks, 256, 0, st>>>(static_cast<uint16_t*>(out),
                                                        static_cast<const uint16_t*>(in), rows, (int)d);
  return launch_status("silu_and_mul_kernel");
}

namespace {
template <typename T>
void launch_moe_activation(int kind, int blocks, hipStream_t st, uint16_t* out, const uint16_t* in, long rows, int d,
                           float limit, float alpha, float beta) {
  switch (kind) {
    case kClampSilu: moe_activation_kernel<T, kClampSilu><<<blocks, 256, 0, st>>>(out, in, rows, d, limit, alpha, beta); break;
    case kGelu: moe_activation_kernel<T, kGelu><<<blocks, 256, 0, st>>>(out, in, rows, d, limit, alpha, beta); break;
    case kGeluTanh: moe_activation_kernel<T, kGeluTanh><<<blocks, 256, 0, st>>>(out, in, rows, d, limit, alpha, beta); break;
    case kSwigluOai: moe_activation_kernel<T, kSwigluOai><<<blocks, 256, 0, st>>>(out, in, rows, d, limit, alpha, beta); break;
    case kSitu: moe_activation_kernel<T, kSitu><<<blocks, 256, 0, st>>>(out, in, rows, d, limit, alpha, beta); break;
    default: moe_activation_kernel<T, kSwigluStep><<<blocks, 256, 0, st>>>(out, in, rows, d, limit, alpha, beta); break;
  }
}
}  // namespace

extern "C" int sonar_moe_activation(void* out, const void* in, int64_t rows, int64_t d, int kind, float limit,
                                    float alpha, float beta, int dtype, void* stream) {
  SONAR_REQUIRE(dtype == SONAR_DTYPE_F16 || dtype == SONAR_DTYPE_BF16, "unsupported dtype");
  SONAR_REQUIRE(kind >= SONAR_ACT_SILU_CLAMP && kind <= SONAR_ACT_SWIGLUSTEP, "moe_activation: unknown kind %d", kind);
  SONAR_REQUIRE(rows >= 0 && d > 0 && d % 8 == 0, "moe_activation: d = %ld must be a positive multiple of 8", (long)d);
  if (kind == SONAR_ACT_SILU_CLAMP || kind == SONAR_ACT_SWIGLUOAI || kind == SONAR_ACT_SWIGLUSTEP)
    SONAR_REQUIRE(limit > 0.0f, "moe_activation: this activation needs a positive clamp limit");
  if (kind == SONAR_ACT_SITU) SONAR_REQUIRE(alpha > 0.0f, "moe_activation: SITU needs a positive beta");
  if (rows == 0) return SONAR_OK;
  SONAR_REQUIRE(out && in && ((uintptr_t)out) % 16 == 0 && ((uintptr_t)in) % 16 == 0,
                "moe_activation: pointers must be 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  const int blocks = blocks_for(rows * (d / 8));
  if (dtype == SONAR_DTYPE_F16)
    launch_moe_activation<_Float16>(kind, blocks, st, static_cast<uint16_t*>(out), static_cast<const uint16_t*>(in),
                                    rows, (int)d, limit, alpha, beta);
  else
    launch_moe_activation<__bf16>(kind, blocks, st, static_cast<uint16_t*>(out), static_cast<const uint16_t*>(in),
                                  rows, (int)d, limit, alpha, beta);
  return launch_status("moe_activation_kernel");
}

extern "C" int sonar_moe_sum(void* out, const void* in, int64_t tokens, int64_t topk, int64_t d, int dtype,
                             void* stream) {
  SONAR_REQUIRE(dtype == SONAR_DTYPE_F16 || dtype == SONAR_DTYPE_BF16, "unsupported dtype");
  SONAR_REQUIRE(tokens >= 0 && topk >= 1 && d > 0 && d % 8 == 0,
                "moe_sum: d = %ld must be a positive multiple of 8 and topk = %ld positive", (long)d, (long)topk);
  if (tokens == 0) return SONAR_OK;
  SONAR_REQUIRE(out && in && ((uintptr_t)out) % 16 == 0 && ((uintptr_t)in) % 16 == 0,
                "moe_sum: pointers must be 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  const int blocks = blocks_for(tokens * (d / 8));
  if (dtype == SONAR_DTYPE_F16)
    moe_sum_kernel<_Float16><<<blocks, 256, 0, st>>>(static_cast<uint16_t*>(out), static_cast<const uint16_t*>(in),
                                                     tokens, (int)topk, (int)d);
  else
    moe_sum_kernel<__bf16><<<blocks, 256, 0, st>>>(static_cast<uint16_t*>(out), static_cast<const uint16_t*>(in),
                                                   tokens, (int)topk, (int)d);
  return launch_status("moe_sum_kernel");
}
