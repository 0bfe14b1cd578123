// Shared helpers of the gfx950 Marlin library: error reporting, vector types
// and the layout constants every kernel agrees on.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstdarg>
#include <cstdio>

#include "sonar_marlin.h"

namespace sonar {

// ---- error reporting ------------------------------------------------------
char* last_error_buffer();  // thread-local, 512 bytes

inline int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(last_error_buffer(), 512, fmt, ap);
  va_end(ap);
  return code;
}

#define SONAR_REQUIRE(cond, ...)                          \
  do {                                                    \
    if (!(cond)) return ::sonar::fail(SONAR_E_INVALID, __VA_ARGS__); \
  } while (0)

#define SONAR_HIP(expr)                                                     \
  do {                                                                      \
    hipError_t e_ = (expr);                                                 \
    if (e_ != hipSuccess)                                                   \
      return ::sonar::fail(SONAR_E_RUNTIME, "%s failed: %s", #expr,         \
                           hipGetErrorString(e_));                          \
  } while (0)

inline int launch_status(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return fail(SONAR_E_RUNTIME, "launch of %s failed: %s", what, hipGetErrorString(e));
  return SONAR_OK;
}

// ---- vector types ---------------------------------------------------------
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef int16_t short2_t __attribute__((ext_vector_type(2)));
typedef uint16_t ushort2_t __attribute__((ext_vector_type(2)));
typedef float floatx2_t __attribute__((ext_vector_type(2)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
// address spaces of the asynchronous global -> LDS copy builtin
typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) const void glb_void_t;

// Asynchronous copy of BYTES (4 or 16) a lane from `base` + the lane's `off` to LDS, lane after lane from byte `lds` on; `base` and
// `lds` are the wavefront's.  (The builtin takes 64-bit addresses a lane, which hold up the wavefront's other instructions some
// 20 cycles more.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"   // m0 is a reserved register: that it changes is what the clobber says
template <int BYTES>
__device__ __forceinline__ void copy_to_lds(uint32_t lds, uint32_t off, const char* base) {
  static_assert(BYTES == 4 || BYTES == 16, "");
  if constexpr (BYTES == 16)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
// Four copies of 1 KiB that follow one another in memory and in LDS (the offset of the instruction counts for both).
// NT: non-temporal.
template <bool NT>
__device__ __forceinline__ void copy_4k_to_lds(uint32_t lds, uint32_t off, const char* base) {
#define SONAR_COPY_4K(NT_BIT)                                                                                              \
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" NT_BIT                                      \
               "\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024" NT_BIT "\n\tglobal_load_lds_dwordx4 %1, %2 offset:2048" NT_BIT \
               "\n\tglobal_load_lds_dwordx4 %1, %2 offset:3072" NT_BIT ::"s"(lds), "v"(off), "s"(base) : "memory", "m0")
  if constexpr (NT) SONAR_COPY_4K(" nt");
  else SONAR_COPY_4K("");
#undef SONAR_COPY_4K
}
#pragma clang diagnostic pop

// ---- layout constants -----------------------------------------------------
// Marlin order: tiles of 16 (k) x 64 (n), 128 words each, stored k-tile major.
constexpr int kMarlinTileK = 16;
constexpr int kMarlinTileN = 64;
constexpr int kMarlinTileWords = 128;
// gfx950 streaming order: 64-column strips, each a run of 32-row chunks of
// 256 words (1 KiB); lane L of a wavefront owns words 4L..4L+3 of a chunk.
constexpr int kStripN = 64;
constexpr int kChunkK = 32;
constexpr int kChunkWords = 256;

}  // namespace sonar
