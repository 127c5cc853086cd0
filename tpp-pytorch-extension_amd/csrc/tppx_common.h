// Shared host/device helpers of the gfx950 quantized-linear library.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#include "tppx.h"

namespace tppx {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) int i32x4;
typedef __attribute__((ext_vector_type(8))) int i32x8;
typedef __attribute__((ext_vector_type(16))) int i32x16;

// ---- error plumbing (host) ------------------------------------------------
int set_error(int code, const char* fmt, ...);
int check_hip(hipError_t e, const char* what);

#define TPPX_REQUIRE(cond, code, ...)          \
  do {                                         \
    if (!(cond))                               \
      return ::tppx::set_error(code, __VA_ARGS__); \
  } while (0)

// ---- launch plan recording (host) -------------------------------------------
// While a plan is being recorded (tppx_plan_linear_*), launch sites describe
// the kernel they would run and launch nothing.
bool plan_recording();
void plan_note(const void* kernel_fn, dim3 grid, dim3 block, size_t lds_bytes);
#define TPPX_PLAN_ONLY(kern, grid, block, lds)                                  \
  do {                                                                          \
    if (::tppx::plan_recording()) {                                             \
      ::tppx::plan_note(reinterpret_cast<const void*>(kern), grid, block, lds); \
      return hipSuccess;                                                        \
    }                                                                           \
  } while (0)

static inline bool aligned16(const void* p) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

// ---- bf16 <-> fp32 (device) -----------------------------------------------
__device__ __forceinline__ float bf16_bits_to_f32(uint32_t h) {
  return __uint_as_float(h << 16);
}

// round to nearest even, NaN kept quiet (same rule as the CPU side): the hardware conversion, equal to the integer
// formula (u + 0x7fff + ((u >> 16) & 1)) >> 16 and to (u >> 16) | 0x40 for a NaN over all 2^32 inputs
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
  return __builtin_bit_cast(uint16_t, (__bf16)f);
}
// two values into one dword: one instruction
__device__ __forceinline__ uint32_t f32x2_to_bf16_bits(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, bf16x2{(__bf16)lo, (__bf16)hi});
}

__device__ __forceinline__ float round_bf16(float f) {
  return bf16_bits_to_f32(f32_to_bf16_bits(f));
}

// Rotation of a pair by (c, s): x1 c - x2 s and x2 c + x1 s, the cosine's product fused into the rounded product of the sine.  In
// a plain sum of two products the compiler chooses which one is fused, by kernel; the launches that rotate have to agree in
// every bit, also where the two nearly cancel, for a cache filled by one of them and read behind another.
__device__ __forceinline__ float rotate_first(float x1, float x2, float c, float s) {
  return fmaf(x1, c, -__fmul_rn(x2, s));
}
__device__ __forceinline__ float rotate_second(float x1, float x2, float c, float s) {
  return fmaf(x2, c, __fmul_rn(x1, s));
}

// ---- post-ops on the bf16-rounded GEMM result -------------------------------
// `v` is bias + dot product in fp32.  The value is rounded to bf16 first and
// every post-op re-rounds where the CPU path stores its bf16 tile.
__device__ __forceinline__ uint32_t apply_post_bits(float v, int post,
                                                    uint32_t in1, uint32_t in2,
                                                    float scale) {
  uint32_t yb = f32_to_bf16_bits(v);
  float y = bf16_bits_to_f32(yb);
  switch (post) {
    case TPPX_POST_SILU: {
      // hardware exp2 / reciprocal: their error (about 1e-7 relative) is far below the bf16 rounding that follows,
      // and the full-precision expf + divide cost as much as 30 MFMA issue slots per output in the prefill epilogue
      float s = round_bf16(__frcp_rn(1.0f + __expf(-y)));
      return f32_to_bf16_bits(y * s);
    }
    case TPPX_POST_MUL:
      return f32_to_bf16_bits(bf16_bits_to_f32(in1) * y);
    case TPPX_POST_ADD_SCALE:
      return f32_to_bf16_bits(fmaf(bf16_bits_to_f32(in1), scale, y));
    case TPPX_POST_ADD2_SCALE: {
      float t = round_bf16(y + bf16_bits_to_f32(in1));
      return f32_to_bf16_bits(fmaf(bf16_bits_to_f32(in2), scale, t));
    }
    case TPPX_POST_GELU:
      return f32_to_bf16_bits(0.5f * y * (1.0f + erff(y * 0.70710678118654752f)));
    case TPPX_POST_RELU:
      return (yb & 0x8000u) ? 0u : yb;
    default:
      return yb;
  }
}

// apply_post_bits for two adjacent outputs, the post-op known at compile time; in1: the packed pair of its input
template <int POST>
__device__ __forceinline__ uint32_t apply_post_pair(float lo, float hi, uint32_t in1, float scale) {
  const uint32_t yb = f32x2_to_bf16_bits(lo, hi);
  const float y0 = bf16_bits_to_f32(yb & 0xffffu), y1 = __uint_as_float(yb & 0xffff0000u);
  if constexpr (POST == TPPX_POST_SILU) {
    const uint32_t s = f32x2_to_bf16_bits(__frcp_rn(1.0f + __expf(-y0)), __frcp_rn(1.0f + __expf(-y1)));
    return f32x2_to_bf16_bits(y0 * bf16_bits_to_f32(s & 0xffffu), y1 * __uint_as_float(s & 0xffff0000u));
  } else if constexpr (POST == TPPX_POST_MUL) {
    return f32x2_to_bf16_bits(bf16_bits_to_f32(in1 & 0xffffu) * y0, __uint_as_float(in1 & 0xffff0000u) * y1);
  } else if constexpr (POST == TPPX_POST_ADD_SCALE) {
    return f32x2_to_bf16_bits(fmaf(bf16_bits_to_f32(in1 & 0xffffu), scale, y0), fmaf(__uint_as_float(in1 & 0xffff0000u), scale, y1));
  } else {
    static_assert(POST == TPPX_POST_NONE, "the other post-ops go through apply_post_bits");
    return yb;
  }
}

// E8M0 byte -> fp32 factor used when de-quantising (byte shifted into the
// exponent field; 0 gives 0.0, 255 gives +Inf).
__device__ __forceinline__ float e8m0_to_f32(uint32_t x) {
  return __uint_as_float((x & 0xffu) << 23);
}

// compile-time loop: f(std::integral_constant<int, I>) for I in [B, E)
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// LDS image of bf16 MFMA operands: the 16-byte chunk c (0..15) of row m's 128 K values lies at position c ^ swz16(m) of 16.
// Lane (g, m) of a read takes chunk g * 4 + j of row m.  A ds_read_b128 is served in four sets of 16 lanes, 64 banks each,
// and a set takes the lanes m = 0..3 and 12..15 of an even g together with m = 4..11 of the next (lanes 0-3, 12-15, 20-27).
// With c ^ m the bits of g and m cancel, the second half of a set has the banks of the first, and every read takes twice
// its cycles (SQ_LDS_BANK_CONFLICT 0.5 of SQ_LDS_IDX_ACTIVE); with bit 3 of m flipped where bit 2 is set they do not.
// The four chunks of an aligned quad stay together: loads into LDS fetch 64 bytes per four lanes (another order that read
// without conflicts, (j * 4 + g) ^ m, spread them over the row and cost 7 % of the whole kernel at 333 rows).
__device__ __forceinline__ constexpr int swz16(int m) {
  return (m ^ ((m & 4) << 1)) & 15;
}

// W4A8 (USE_MXFP4_INT8): the integer the reference multiplies for an E2M1 code = its value times 127 / 6, rounded
// four 4-bit E2M1 codes (one per byte, the upper four bits clear) -> four int8 values {0 11 21 32 42 64 85 127} with sign.
// Two byte permutes look up all sixteen codes: selector bytes 0..7 pick a table byte (0..3 from the second operand, 4..7
// from the first), 8..11 give the sign of the pair's bytes 1, 3, 5, 7 in every bit, 12 zero, 13..15 0xFF.  So the first
// lookup is a constant (0 or 0xFF) for codes 8..15 and the second one, on the code with its sign bit flipped, for codes
// 0..7; the other table's bytes are stored with that constant folded in, and the exclusive or of the two is the value
// (four instructions; a lookup of the magnitude, one of its negative and a select by the sign bit are eight).
__device__ __forceinline__ uint32_t w4a8_expand(uint32_t codes) {
  return __builtin_amdgcn_perm(0x80AABF2Au, 0x20150BFFu, codes) ^
         __builtin_amdgcn_perm(0x7E543FD6u, 0x1F14F500u, codes ^ 0x08080808u);
}

} // namespace tppx
