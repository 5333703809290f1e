// Device code shared by the MXFP8 kernels: bf16 and E4M3 conversions, block quantisation, the LDS operand layout of the scaled MFMA.
#pragma once
#include "common.h"

typedef int v8i32 __attribute__((ext_vector_type(8)));
typedef float v4f32 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float bf16_to_f(uint16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }
__device__ __forceinline__ float bf16_lo(uint32_t p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t p) { return __builtin_bit_cast(float, p & 0xFFFF0000u); }
__device__ __forceinline__ uint16_t f_to_bf16(float f) {   // round to nearest even (tinygrad/dtype.py:224-226)
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
  return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1)) >> 16);
}
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {          // round to nearest even (tinygrad/dtype.py:224-226); one v_cvt_pk_bf16_f32
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t));
}

// E8M0 of a block with largest magnitude amax: clamp(floor(log2(max(amax, 1e-38))) + 127, 0, 254), i.e. the exponent field (0 below the smallest normal float, where
// the floor gives -127; 126 for an infinite amax, which has no exponent)
__device__ __forceinline__ int mx_e8(float amax) {
  const int e = (int)(__builtin_bit_cast(uint32_t, amax) >> 23);
  return e >= 255 ? 126 : e;
}
__device__ __forceinline__ float mx_scale(int e) { return __builtin_bit_cast(float, e == 254 ? 0x00400000u : (uint32_t)(254 - e) << 23); }   // 2^(127 - e), exact
__device__ __forceinline__ float mx_clamp(float s) { return fminf(fmaxf(s, -448.0f), 448.0f); }
// four values already scaled -> four E4M3 bytes (v_cvt_pk_fp8_f32: OCP E4M3 on this part, round to nearest even incl. subnormals; checked over all 2^32 inputs
// against the arithmetic of tinygrad/dtype.py:237-260)
__device__ __forceinline__ uint32_t e4m3x4(float a, float b, float c, float d) {
  int r = __builtin_amdgcn_cvt_pk_fp8_f32(mx_clamp(a), mx_clamp(b), 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(mx_clamp(c), mx_clamp(d), r, true);
}
__device__ __forceinline__ uint32_t e4m3x2(float a, float b) { return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(mx_clamp(a), mx_clamp(b), 0, false) & 0xFFFFu; }
// 1 / (1 + exp(-x)) of a bf16 value on its way to bf16.  The scaling by 2^-24 keeps the reciprocal out of the subnormal numbers, which v_rcp_f32 flushes to zero (x = -87.5 .. -88.5); after the
// rounding to bf16 the result is that of expf and a rounded division for all 2^16 inputs (enumerated), in a fifth of the operations.
__device__ __forceinline__ float mx_sigmoid_bf16(float x) { return __builtin_amdgcn_rcpf(__builtin_fmaf(__builtin_amdgcn_exp2f(-1.4426950408889634f * x), 0x1p-24f, 0x1p-24f)) * 0x1p-24f; }

__device__ __forceinline__ float quad_max(float v) {                    // over the four lanes of a quad
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true)));     // quad_perm [1,0,3,2]
  return fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true))); // quad_perm [2,3,0,1]
}

// Byte offset inside an operand region in LDS of (row R, 16-byte chunk c) of a 128-byte K step: the order the scaled MFMA consumes (see grouped_mxfp8_gemm_tile)
__device__ __forceinline__ int gg_slot_off(int R, int c) {
  const int sub = R >> 4, r = R & 15, p = c >> 2, g = c & 3;
  return sub * 2048 + p * 1024 + ((16 * g + (r ^ (g + 4 * p))) << 4);
}
