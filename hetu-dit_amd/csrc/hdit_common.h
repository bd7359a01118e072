// Shared device helpers for the gfx950 (CDNA4, wave64) kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/hdit.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) int i32x4;
typedef __attribute__((ext_vector_type(2))) int i32x2;
typedef __attribute__((ext_vector_type(4))) short s16x4;

#define HDIT_WAVE 64

namespace hdit {

__device__ __forceinline__ float bf16_to_f32(__bf16 x) { return (float)x; }

// 8 bf16 held in an int4 <-> 8 floats
__device__ __forceinline__ void unpack8(const i32x4& raw, float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    uint32_t u = (uint32_t)raw[i];
    f[2 * i] = __uint_as_float(u << 16);
    f[2 * i + 1] = __uint_as_float(u & 0xffff0000u);
  }
}

__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  f32x2 v = {lo, hi};
  bf16x2 b = __builtin_convertvector(v, bf16x2);  // v_cvt_pk_bf16_f32, round-nearest-even
  return __builtin_bit_cast(uint32_t, b);
}

__device__ __forceinline__ i32x4 pack8(const float (&f)[8]) {
  i32x4 r;
#pragma unroll
  for (int i = 0; i < 4; i++) r[i] = (int)pack2(f[2 * i], f[2 * i + 1]);
  return r;
}

// v of the 64 lanes added up, in every lane: the partner of a step is lane ^ 32, ^ 16, ^ 8, ^ 4, ^ 2, ^ 1.  In registers
// (lane swaps, then rotations inside the rows of 16 lanes, whose values repeat every 2 * n lanes by then): an exchange
// through LDS costs its latency six times over.  512 rows of 1536 fp32, normalised: 4.44 -> 4.18 us, 1357 rows
// 5.63 -> 5.42.
template <int N>
__device__ __forceinline__ float row_rotate(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xf, 0xf, true));  // row_ror:N
}
__device__ __forceinline__ float wave_sum(float v) {
  auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
  v = __int_as_float(s32[0]) + __int_as_float(s32[1]);
  auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
  v = __int_as_float(s16[0]) + __int_as_float(s16[1]);
  v += row_rotate<8>(v);
  v += row_rotate<4>(v);
  v += row_rotate<2>(v);
  v += row_rotate<1>(v);
  return v;
}

__device__ __forceinline__ float gelu_tanh_f(float x) {
  // 0.5 x (1 + tanh(u)), u = sqrt(2/pi) (x + 0.044715 x^3), equals x * sigmoid(2u) = x / (1 + 2^(-2u log2 e)).
  // Written on v_exp_f32 / v_rcp_f32 directly: five full-rate VALU ops and two transcendentals per value.
  const float k = 2.0f * 0.7978845608028654f * 1.4426950408889634f;  // 2 sqrt(2/pi) log2(e)
  const float t = x * x;
  const float p = __builtin_fmaf(t, 0.044715f * k, k);
  const float e = __builtin_amdgcn_exp2f(-(x * p));
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}

__device__ __forceinline__ float silu_f(float x) {
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * x));
}

}  // namespace hdit

// Host-side error plumbing shared by the C-ABI entry points.
namespace hdit_host {
void set_error(const char* msg);
int check_launch(const char* what);
int num_cus();
}  // namespace hdit_host
