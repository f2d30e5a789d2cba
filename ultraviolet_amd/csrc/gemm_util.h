// Helpers shared by the GEMM kernels (gfx950): MFMA wrappers on 16-byte operand words and rounding / packing to the
// activation type.
#pragma once
#include "common.h"

namespace uvmi {

typedef _Float16 gh8 __attribute__((ext_vector_type(8)));
typedef __bf16 gb8 __attribute__((ext_vector_type(8)));
typedef float gf4 __attribute__((ext_vector_type(4)));
typedef unsigned int gu4 __attribute__((ext_vector_type(4)));

#define UVMI_LDSP(p) ((__attribute__((address_space(3))) void*)(p))

// 16 bytes per lane from byte off + at of a buffer to 1 KB of LDS (a template's own code cannot hold the builtin: the host's pass checks it)
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, unsigned char* lds, uint32_t off, int at) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, UVMI_LDSP(lds), 16, off, at, 0, 0);
}

template <int N> __device__ __forceinline__ void wait_vm() {   // all but the newest N loads have landed
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
}

template <int DT>
__device__ __forceinline__ gf4 gmfma(gu4 a, gu4 b, gf4 c) {
  if constexpr (DT == UVMI_F16) {
    gh8 x, y;
    __builtin_memcpy(&x, &a, 16);
    __builtin_memcpy(&y, &b, 16);
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(x, y, c, 0, 0, 0);
  } else {
    gb8 x, y;
    __builtin_memcpy(&x, &a, 16);
    __builtin_memcpy(&y, &b, 16);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0);
  }
}

template <int DT> __device__ __forceinline__ float ground(float v) {
  if constexpr (DT == UVMI_F16) return (float)(half_t)v;
  else return bf16_to_float(float_to_bf16(v));
}
// silu(g) rounded to the activation type, for a g already on that type's grid.  bf16 divides through the hardware reciprocal
// (1 ulp in fp32, ahead of a rounding to 8 bits), as the standalone SwiGLU kernel does: a full IEEE division is ten
// instructions per element of the gate-up epilogue.
template <int DT> __device__ __forceinline__ float silu_round(float gv) {
  if constexpr (DT == UVMI_BF16) return ground<DT>(gv * __builtin_amdgcn_rcpf(1.0f + __expf(-gv)));
  else return ground<DT>(gv / (1.0f + __expf(-gv)));
}
template <int DT> __device__ __forceinline__ uint32_t gpack(float a, float b) {
  if constexpr (DT == UVMI_BF16) return float2_to_bf16x2(a, b);   // one conversion for the two
  else return (uint32_t)float_to_half_bits(a) | ((uint32_t)float_to_half_bits(b) << 16);
}
template <int DT> __device__ __forceinline__ void gunpack(uint32_t w, float& lo, float& hi) {
  if (DT == UVMI_BF16) { lo = __uint_as_float(w << 16); hi = __uint_as_float(w & 0xffff0000u); }
  else { lo = half_bits_to_float((uint16_t)(w & 0xffff)); hi = half_bits_to_float((uint16_t)(w >> 16)); }
}
// silu(gate) * up for two outputs: everything is rounded to the activation type in pairs (a third fewer instructions than one by one)
template <int DT> __device__ __forceinline__ uint32_t gswiglu2(float g0, float g1, float u0, float u1) {
  float a, b, c, d;
  gunpack<DT>(gpack<DT>(g0, g1), a, b);
  gunpack<DT>(gpack<DT>(u0, u1), c, d);
  if constexpr (DT == UVMI_BF16) {   // (silu_round for two)
    float sa, sb;
    gunpack<DT>(gpack<DT>(a * __builtin_amdgcn_rcpf(1.0f + __expf(-a)), b * __builtin_amdgcn_rcpf(1.0f + __expf(-b))), sa, sb);
    return gpack<DT>(sa * c, sb * d);
  } else {
    return gpack<DT>(silu_round<DT>(a) * c, silu_round<DT>(b) * d);
  }
}

}  // namespace uvmi
