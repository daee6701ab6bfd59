// fk_mfma.h — what the matrix-core kernels share: the operand vector types of
// the gfx950 v_mfma_f32_*_f16 builtins, raw buffer descriptors, and the
// binary32 -> binary16 conversion of their f16 outputs.
#pragma once

#include "fk_common.h"

typedef _Float16 fk_half8 __attribute__((ext_vector_type(8)));
typedef float fk_float4v __attribute__((ext_vector_type(4)));
typedef float fk_float16v __attribute__((ext_vector_type(16)));

namespace fk {

// Eight f16 operands, as the builtin takes them or as 16 bytes of memory.
union Half8 {
  fk_half8 h;
  uint4 u;
};

// A raw buffer over [base, base + bytes): loads past its end read zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void *base, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0,
                                           (int)(uint32_t)(bytes < 0xffffffffu ? bytes : 0xffffffffu), 0x00020000);
}

// binary32 -> binary16, to nearest even (v_cvt_f16_f32).
__device__ __forceinline__ uint16_t to_f16(float x) { return __builtin_bit_cast(uint16_t, (_Float16)x); }

// The gated MLP's activation of a matrix product's element, on its way to f16:
// silu(g) = g / (1 + e^-g), or gelu(g) = 0.5 g (1 + tanh(y)) with tanh(y) =
// 1 - 2 / (1 + e^2y), with the hardware's exp and reciprocal (a few ulp of
// binary32): the f16 rounding after it (2^-11) bounds the error.  An
// exponential overflowing gives the limits (silu 0, tanh 1).
template <bool GELU>
__device__ __forceinline__ float act_hw(float g) {
  if constexpr (GELU) {
    const float y = 0.7978845608028654f * (g + ((0.044715f * g) * g) * g);
    const float th = 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + __expf(2.0f * y));
    return (0.5f * g) * (1.0f + th);
  } else {
    return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g));
  }
}

}  // namespace fk
