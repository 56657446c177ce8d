// nm_mfma.h — the gfx950 matrix-core operands shared by the matrix-core
// kernels (nm_spmm_mc.hip, nm_attention.hip).
#pragma once

#include "nm_gemv_kernel.h"

namespace nm_hip {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s4 lds_s4;

// MFMA 16x16x32 register layout (gfx950; checked on the GPU): A[16 x 32]:
// lane l holds row l % 16, K elements 8*(l/16) .. +7; B[32 x 16]: column
// l % 16, K elements 8*(l/16) .. +7; D[16 x 16]: column l % 16, rows
// 4*(l/16) .. +3.
template <int DT>
__device__ inline f4 mfma16x16x32(s8 a, s8 b, f4 c);
template <>
__device__ inline f4 mfma16x16x32<NM_DTYPE_F16>(s8 a, s8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c, 0, 0, 0);
}
template <>
__device__ inline f4 mfma16x16x32<NM_DTYPE_BF16>(s8 a, s8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
}

}  // namespace nm_hip
