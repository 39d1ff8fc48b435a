// Matrix-core building blocks shared by the scorers (gfx950).
#pragma once

#include "tri_common.h"

namespace tri {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// One 16x16x32 matrix-core step in the operand type of the keys (fp8 keys are converted to bf16).
template <int DT>
__device__ __forceinline__ f32x4 mfma_16x16x32(const uint4& a, const uint4& b, f32x4 c) {
  if constexpr (DT == TRI_KV_FP16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// m[i] = sqrt(x[i].lo^2 + x[i].hi^2) for four packed bf16 pairs, in fp32.  Written out for
// two reasons: the compiler only selects the accumulating two-operand dot product
// (v_dot2c_f32_bf16) and spends a v_mov per value on zeroing its destination, and it does
// not see the opcodes inside an asm statement, so the spacing gfx950 requires between a dot
// product's write and another vector instruction's read of that register (three
// instructions) and after a transcendental's write (one) is provided here: four dot
// products, then the four square roots in the same order, then one idle cycle.
template <int DT>
__device__ __forceinline__ void magnitudes4(const uint32_t (&x)[4], float* m) {
  if constexpr (DT == TRI_KV_FP16) {
    asm("v_dot2_f32_f16 %0, %4, %4, 0\n\t"
        "v_dot2_f32_f16 %1, %5, %5, 0\n\t"
        "v_dot2_f32_f16 %2, %6, %6, 0\n\t"
        "v_dot2_f32_f16 %3, %7, %7, 0\n\t"
        "v_sqrt_f32 %0, %0\n\t"
        "v_sqrt_f32 %1, %1\n\t"
        "v_sqrt_f32 %2, %2\n\t"
        "v_sqrt_f32 %3, %3\n\t"
        "s_nop 0"
        : "=&v"(m[0]), "=&v"(m[1]), "=&v"(m[2]), "=&v"(m[3])
        : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]));
  } else {
    asm("v_dot2_f32_bf16 %0, %4, %4, 0\n\t"
        "v_dot2_f32_bf16 %1, %5, %5, 0\n\t"
        "v_dot2_f32_bf16 %2, %6, %6, 0\n\t"
        "v_dot2_f32_bf16 %3, %7, %7, 0\n\t"
        "v_sqrt_f32 %0, %0\n\t"
        "v_sqrt_f32 %1, %1\n\t"
        "v_sqrt_f32 %2, %2\n\t"
        "v_sqrt_f32 %3, %3\n\t"
        "s_nop 0"
        : "=&v"(m[0]), "=&v"(m[1]), "=&v"(m[2]), "=&v"(m[3])
        : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]));
  }
}

}  // namespace
}  // namespace tri
