// nx_split_dev.hpp — operands of the split-activation MFMA kernels
// (nx_mfv.hip, nx_mfd.hip): f32 activations as two fp16 halves against
// quantized codes that enter the matrix cores as exact fp16 values.
#pragma once

#include "nx_device.hpp"

namespace nx {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// 4 x 4 transpose of dwords across the four 16-lane groups: on return
// c[k] of lane group g holds what c[g] of lane group k held (register
// swaps between lane halves, then between neighbouring lane groups)
__device__ __forceinline__ void transpose_groups(uint32_t (&c)[4]) {
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const auto v = __builtin_amdgcn_permlane32_swap(c[k], c[k + 2], false, false);
    c[k] = v[0];
    c[k + 2] = v[1];
  }
#pragma unroll
  for (int k = 0; k < 4; k += 2) {
    const auto v = __builtin_amdgcn_permlane16_swap(c[k], c[k + 1], false, false);
    c[k] = v[0];
    c[k + 1] = v[1];
  }
}

}  // namespace nx
