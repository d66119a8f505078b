// cbz_mfma.h — pieces of the matrix-core kernels of the surrogate network.
#pragma once
#include <hip/hip_runtime.h>

#include "cbz_mlp.h"

namespace cbz {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// SiLU with the hardware reciprocal (about 1 ulp): its result is rounded to
// BF16 for the next layer
__device__ __forceinline__ float silu(float z) { return z * __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }

// Element (row, k) of a 256-wide BF16 tile in LDS sits at row * 256 +
// (((k / 8) ^ (row % 32)) * 8) + k % 8: the 16-byte fragments that the 32
// rows of a tile read at one k land in different banks.
__device__ __forceinline__ int fswz(int row, int k) { return row * kHidden + ((((k >> 3) ^ (row & 31))) << 3) + (k & 7); }

}  // namespace cbz
