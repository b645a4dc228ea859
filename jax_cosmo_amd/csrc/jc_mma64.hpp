// FP64 matrix products of 16 x 16 tiles (v_mfma_f64_16x16x4).
#pragma once
#include <hip/hip_runtime.h>

namespace jc {

typedef double d4 __attribute__((ext_vector_type(4)));

// D[i][j] += sum_k A[i][k] B[k][j] over 4 k: lane l passes A[l % 16][l / 16]
// and B[l / 16][l % 16] and holds D[l / 16 + 4 r][l % 16] in register r
__device__ __forceinline__ d4 mfma64(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// The same over 16 k: lane l passes k = 4 (l / 16) .. + 3 of row (column) l % 16
// of both operands (element q of both in one instruction, so any assignment of k
// to lanes serves).
__device__ __forceinline__ void mma16(const d4& a, const d4& b, d4& c) {
#pragma unroll
  for (int q = 0; q < 4; ++q) c = mfma64(a[q], b[q], c);
}

}  // namespace jc
