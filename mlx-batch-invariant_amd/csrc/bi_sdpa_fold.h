// The fold of a segment's result into the running result of the matrix-core
// attention's fixed arithmetic (bi_sdpa_mfma_kernel.h), shared by the kernels
// that walk every segment and by the one that folds partial results.
#pragma once

#include <hip/hip_runtime.h>

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
constexpr float kLog2e = 1.4426950408889634f;

// Folds a segment's (M, L, O) into the running (R, S, Q).
struct FoldW {
  float e, f;  // weights of the running state and of the segment
};
__device__ __forceinline__ FoldW fold_stats(float& R, float& S, float M, float L) {
  const float n = fmaxf(R, M);
  const FoldW w = {__builtin_amdgcn_exp2f(R - n), __builtin_amdgcn_exp2f(M - n)};
  S = __builtin_fmaf(L, w.f, S * w.e);
  R = n;
  return w;
}
__device__ __forceinline__ void fold_out(f32x4_t& Q, const f32x4_t& O, FoldW w) {
#pragma unroll
  for (int e = 0; e < 4; e++) Q[e] = __builtin_fmaf(O[e], w.f, Q[e] * w.e) + 0.f;
}

}  // namespace
