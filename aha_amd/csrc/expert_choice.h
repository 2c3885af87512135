// The `top` largest of up to 64 router logits, one per lane of a wave: what a round of the choice decides, for the wave (kernels_gemv_experts.hip) and for
// its restatement on the host (capi.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

namespace aha {

// A logit that is not a number counts as -inf: with 64 experts no lane is spare, and a maximum of NaN alone would be held by none of them (an index in
// front of the experts' weights).
__host__ __device__ __forceinline__ float choice_logit(float z) { return z == z ? z : -INFINITY; }
// m: the largest logit left, at: the lanes that hold it.  Ties go to the lower index; nothing left but -inf: the last expert.
__host__ __device__ __forceinline__ int choice_lane(float m, uint64_t at, int experts) { return m == -INFINITY ? experts - 1 : __builtin_ctzll(at); }
__host__ __device__ __forceinline__ float choice_weight(float m) { return 1.0f / (1.0f + expf(-m)); }

}  // namespace aha
