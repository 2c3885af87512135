#pragma once
#include "common.h"

namespace aha {

// first maximal index (candle argmax / Sampling::ArgMax)
__device__ __forceinline__ void argmax_combine(float& bv, uint32_t& bi, float v, uint32_t i) {
  if (v > bv || (v == bv && i < bi)) { bv = v; bi = i; }
}
__device__ __forceinline__ void wave_argmax(float& bv, uint32_t& bi) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o, 64);
    const uint32_t oi = __shfl_xor(bi, o, 64);
    argmax_combine(bv, bi, ov, oi);
  }
}

}  // namespace aha
