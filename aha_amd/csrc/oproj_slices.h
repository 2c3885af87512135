// o_proj in slices of 256 or 512 columns, one or two kv heads with two query heads each: what a block does with its rows (attn_oproj_kernel,
// oproj_slice_kernel).  The slices' f32 sums go to (slices, n); the norm behind o_proj adds them up (gemv_row_body.h RowSlicesPro).
#pragma once
#include "common.h"

namespace aha {

// R requests per wave, 512 / COLS consecutive rows each; a lane eight columns
template <int R, int COLS>
struct OprojRows {
  static constexpr int LANES = COLS / 8, PER = 64 / LANES;   // lanes per row, rows per request
  u32x4_t w[R];
  // this lane's first row; waves: of the block
  static __device__ __forceinline__ int row0(int slab, int waves) { return (slab * waves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * (R * PER) + (threadIdx.x & 63) / LANES; }
  __device__ __forceinline__ void request(const bf16_t* W, int ld, int slice, int row0) {
    const bf16_t* p = W + (int64_t)row0 * ld + slice * COLS + threadIdx.x % LANES * 8;
#pragma unroll
    for (int j = 0; j < R; ++j) w[j] = ld_nt16(p + (int64_t)j * PER * ld);
  }
  // h: the slice's columns, f32 (LDS)
  __device__ __forceinline__ void multiply(const float* h, float* y, int row0) const {
    const int at = threadIdx.x % LANES * 8;
    const float4 lo = *reinterpret_cast<const float4*>(h + at), hi = *reinterpret_cast<const float4*>(h + at + 4);
    float s[R];
#pragma unroll
    for (int j = 0; j < R; ++j) {
      float v = lo.x * lo_bf(w[j][0]);
      v = fmaf(lo.y, hi_bf(w[j][0]), v);
      v = fmaf(lo.z, lo_bf(w[j][1]), v);
      v = fmaf(lo.w, hi_bf(w[j][1]), v);
      v = fmaf(hi.x, lo_bf(w[j][2]), v);
      v = fmaf(hi.y, hi_bf(w[j][2]), v);
      v = fmaf(hi.z, lo_bf(w[j][3]), v);
      s[j] = fmaf(hi.w, hi_bf(w[j][3]), v);
    }
#pragma unroll
    for (int j = 0; j < R; ++j) s[j] = LANES == 64 ? wave_sum(s[j]) : half_wave_sum(s[j]);
    if (threadIdx.x % LANES == 0) {
#pragma unroll
      for (int j = 0; j < R; ++j) y[row0 + j * PER] = s[j];
    }
  }
};

}  // namespace aha
