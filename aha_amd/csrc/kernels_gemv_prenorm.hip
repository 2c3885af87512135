// Decode matvecs of the pre-norm stacks (layered_prenorm.hip), as kernels_gemv_fused.hip:
//   LayerNorm:    h = (x - mean) / sqrt(var + eps) * w + b
//   parts norm:   h = g / rms(g's part) * w, the sums of squares prepared by the recurrence's step kernel
#include "gemv_prologues.h"
#include "gemv_row_body.h"

namespace aha {

namespace {

template <int XP>
struct PartsNormPro {
  GemvPartsNorm p;
  int K;
  float4 g[XP];
  uint2 w[XP];
  __device__ __forceinline__ void request(int tid) {
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      const int k = (tid + j * GEMV_THREADS) * 4;
      g[j] = make_float4(0.f, 0.f, 0.f, 0.f);
      w[j] = make_uint2(0u, 0u);
      if (k < p.n) {
        g[j] = *reinterpret_cast<const float4*>(p.g + k);
        w[j] = *reinterpret_cast<const uint2*>((const bf16_t*)p.w + k);
      }
    }
  }
  __device__ __forceinline__ void stage(float* xs, float* red, int tid, int bid, int nchunks) {
    const int per = p.n / p.parts >> 4;   // 16-column sums per part
    float* rinv = xs + (nchunks << 9) + 16;
    for (int q = tid >> 6; q < p.parts; q += GEMV_WAVES) {
      float s = 0.f;
      for (int i = tid & 63; i < per; i += 64) s += p.ssq[q * per + i];
      s = wave_sum(s);
      if ((tid & 63) == 0) rinv[q] = 1.0f / sqrtf(s / (float)p.part + p.eps);
    }
    __syncthreads();
    const int pw = p.n / p.parts;
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      const int k = (tid + j * GEMV_THREADS) * 4;
      if (k >= (nchunks << 9)) continue;
      const float r = k < p.n ? rinv[k / pw] : 0.f;   // (a part is a whole number of 16-column pieces)
      const float4 w4 = bf4(w[j]);
      *xs4(xs, k) = make_float4(g[j].x * r * w4.x, g[j].y * r * w4.y, g[j].z * r * w4.z, g[j].w * r * w4.w);
    }
  }
  __device__ __forceinline__ void finish(int, int) {}
};

template <int R, int U, int EPI, bool FAST, int XP>
__global__ __launch_bounds__(GEMV_THREADS) void gemv_layernorm_kernel(GemvArgs a, GemvLayerNorm p) {
  extern __shared__ __attribute__((aligned(16))) float xs[];
  LayerNormPro<XP> pro;
  pro.p = p;
  pro.K = a.K;
  gemv_body<R, U, EPI, false, FAST>(a, xs, (int)blockIdx.x, (int)gridDim.x, [] {}, pro);
}
template <int R, int U, bool FAST, int XP>
__global__ __launch_bounds__(GEMV_THREADS) void gemv_partsnorm_kernel(GemvArgs a, GemvPartsNorm p) {
  extern __shared__ __attribute__((aligned(16))) float xs[];
  PartsNormPro<XP> pro;
  pro.p = p;
  pro.K = a.K;
  gemv_body<R, U, GEMV_AXPY_F32, false, FAST>(a, xs, (int)blockIdx.x, (int)gridDim.x, [] {}, pro);
}

// parts norm for K = n = 512 U (instantiated: 2048) in parts of 256 columns: their 16 sums of squares each are added up by the 16 lanes of a DPP row
template <int U>
struct RowPartsNormPro {
  const float *g, *ssq;
  const bf16_t* w;
  float eps;
  int part;
  float4 v[U][2];
  u32x4_t wr[U];
  float sq[U / 2];
  __device__ __forceinline__ void request() {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < U / 2; ++j) sq[j] = ssq[j * 64 + lane];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      v[u][0] = *reinterpret_cast<const float4*>(g + u * 512 + lane * 8);
      v[u][1] = *reinterpret_cast<const float4*>(g + u * 512 + lane * 8 + 4);
      wr[u] = ld16(w + u * 512 + lane * 8);
    }
  }
  __device__ __forceinline__ void make(float (&h)[U][8]) {
    float sum[2 * U];   // of a part
#pragma unroll
    for (int j = 0; j < U / 2; ++j) {
      float s = sq[j];
      s += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(s), 0x128, 0xf, 0xf, false));
      s += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(s), 0x124, 0xf, 0xf, false));
      s += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(s), 0x122, 0xf, 0xf, false));
      s += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(s), 0x121, 0xf, 0xf, false));
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[j * 4 + i] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s), i * 16));
    }
    const bool hi = (threadIdx.x & 63) >= 32;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float s0 = sum[2 * u], s1 = sum[2 * u + 1];   // (values: a choice between array members becomes an array in LDS)
      const float r = 1.0f / sqrtf((hi ? s1 : s0) / (float)part + eps);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        h[u][4 * i] = v[u][i].x * r * lo_bf(wr[u][2 * i]);
        h[u][4 * i + 1] = v[u][i].y * r * hi_bf(wr[u][2 * i]);
        h[u][4 * i + 2] = v[u][i].z * r * lo_bf(wr[u][2 * i + 1]);
        h[u][4 * i + 3] = v[u][i].w * r * hi_bf(wr[u][2 * i + 1]);
      }
    }
  }
};

template <int R, int U, int EPI>
__global__ __launch_bounds__(GEMV_THREADS) void gemv_row_layernorm_kernel(const float* x, const void* W, const void* w, const void* b, float eps, int width, int N, int nblk, GemvArgs rest) {
  RowLayerNormPro<U> pro{x, (const bf16_t*)w, (const bf16_t*)b, eps, width};
  gemv_row_body<R, U, EPI>(rest, W, nullptr, nullptr, N, (int)blockIdx.x, nblk, pro);
}
template <int U>
__global__ __launch_bounds__(GEMV_THREADS) void gemv_row_partsnorm_kernel(const float* g, const float* ssq, const void* w, const void* W, const float* res, float eps, int part, int N, int nblk,
                                                                          GemvArgs rest) {
  RowPartsNormPro<U> pro{g, ssq, (const bf16_t*)w, eps, part};
  gemv_row_body<1, U, GEMV_AXPY_F32>(rest, W, res, nullptr, N, (int)blockIdx.x, nblk, pro);
}

}  // namespace

void launch_gemv_layernorm(const GemvArgs& a, const GemvLayerNorm& p, GemvEpi epi, hipStream_t st) {
  const GemvPlan pl = plan_gemv(a.N, a.K, epi);
  if (a.K == 1024 && pl.R <= 2 && a.W2 == nullptr && gemv_row_on()) {   // (gemv_row_body.h; the one width that is instantiated)
    auto row = [&](auto r) {
      constexpr int R = decltype(r)::value;
      const int nblk = gemv_row_grid(a.N, R);
      if (epi != GEMV_SILU_MUL)
        hipLaunchKernelGGL((gemv_row_layernorm_kernel<R, 2, GEMV_PARTIAL_F32>), dim3(nblk), dim3(GEMV_THREADS), 0, st, p.x, a.W, p.w, p.b, p.eps, p.width, a.N, nblk, a);
      else
        hipLaunchKernelGGL((gemv_row_layernorm_kernel<R, 2, GEMV_SILU_MUL>), dim3(nblk), dim3(GEMV_THREADS), 0, st, p.x, a.W, p.w, p.b, p.eps, p.width, a.N, nblk, a);
    };
    if (pl.R == 2) row(std::integral_constant<int, 2>{});
    else row(std::integral_constant<int, 1>{});
    return;
  }
  const dim3 grid(pl.grid), block(GEMV_THREADS);
  dispatch_plan(pl, fused_fast(a, pl), [&](auto r, auto u, auto fast) {
    constexpr int R = decltype(r)::value, U = decltype(u)::value;
    constexpr bool FAST = decltype(fast)::value;
    by_xp<FAST>(a.K, [&](auto xp) {
      constexpr int XP = decltype(xp)::value;
      if (epi != GEMV_SILU_MUL) hipLaunchKernelGGL((gemv_layernorm_kernel<R, U, GEMV_PARTIAL_F32, FAST, XP>), grid, block, fused_lds(a), st, a, p);
      else if constexpr (R <= 2) hipLaunchKernelGGL((gemv_layernorm_kernel<R, U, GEMV_SILU_MUL, FAST, XP>), grid, block, fused_lds(a), st, a, p);   // (plan_gemv: two matrices, at most two rows each)
    });
  });
}

void launch_gemv_partsnorm(const GemvArgs& a, const GemvPartsNorm& p, hipStream_t st) {
  const GemvPlan pl = plan_gemv(a.N, a.K, GEMV_AXPY_F32);
  if (a.K == 2048 && p.n == a.K && pl.R == 1 && p.n == p.parts * 256 && gemv_row_on()) {
    hipLaunchKernelGGL(gemv_row_partsnorm_kernel<4>, dim3(gemv_row_grid(a.N, 1)), dim3(GEMV_THREADS), 0, st, p.g, p.ssq, p.w, a.W, a.res_f32, p.eps, p.part, a.N, gemv_row_grid(a.N, 1), a);
    return;
  }
  dispatch_plan(pl, fused_fast(a, pl), [&](auto r, auto u, auto fast) {
    constexpr int R = decltype(r)::value, U = decltype(u)::value;
    constexpr bool FAST = decltype(fast)::value;
    auto run = [&](auto xp) {
      hipLaunchKernelGGL((gemv_partsnorm_kernel<R, U, FAST, decltype(xp)::value>), dim3(pl.grid), dim3(GEMV_THREADS), fused_lds(a) + (size_t)p.parts * 4, st, a, p);
    };
    if (FAST && a.K <= 4096) run(std::integral_constant<int, FAST ? 4 : 16>{});
    else run(std::integral_constant<int, 16>{});
  });
}

}  // namespace aha
