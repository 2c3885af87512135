// Decode matvecs of the routed experts (layered_prenorm.hip), as kernels_gemv_fused.hip: the chosen experts found in the prologue, their gate and up
// rows and the shared expert's streamed as one matrix behind LayerNorm; then down of all of them as one product over the concatenated activations.
#include "expert_choice.h"
#include "gemv_prologues.h"
#include "gemv_row_body.h"

namespace aha {

namespace {

// the `top` largest router logits, by every wave for itself (ties to the lower index, as moe_topk_kernel)
template <class F>
__device__ __forceinline__ void wave_topk(const float* z, int experts, int top, int lane, F&& each) {
  float v[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) v[j] = j * 64 + lane < experts ? z[j * 64 + lane] : -INFINITY;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int bi = 1 << 30;
#pragma unroll
    for (int j = 0; j < 16; ++j)
      if (v[j] > best) {
        best = v[j];
        bi = j * 64 + lane;
      }
    const float m = wave_max(best);
    if (best != m) bi = 1 << 30;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) bi = min(bi, __shfl_xor(bi, o, 64));
    bi = min(bi, experts - 1);
#pragma unroll
    for (int j = 0; j < 16; ++j)
      if (j * 64 + lane == bi) v[j] = -INFINITY;
    each(k, bi, m);
  }
}

// activation row = choice * effp + row inside the expert; choice top: the shared expert
template <int XP>
struct ExpertsUpPro {
  static constexpr bool MAPPED = true;
  LayerNormPro<XP> ln;
  GemvExperts e;
  int K, sel;   // sel, w: lane k holds the k-th choice
  float w;
  __device__ __forceinline__ void request(int tid) {
    ln.request(tid);
    const int lane = tid & 63;
    sel = 0;
    w = 1.f;
    wave_topk(e.z, e.experts, e.top, lane, [&](int k, int bi, float m) {
      if (lane == k) {
        sel = bi;
        w = 1.0f / (1.0f + expf(-m));
      }
    });
    if (blockIdx.x == 0 && tid < e.top) e.sel[tid] = sel;
  }
  __device__ __forceinline__ int choice(int& r) const {   // r -> row inside the choice
    int c = 0;
    for (; c < e.top && r >= e.effp; r -= e.effp) ++c;
    return c;
  }
  __device__ __forceinline__ const bf16_t* ptr(int row, int k) const {
    int r = __builtin_amdgcn_readfirstlane(row);   // (a wave's row)
    const int c = choice(r);
    const bf16_t* m = c < e.top ? (const bf16_t*)e.w_experts + (int64_t)__builtin_amdgcn_readlane(sel, c) * 2 * e.effp * K : (const bf16_t*)e.w_shared;
    return m + ((int64_t)(r >> 4) * 32 + (r & 15)) * K + k;
  }
  __device__ __forceinline__ float scale(int row) const {
    int r = __builtin_amdgcn_readfirstlane(row);
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), choice(r)));   // (lane top: 1)
  }
  __device__ __forceinline__ void stage(float* xs, float* red, int tid, int bid, int nchunks) { ln.stage(xs, red, tid, bid, nchunks); }
  __device__ __forceinline__ void finish(int, int) {}
};

// input vector: the choices' activations one after the other, then the shared expert's; weights: the experts' down matrices, then the shared one
template <int XP>   // K <= XP * 1024
struct ExpertsDownPro {
  static constexpr bool MAPPED = true;
  GemvExpertsDown d;
  const bf16_t* x;
  int K, sel;
  uint2 v[XP];
  __device__ __forceinline__ void request(int tid) {
    const int lane = tid & 63;
    sel = lane < d.top ? d.sel[lane] : 0;
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      const int k = (tid + j * GEMV_THREADS) * 4;
      v[j] = k < K ? *reinterpret_cast<const uint2*>(x + k) : make_uint2(0u, 0u);
    }
  }
  __device__ __forceinline__ int choice(int& k) const {   // k -> k inside the choice's own columns
    int c = 0;
    for (; c < d.top && k >= d.effp; k -= d.effp) ++c;
    return c;
  }
  __device__ __forceinline__ const bf16_t* ptr(int row, int k) const {
    if ((d.effp & 511) == 0) {   // the 512 columns of a wave's load belong to one choice
      const int r = __builtin_amdgcn_readfirstlane(row), k0 = __builtin_amdgcn_readfirstlane(k) & ~511;
      int in = k0;
      const int c = choice(in);
      const bf16_t* p = c < d.top ? (const bf16_t*)d.w_experts + ((int64_t)__builtin_amdgcn_readlane(sel, c) * d.n_rows + r) * d.effp : (const bf16_t*)d.w_shared + (int64_t)r * d.ffp;
      return p + max(in + k - k0, 0);   // (lanes past the end ask for k = 0)
    }
    const int c = choice(k);
    const int ex = __shfl(sel, c, 64);
    return c < d.top ? (const bf16_t*)d.w_experts + ((int64_t)ex * d.n_rows + row) * d.effp + k : (const bf16_t*)d.w_shared + (int64_t)row * d.ffp + k;
  }
  __device__ __forceinline__ void stage(float* xs, float* red, int tid, int bid, int nchunks) {
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      const int k = (tid + j * GEMV_THREADS) * 4;
      if (k < nchunks << 9) *xs4(xs, k) = bf4(v[j]);
    }
  }
  __device__ __forceinline__ void finish(int, int) {}
};

// i / effp, at most top (exact for i < 2^20: the nearest multiple is half a column away)
__device__ __forceinline__ int choice_of(int i, float inv_effp, int top) { return min((int)(((float)i + 0.5f) * inv_effp), top); }

// The row forms (gemv_row_body.h) of the 0.6B stack's widths: up to 64 experts, one logit per lane; K = 1024 (up), 3072 (down, whatever the choices' and the
// shared expert's parts of it).  Other widths have no instantiation and take the block form.
struct RowExpertsUpPro : RowLayerNormPro<2> {
  static constexpr bool MAPPED = true;
  const float* z;
  const bf16_t *w_experts, *w_shared;
  int experts, top, effp;
  int32_t* sel_out;
  int sel;   // sel, sw: lane k holds the k-th choice
  float sw, inv_effp;
  __device__ __forceinline__ void request() {
    const int lane = threadIdx.x & 63;
    float v = lane < experts ? z[lane] : -INFINITY;
    RowLayerNormPro<2>::request();
    sel = 0;
    sw = 1.f;
    v = choice_logit(v);
    for (int k = 0; k < top; ++k) {   // (wave_topk's choices)
      const float m = wave_max(v);
      const int bi = choice_lane(m, __ballot(v == m), experts);
      if (lane == bi) v = -INFINITY;
      if (lane == k) {
        sel = bi;
        sw = choice_weight(m);
      }
    }
    if (blockIdx.x == 0 && (int)threadIdx.x < top) sel_out[threadIdx.x] = sel;
  }
  __device__ __forceinline__ const bf16_t* ptr(int row, int u) const {
    const int c = __builtin_amdgcn_readfirstlane(choice_of(row, inv_effp, top)), r = __builtin_amdgcn_readfirstlane(row) - c * effp;   // (a wave's row)
    const bf16_t* m = c < top ? w_experts + (int64_t)__builtin_amdgcn_readlane(sel, c) * 2 * effp * 1024 : w_shared;
    return m + ((int64_t)(r >> 4) * 32 + (r & 15)) * 1024 + u * 512 + (threadIdx.x & 63) * 8;
  }
  __device__ __forceinline__ float scale(int row) const {
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(sw), __builtin_amdgcn_readfirstlane(choice_of(row, inv_effp, top))));   // (lane top: 1)
  }
};
__global__ __launch_bounds__(GEMV_THREADS) void gemv_row_experts_up_kernel(const float* z, const float* x, const void* w_experts, const void* w_shared, int experts_top, int effp, int N, int nblk,
                                                                           GemvArgs rest, GemvLayerNorm p, GemvExperts e) {
  RowExpertsUpPro pro;
  pro.x = x;
  pro.w = (const bf16_t*)p.w;
  pro.b = (const bf16_t*)p.b;
  pro.eps = p.eps;
  pro.width = p.width;
  pro.z = z;
  pro.w_experts = (const bf16_t*)w_experts;
  pro.w_shared = (const bf16_t*)w_shared;
  pro.experts = experts_top & 0xffff;
  pro.top = experts_top >> 16;
  pro.effp = effp;
  pro.inv_effp = 1.0f / (float)effp;
  pro.sel_out = e.sel;
  gemv_row_body<1, 2, GEMV_SILU_MUL>(rest, nullptr, nullptr, nullptr, N, (int)blockIdx.x, nblk, pro);
}

struct RowExpertsDownPro : RowNormPro<6, false> {
  static constexpr bool MAPPED = true;
  const int32_t* sel_in;
  const bf16_t *w_experts, *w_shared;
  int top, effp, n_rows;
  const bf16_t* base[6];   // of row 0
  int pitch[6];
  __device__ __forceinline__ void request() {
    const int lane = threadIdx.x & 63;
    const int sel = lane < top ? sel_in[lane] : 0;
    const float inv_effp = 1.0f / (float)effp;
    RowNormPro<6, false>::request();
    int c[6], ex[6];
#pragma unroll
    for (int u = 0; u < 6; ++u) c[u] = choice_of(u * 512 + lane * 8, inv_effp, top);   // (top: the shared expert's columns)
#pragma unroll
    for (int u = 0; u < 6; ++u) ex[u] = __shfl(sel, c[u], 64);   // (sel is 0 from lane top on)
#pragma unroll
    for (int u = 0; u < 6; ++u) {
      pitch[u] = c[u] < top ? effp : 3072 - top * effp;
      base[u] = (c[u] < top ? w_experts : w_shared) + ((int64_t)ex[u] * n_rows * effp + (u * 512 + lane * 8 - c[u] * effp));
    }
  }
  __device__ __forceinline__ const bf16_t* ptr(int row, int u) const { return base[u] + (int64_t)row * pitch[u]; }
};
__global__ __launch_bounds__(GEMV_THREADS) void gemv_row_experts_down_kernel(const void* x, const int32_t* sel, const void* w_experts, const void* w_shared, const float* res, int top, int effp, int N,
                                                                             int nblk, GemvArgs rest) {
  RowExpertsDownPro pro;
  pro.x = (const bf16_t*)x;
  pro.w = nullptr;
  pro.eps = 0.f;
  pro.sel_in = sel;
  pro.w_experts = (const bf16_t*)w_experts;
  pro.w_shared = (const bf16_t*)w_shared;
  pro.top = top;
  pro.effp = effp;
  pro.n_rows = N;
  gemv_row_body<1, 6, GEMV_AXPY_F32>(rest, nullptr, res, nullptr, N, (int)blockIdx.x, nblk, pro);
}

template <int R, int U, bool FAST, int XP>
__global__ __launch_bounds__(GEMV_THREADS) void gemv_experts_up_kernel(GemvArgs a, GemvLayerNorm p, GemvExperts e) {
  extern __shared__ __attribute__((aligned(16))) float xs[];
  ExpertsUpPro<XP> pro;
  pro.ln.p = p;
  pro.ln.K = pro.K = a.K;
  pro.e = e;
  gemv_body<R, U, GEMV_SILU_MUL, false, FAST>(a, xs, (int)blockIdx.x, (int)gridDim.x, [] {}, pro);
}
template <int R, int U, bool FAST, int XP>
__global__ __launch_bounds__(GEMV_THREADS) void gemv_experts_down_kernel(GemvArgs a, GemvExpertsDown d) {
  extern __shared__ __attribute__((aligned(16))) float xs[];
  ExpertsDownPro<XP> pro;
  pro.d = d;
  pro.x = (const bf16_t*)a.x;
  pro.K = a.K;
  gemv_body<R, U, GEMV_AXPY_F32, false, FAST>(a, xs, (int)blockIdx.x, (int)gridDim.x, [] {}, pro);
}

}  // namespace

void launch_gemv_experts_up(const GemvArgs& a, const GemvLayerNorm& p, const GemvExperts& e, hipStream_t st) {
  const GemvPlan pl = plan_gemv(a.N, a.K, GEMV_SILU_MUL);
  if (a.K == 1024 && e.experts <= 64 && pl.R == 1 && gemv_row_on()) {
    const int nblk = gemv_row_grid(a.N, 1);
    hipLaunchKernelGGL(gemv_row_experts_up_kernel, dim3(nblk), dim3(GEMV_THREADS), 0, st, e.z, p.x, e.w_experts, e.w_shared, e.experts | e.top << 16, e.effp, a.N, nblk, a, p, e);
    return;
  }
  dispatch_plan(pl, fused_fast(a, pl), [&](auto r, auto u, auto fast) {
    constexpr int R = decltype(r)::value, U = decltype(u)::value;
    constexpr bool FAST = decltype(fast)::value;
    if constexpr (R <= 2)   // (plan_gemv: two matrices, at most two rows each)
      by_xp<FAST>(a.K, [&](auto xp) { hipLaunchKernelGGL((gemv_experts_up_kernel<R, U, FAST, decltype(xp)::value>), dim3(pl.grid), dim3(GEMV_THREADS), fused_lds(a), st, a, p, e); });
  });
}

void launch_gemv_experts_down(const GemvArgs& a, const GemvExpertsDown& d, hipStream_t st) {
  const GemvPlan pl = plan_gemv(a.N, a.K, GEMV_AXPY_F32);
  if (a.K == 3072 && pl.R == 1 && d.n_rows == a.N && gemv_row_on()) {
    const int nblk = gemv_row_grid(a.N, 1);
    hipLaunchKernelGGL(gemv_row_experts_down_kernel, dim3(nblk), dim3(GEMV_THREADS), 0, st, a.x, d.sel, d.w_experts, d.w_shared, a.res_f32, d.top, d.effp, a.N, nblk, a);
    return;
  }
  dispatch_plan(pl, fused_fast(a, pl), [&](auto r, auto u, auto fast) {
    constexpr int R = decltype(r)::value, U = decltype(u)::value;
    constexpr bool FAST = decltype(fast)::value;
    auto run = [&](auto xp) { hipLaunchKernelGGL((gemv_experts_down_kernel<R, U, FAST, decltype(xp)::value>), dim3(pl.grid), dim3(GEMV_THREADS), fused_lds(a), st, a, d); };
    if (FAST && a.K <= 4096) run(std::integral_constant<int, FAST ? 4 : 16>{});
    else run(std::integral_constant<int, 16>{});
  });
}

}  // namespace aha
