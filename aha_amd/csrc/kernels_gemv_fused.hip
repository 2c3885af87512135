// Decode matvecs of the layer-list decoders (layered.hip): the weight stream of kernels_gemv.hip behind another prologue.
//   postnorm + input convolution:  h = x + conv(x),  x = s / sqrt(mean(s^2) + eps) * (1 + w),  s = alpha x_old + sublayer output (f32)
//       every block rebuilds h (the matvec's input) in LDS; what the convolution takes from earlier tokens arrives as ONE vector, the
//       weighted sum prepared when those tokens ran (ConvIn::hist).  Block j < XP also writes column group j of x and, behind its weight
//       stream, of the sequence's new history and the next token's weighted sum.
//   attention merge:               h = the split-KV attention partials of a decode step joined (attn_decode_body.h, DEFER)
//   PolyNorm:                      h = a N(z) + b N(z^2) + c N(z^3) + e: the three row sums in the prologue
#include "gemv_prologues.h"
#include "gemv_row_body.h"
#include "oproj_slices.h"

namespace aha {

namespace {

// XP groups of 4 elements per thread are requested ahead of the weights (K <= XP * 1024)
template <int XP>
struct PostNormPro {
  GemvPostNorm p;
  int K;
  float eps;
  float4 s[XP], pre[XP];
  uint2 nw[XP], wl[XP];
  int slot, pos0;
  const float* hin;
  __device__ __forceinline__ void request(int tid) {
    slot = p.entry.slot;
    pos0 = p.entry.pos0;
    const int taps = p.conv.taps;
    hin = p.conv.hist + (int64_t)slot * p.conv.slot_stride + (int64_t)p.entry.hist_in * taps * p.conv.ldw;
    const float* pr = hin + (int64_t)(taps - 1) * p.conv.ldw;
    const bf16_t* w_last = (const bf16_t*)p.conv.w + (int64_t)(taps - 1) * p.conv.ldw;
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      const int k = (tid + j * GEMV_THREADS) * 4;
      s[j] = pre[j] = make_float4(0.f, 0.f, 0.f, 0.f);
      nw[j] = wl[j] = make_uint2(0u, 0u);
      if (k < K) {
        s[j] = *reinterpret_cast<const float4*>(p.s + k);
        nw[j] = *reinterpret_cast<const uint2*>((const bf16_t*)p.norm_w + k);
        wl[j] = *reinterpret_cast<const uint2*>(w_last + k);
        if (pos0 > 0) pre[j] = *reinterpret_cast<const float4*>(pr + k);
      }
    }
  }
  __device__ __forceinline__ void stage(float* xs, float* red, int tid, int bid, int nchunks) {
    float ss[1] = {0.f};
#pragma unroll
    for (int j = 0; j < XP; ++j) ss[0] += (s[j].x * s[j].x + s[j].y * s[j].y) + (s[j].z * s[j].z + s[j].w * s[j].w);   // (pad columns are zero)
    block_sums(ss, red, tid);
    const float rinv = 1.0f / sqrtf(ss[0] / (float)p.width + eps);
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      const int k = (tid + j * GEMV_THREADS) * 4;
      if (k >= (nchunks << 9)) continue;
      const float4 n4 = bf4(nw[j]), w4 = bf4(wl[j]);
      float4 x, h;
      x.x = s[j].x * rinv * (1.f + n4.x); x.y = s[j].y * rinv * (1.f + n4.y); x.z = s[j].z * rinv * (1.f + n4.z); x.w = s[j].w * rinv * (1.f + n4.w);
      h.x = x.x + fmaf(w4.x, x.x, pre[j].x); h.y = x.y + fmaf(w4.y, x.y, pre[j].y);
      h.z = x.z + fmaf(w4.z, x.z, pre[j].z); h.w = x.w + fmaf(w4.w, x.w, pre[j].w);
      *xs4(xs, k) = h;
      if (bid == j && k < K) *reinterpret_cast<float4*>(p.x_out + k) = x;
    }
  }
  __device__ __forceinline__ void finish(int tid, int bid) {
    const int k = (tid + bid * GEMV_THREADS) * 4, taps = p.conv.taps;
    if (bid >= XP || k >= K) return;
    const int64_t ldw = p.conv.ldw;
    float* hout = p.conv.hist + (int64_t)slot * p.conv.slot_stride + (int64_t)p.entry.hist_out * taps * ldw;
    // history: row i = the input i + 1 tokens back as the next token sees it; last row = their weighted sum
    float4 nx = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 cur = *reinterpret_cast<const float4*>(p.x_out + k);   // (this thread's own store)
    for (int i = 0; i < taps - 1; ++i) {
      const float4 wj = bf4(*reinterpret_cast<const uint2*>((const bf16_t*)p.conv.w + (int64_t)(taps - 2 - i) * ldw + k));
      *reinterpret_cast<float4*>(hout + (int64_t)i * ldw + k) = cur;
      nx.x = fmaf(wj.x, cur.x, nx.x); nx.y = fmaf(wj.y, cur.y, nx.y); nx.z = fmaf(wj.z, cur.z, nx.z); nx.w = fmaf(wj.w, cur.w, nx.w);
      if (i + 1 < taps - 1) cur = pos0 - 1 - i >= 0 ? *reinterpret_cast<const float4*>(hin + (int64_t)i * ldw + k) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    *reinterpret_cast<float4*>(hout + (int64_t)(taps - 1) * ldw + k) = nx;
  }
};

template <int XP>
struct PolyNormPro {
  const float* zp;
  float ca, cb, cc, ce, eps;
  int ff, K;
  float4 z[XP];
  __device__ __forceinline__ void request(int tid) {
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      const int k = (tid + j * GEMV_THREADS) * 4;
      z[j] = k < K ? *reinterpret_cast<const float4*>(zp + k) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  __device__ __forceinline__ void stage(float* xs, float* red, int tid, int bid, int nchunks) {
    float ss[3] = {0.f, 0.f, 0.f};
    auto add = [&](float v) {
      const float v2 = v * v, v4 = v2 * v2;
      ss[0] += v2;
      ss[1] += v4;
      ss[2] = fmaf(v4, v2, ss[2]);
    };
#pragma unroll
    for (int j = 0; j < XP; ++j) { add(z[j].x); add(z[j].y); add(z[j].z); add(z[j].w); }   // (pad columns are zero)
    block_sums(ss, red, tid);
    const float inv = 1.0f / (float)ff;
    const float r1 = ca / sqrtf(ss[0] * inv + eps), r2 = cb / sqrtf(ss[1] * inv + eps), r3 = cc / sqrtf(ss[2] * inv + eps);
    auto act = [&](float v) { return fmaf(v, fmaf(v, fmaf(v, r3, r2), r1), ce); };
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      const int k = (tid + j * GEMV_THREADS) * 4;
      if (k >= (nchunks << 9)) continue;
      *xs4(xs, k) = make_float4(k < ff ? act(z[j].x) : 0.f, k + 1 < ff ? act(z[j].y) : 0.f, k + 2 < ff ? act(z[j].z) : 0.f, k + 3 < ff ? act(z[j].w) : 0.f);
    }
  }
  __device__ __forceinline__ void finish(int, int) {}
};

// Every block joins all heads: nsplit x 16 KB (32 heads) from L2, requested ahead of the first weight tile -- under a microsecond of it shows.  A wave's
// group j of 256 columns is two heads; weights and normalisation per head are recomputed by its 32 threads.
template <int XP, int MS>
struct MergePro {
  GemvMerge p;
  int K;
  float4 v[XP][MS];
  float2 ml[XP][MS];
  __device__ __forceinline__ void request(int tid) {
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      const int k = min((tid + j * GEMV_THREADS) * 4, K - 4), head = k >> 7;
#pragma unroll
      for (int s = 0; s < MS; ++s) {
        const int64_t at = (int64_t)min(s, p.nsplit - 1) * p.heads;
        ml[j][s] = *reinterpret_cast<const float2*>(p.part_ml + (at + head) * 2);
        v[j][s] = *reinterpret_cast<const float4*>(p.part_o + at * 128 + k);
      }
    }
  }
  __device__ __forceinline__ void stage(float* xs, float*, int tid, int, int nchunks) {
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      const int k = (tid + j * GEMV_THREADS) * 4;
      if (k >= (nchunks << 9)) continue;
      float M = ml[j][0].x;
#pragma unroll
      for (int s = 1; s < MS; ++s) M = fmaxf(M, ml[j][s].x);   // (surplus slots repeat the last split)
      float4 h = make_float4(0.f, 0.f, 0.f, 0.f);
      float z = 0.f;
#pragma unroll
      for (int s = 0; s < MS; ++s) {
        const float w = s < p.nsplit && ml[j][s].x != -INFINITY ? __expf(ml[j][s].x - M) : 0.f;
        z = fmaf(w, ml[j][s].y, z);
        h.x = fmaf(w, v[j][s].x, h.x); h.y = fmaf(w, v[j][s].y, h.y); h.z = fmaf(w, v[j][s].z, h.z); h.w = fmaf(w, v[j][s].w, h.w);
      }
      const float inv = 1.0f / z;
      // the attention output tensor is bf16
      *xs4(xs, k) = k < K ? make_float4(rbf(h.x * inv), rbf(h.y * inv), rbf(h.z * inv), rbf(h.w * inv)) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  __device__ __forceinline__ void finish(int, int) {}
};

// The same for K = 512 * U: a thread's group j of 4 columns is merged as above, the result read back from LDS as the columns of the lane's weights.
template <int U, int MS>
struct RowMergePro {
  static constexpr int K = U * 512, XP = K / (4 * GEMV_THREADS);
  const float* part_o;
  const float* part_ml;
  int nsplit;
  float* xs;   // LDS, K floats
  float4 v[XP][MS];
  float2 ml[XP][MS];
  __device__ __forceinline__ void request() {
#pragma unroll
    for (int s = 0; s < MS; ++s) {
      const int64_t at = min(s, nsplit - 1) * (K / 128);   // (surplus slots repeat the last split: its lines are on their way)
#pragma unroll
      for (int j = 0; j < XP; ++j) ml[j][s] = *reinterpret_cast<const float2*>(part_ml + at * 2 + (j * GEMV_THREADS + threadIdx.x) / 32 * 2);
    }
#pragma unroll
    for (int s = 0; s < MS; ++s) {
      const int64_t at = min(s, nsplit - 1) * K;
#pragma unroll
      for (int j = 0; j < XP; ++j) v[j][s] = *reinterpret_cast<const float4*>(part_o + at + (j * GEMV_THREADS + threadIdx.x) * 4);
    }
  }
  __device__ __forceinline__ void make(float (&h)[U][8]) {
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      float M = ml[j][0].x;
#pragma unroll
      for (int s = 1; s < MS; ++s) M = fmaxf(M, ml[j][s].x);
      float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
      float z = 0.f;
#pragma unroll
      for (int s = 0; s < MS; ++s) {
        const float w = s < nsplit && ml[j][s].x != -INFINITY ? __expf(ml[j][s].x - M) : 0.f;
        z = fmaf(w, ml[j][s].y, z);
        o.x = fmaf(w, v[j][s].x, o.x); o.y = fmaf(w, v[j][s].y, o.y); o.z = fmaf(w, v[j][s].z, o.z); o.w = fmaf(w, v[j][s].w, o.w);
      }
      const float inv = 1.0f / z;
      *xs4(xs, (j * GEMV_THREADS + threadIdx.x) * 4) = make_float4(rbf(o.x * inv), rbf(o.y * inv), rbf(o.z * inv), rbf(o.w * inv));
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float4 lo = *xs4(xs, u * 512 + lane * 8), hi = *xs4(xs, u * 512 + lane * 8 + 4);
      h[u][0] = lo.x; h[u][1] = lo.y; h[u][2] = lo.z; h[u][3] = lo.w;
      h[u][4] = hi.x; h[u][5] = hi.y; h[u][6] = hi.z; h[u][7] = hi.w;
    }
  }
};

template <int U, int MS>
__global__ __launch_bounds__(GEMV_THREADS) void gemv_row_merge_kernel(const float* part_o, const float* part_ml, const void* W, const void* residual, unsigned long long* trace, int N, int nsplit, int nblk,
                                                                      GemvArgs rest) {
  __shared__ __attribute__((aligned(16))) float xs[U * 512];
  RowMergePro<U, MS> pro{part_o, part_ml, nsplit, xs};
  gemv_row_body<1, U, GEMV_RESIDUAL>(rest, W, residual, trace, N, (int)blockIdx.x, nblk, pro);
}
// o_proj behind split attention, in slices (oproj_slices.h): block (two kv heads, 16 rows) merges the partials of its four heads alone, two KB a split and
// block, where a block of gemv_row_merge_kernel merges all of them (eight splits: 64 KB, twice per CU).  A wave per head: lane l < 16 has split l for the weights,
// every lane two columns of all splits.  2048 + 256 positions of 0.6B: attention + o_proj + gate + up 6.5 + 4.0 + 4.4 us with eight splits, 5.5 + 3.4 + 4.8 with sixteen
// in slices (166.4 -> 159.5 ms in all); more splits cost the merge of all heads what they save the attention.
__global__ __launch_bounds__(256) void oproj_slice_kernel(const float* part_o, const float* part_ml, const void* W, float* y, int heads, int n, int nsplit) {
  __shared__ __attribute__((aligned(16))) float hs[512];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), slice = (int)blockIdx.x, head = slice * 4 + wave;
  const float2 ml = *reinterpret_cast<const float2*>(part_ml + (min(lane & 15, nsplit - 1) * heads + head) * 2);
  float2 v[16];
#pragma unroll
  for (int s = 0; s < 16; ++s) v[s] = *reinterpret_cast<const float2*>(part_o + (min(s, nsplit - 1) * heads + head) * 128 + lane * 2);   // (surplus ones repeat the last split)
  OprojRows<4, 512> rows;
  const int row0 = rows.row0((int)blockIdx.y, 4);
  __builtin_amdgcn_sched_barrier(0);
  rows.request((const bf16_t*)W, heads * 128, slice, row0);
  __builtin_amdgcn_sched_barrier(0);
  float M = ml.x;
#pragma unroll
  for (int d = 8; d >= 1; d >>= 1) M = fmaxf(M, __shfl_xor(M, d, 64));
  const float e = (lane & 15) < nsplit && ml.x != -INFINITY ? __expf(ml.x - M) : 0.f;
  float z = e * ml.y;
#pragma unroll
  for (int d = 8; d >= 1; d >>= 1) z += __shfl_xor(z, d, 64);
  float2 o = make_float2(0.f, 0.f);
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    const float w = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(e), s));
    o.x = fmaf(w, v[s].x, o.x);
    o.y = fmaf(w, v[s].y, o.y);
  }
  const float inv = 1.0f / z;
  *reinterpret_cast<float2*>(hs + wave * 128 + lane * 2) = make_float2(rbf(o.x * inv), rbf(o.y * inv));   // (the attention output tensor is bf16)
  __syncthreads();
  rows.multiply(hs, y + slice * n, row0);
}
template <int P>
__global__ __launch_bounds__(GEMV_THREADS) void gemv_row_slices_kernel(const void* x, const float* parts, const void* W, const void* norm_w, void* x_out, unsigned long long* trace, int N, float eps, int nblk, GemvArgs rest) {
  __shared__ __attribute__((aligned(16))) float xs[1024 + 4];
  RowSlicesPro<P> pro{(const bf16_t*)x, (const bf16_t*)norm_w, parts, (bf16_t*)x_out, eps, (int)blockIdx.x, xs};
  gemv_row_body<1, 2, GEMV_SILU_MUL>(rest, W, nullptr, trace, N, (int)blockIdx.x, nblk, pro);
}
template <int R, int U, bool FAST, int XP, int MS, int KX = 0>
__global__ __launch_bounds__(GEMV_THREADS) void gemv_merge_kernel(const float* part_o, const float* part_ml, const void* W, const void* residual, unsigned long long* trace, int N, int K, int nsplit, int nblk,
                                                                    GemvArgs rest) {
  extern __shared__ __attribute__((aligned(16))) float xs[];
  MergePro<XP, MS> pro;
  if (KX > 0) K = KX * 2048;
  pro.p = GemvMerge{part_o, part_ml, nsplit, K >> 7};
  pro.K = K;
  gemv_body<R, U, GEMV_RESIDUAL, false, FAST, KX>(gemv_args<GEMV_RESIDUAL>(rest, nullptr, W, nullptr, residual, trace, N, K, 0.f), xs, (int)blockIdx.x, nblk, [] {}, pro);
}
template <int R, int U, int EPI, bool FAST, int XP>
__global__ __launch_bounds__(GEMV_THREADS) void gemv_postnorm_kernel(GemvArgs a, GemvPostNorm p) {
  extern __shared__ __attribute__((aligned(16))) float xs[];
  PostNormPro<XP> pro;
  pro.p = p;
  pro.K = a.K;
  pro.eps = a.eps;
  gemv_body<R, U, EPI, false, FAST>(a, xs, (int)blockIdx.x, (int)gridDim.x, [] {}, pro);
}
template <int R, int U, int EPI, bool FAST, int XP>
__global__ __launch_bounds__(GEMV_THREADS) void gemv_polynorm_kernel(GemvArgs a, PolyNormArgs p) {
  extern __shared__ __attribute__((aligned(16))) float xs[];
  PolyNormPro<XP> pro;
  pro.zp = (const float*)p.z;
  pro.ca = p.coef[0]; pro.cb = p.coef[1]; pro.cc = p.coef[2]; pro.ce = p.coef[3];
  pro.eps = p.eps;
  pro.ff = p.ff;
  pro.K = a.K;
  gemv_body<R, U, EPI, false, FAST>(a, xs, (int)blockIdx.x, (int)gridDim.x, [] {}, pro);
}

}  // namespace

bool gemv_fused_ok(int width_ld, int ff_ld) { return width_ld <= 8192 && ff_ld <= 15872; }   // (64 KB of dynamic LDS for the input vector)

void launch_gemv_postnorm(const GemvArgs& a, const GemvPostNorm& p, GemvEpi epi, hipStream_t st) {
  const GemvPlan pl = plan_gemv(a.N, a.K, epi);
  const size_t lds = (size_t)((a.K + 511) / 512) * 512 * 4 + 64;
  const dim3 grid(pl.grid), block(GEMV_THREADS);
  dispatch_plan(pl, a.K % 512 == 0 && a.K / 512 % (pl.U >= 8 ? 8 : pl.U >= 4 && pl.R == 4 ? 4 : pl.U >= 2 ? 2 : 1) == 0, [&](auto r, auto u, auto fast) {
    constexpr int R = decltype(r)::value, U = decltype(u)::value;
    constexpr bool FAST = decltype(fast)::value;
    auto run = [&](auto xp) {
      constexpr int XP = decltype(xp)::value;
      if (epi == GEMV_AXPY_F32) hipLaunchKernelGGL((gemv_postnorm_kernel<R, U, GEMV_AXPY_F32, FAST, XP>), grid, block, lds, st, a, p);
      else hipLaunchKernelGGL((gemv_postnorm_kernel<R, U, GEMV_PARTIAL_F32, FAST, XP>), grid, block, lds, st, a, p);
    };
    if (a.K <= 1024) run(std::integral_constant<int, 1>{});
    else if (a.K <= 4096) run(std::integral_constant<int, 4>{});
    else run(std::integral_constant<int, 8>{});
  });
}

void launch_gemv_merge(const GemvArgs& a, const GemvMerge& p, hipStream_t st) {
  const GemvPlan pl = plan_gemv(a.N, a.K, GEMV_RESIDUAL);
  if (a.K == 2048 && pl.R == 1 && gemv_row_on()) {   // (gemv_row_body.h; the one width that is instantiated)
    auto row = [&](auto ms) {
      hipLaunchKernelGGL((gemv_row_merge_kernel<4, decltype(ms)::value>), dim3(gemv_row_grid(a.N, 1)), dim3(GEMV_THREADS), 0, st, p.part_o, p.part_ml, a.W, a.residual, a.trace, a.N, p.nsplit, gemv_row_grid(a.N, 1), a);
    };
    if (p.nsplit > 4) row(std::integral_constant<int, 8>{});
    else if (p.nsplit > 2) row(std::integral_constant<int, 4>{});
    else row(std::integral_constant<int, 2>{});
    return;
  }
  auto go = [&](auto r, auto u) {
    constexpr int R = decltype(r)::value, U = decltype(u)::value;
    const dim3 grid(pl.grid), block(GEMV_THREADS);
    auto run = [&](auto fast, auto xp, auto ms) {
      hipLaunchKernelGGL((gemv_merge_kernel<R, U, decltype(fast)::value, decltype(xp)::value, decltype(ms)::value>), grid, block, fused_lds(a), st, p.part_o, p.part_ml, a.W, a.residual, a.trace, a.N, a.K, p.nsplit, pl.grid,
                         a);
    };
    using std::integral_constant;
    auto by_k = [&](auto fast) {
      if constexpr (U == 8 && decltype(fast)::value)
        if (a.K == 4096) {
          hipLaunchKernelGGL((gemv_merge_kernel<R, U, true, 4, 4, 2>), grid, block, fused_lds(a), st, p.part_o, p.part_ml, a.W, a.residual, a.trace, a.N, a.K, p.nsplit, pl.grid, a);
          return;
        }
      if (a.K > 2048) run(fast, integral_constant<int, 4>{}, integral_constant<int, 4>{});
      else if (p.nsplit > 4) run(fast, integral_constant<int, 2>{}, integral_constant<int, 8>{});
      else run(fast, integral_constant<int, 2>{}, integral_constant<int, 4>{});
    };
    if (a.K % (512 * U) != 0) by_k(std::false_type{});
    else by_k(std::true_type{});
  };
  using std::integral_constant;   // (the load groups of kernels_gemv.hip; an output this long with K <= 4096 has 16 loads in flight per wave)
  if (pl.R == 4) go(integral_constant<int, 4>{}, integral_constant<int, 4>{});
  else if (pl.R == 2) pl.U >= 8 ? go(integral_constant<int, 2>{}, integral_constant<int, 8>{}) : go(integral_constant<int, 2>{}, integral_constant<int, 2>{});
  else if (pl.U >= 8) go(integral_constant<int, 1>{}, integral_constant<int, 8>{});
  else if (pl.U >= 4) go(integral_constant<int, 1>{}, integral_constant<int, 4>{});
  else go(integral_constant<int, 1>{}, integral_constant<int, 1>{});
}

// The sizes that both kernels and the norm behind them are written for, which are the only ones measured: a slice of 256 columns and a wave's 128-dim heads, 1024 columns of
// x, a float4 per thread (RowSlicesPro).  Other stacks keep o_proj in a launch of its own.  What decides is not the sizes but that o_proj's 4 MB take less time than the
// link of the chain that its launch is; at 2048 columns they are 8 to 16 MB, and the norm would read twice the slices in front of gate + up.
bool oproj_slices_ok(int width, int heads, int kv_heads, int head_dim, int ff) {
  return width == 1024 && heads == 16 && kv_heads == 8 && head_dim == 128 && gemv_row_groups(ff, width, GEMV_SILU_MUL) == 2 && plan_gemv(ff, width, GEMV_SILU_MUL).R == 1;
}
void launch_oproj_slices(const GemvMerge& p, const void* W, float* y, int n, hipStream_t st) {
  hipLaunchKernelGGL(oproj_slice_kernel, dim3((unsigned)(p.heads / 4), (unsigned)(n / 16)), dim3(256), 0, st, p.part_o, p.part_ml, W, y, p.heads, n, p.nsplit);
}
void launch_gemv_slices(const GemvArgs& a, const float* parts, int n, void* x_out, hipStream_t st) {
  const int nblk = gemv_row_grid(a.N, 1);
  auto go = [&](auto k) { hipLaunchKernelGGL(k, dim3(nblk), dim3(GEMV_THREADS), 0, st, a.x, parts, a.W, a.norm_w, x_out, a.trace, a.N, a.eps, nblk, a); };
  if (n == 4) go(gemv_row_slices_kernel<4>);
  else go(gemv_row_slices_kernel<8>);
}

void launch_gemv_polynorm(const GemvArgs& a, const PolyNormArgs& p, GemvEpi epi, hipStream_t st) {
  const GemvPlan pl = plan_gemv(a.N, a.K, epi);
  const size_t lds = (size_t)((a.K + 511) / 512) * 512 * 4 + 64;
  const dim3 grid(pl.grid), block(GEMV_THREADS);
  dispatch_plan(pl, a.K % 512 == 0 && a.K / 512 % (pl.U >= 8 ? 8 : pl.U >= 4 && pl.R == 4 ? 4 : pl.U >= 2 ? 2 : 1) == 0, [&](auto r, auto u, auto fast) {
    constexpr int R = decltype(r)::value, U = decltype(u)::value;
    constexpr bool FAST = decltype(fast)::value;
    auto run = [&](auto xp) {
      constexpr int XP = decltype(xp)::value;
      hipLaunchKernelGGL((gemv_polynorm_kernel<R, U, GEMV_AXPY_F32, FAST, XP>), grid, block, lds, st, a, p);
    };
    if (a.K <= 4096) run(std::integral_constant<int, 4>{});
    else run(std::integral_constant<int, 16>{});
  });
}

}  // namespace aha
