// Body of the short decode matvecs: one load group per row (K = 512 * U exactly).  Such a launch is one memory round trip for its weights; what it costs
// is what stands in front of the first request and behind the last return, so everything is known when the kernel is compiled: no divisions, no
// predicates, a hundred instructions in all (the block form of gemv_body.h runs three hundred in front of its first weight, fetched cold).
#pragma once
#include "gemv_body.h"

namespace aha {

// Blocks of a launch: two per CU at most, and whole rounds of tiles.  Three per CU (gemv_kernel's) find the second and third waiting for the first's
// requests anyway and make the vector travel once more each: 2048 + 256 tokens of 0.6B 167.8 ms with 768 blocks, 166.1 with 384 and 512, 169.0 with 1024.
inline int gemv_row_grid(int N, int R) {
  const int ntiles = (N + 4 * R - 1) / (4 * R), rounds = (ntiles + 511) / 512;
  return (ntiles + rounds - 1) / rounds;
}

// The input vector as a prologue leaves it: a lane's share of it is the columns of its own weights, h[u][i] = column 512 u + 8 lane + i.  A prologue is
// a type with request(), its loads, issued ahead of the first weight tile (returns are in order within a wave), and make(h).  With MAPPED it says too where
// the weights are, ptr(row, u) -> this lane's columns of load u (GEMV_SILU_MUL: of the gate row; the up row 16 further), and what a row's sums are
// multiplied by, scale(row) (GEMV_SILU_MUL only).
//
// h = x, or h = bf16(RMSNorm(x) * norm_w): every wave norms the whole row in its registers, no LDS and no barrier; the partial sums in the order of the
// block form (chunks 0, 4, .. | 1, 5, .. | 2, 6, .. | 3, 7, ..), so the bits are the same.
template <int U, bool NORM>
struct RowNormPro {
  const bf16_t* x;
  const bf16_t* w;
  float eps;
  u32x4_t xr[U], nr[U];
  __device__ __forceinline__ void request() {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int u = 0; u < U; ++u) xr[u] = ld16(x + u * 512 + lane * 8);
    if (NORM) {
#pragma unroll
      for (int u = 0; u < U; ++u) nr[u] = ld16(w + u * 512 + lane * 8);
    }
  }
  __device__ __forceinline__ void make(float (&h)[U][8]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) { h[u][2 * j] = lo_bf(xr[u][j]); h[u][2 * j + 1] = hi_bf(xr[u][j]); }
    if (!NORM) return;
    float ss[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 8; ++j) ss[u & 3] += h[u][j] * h[u][j];
#pragma unroll
    for (int i = 0; i < 4 && i < U; ++i) ss[i] = wave_sum(ss[i]);
    const float rinv = 1.0f / sqrtf((ss[0] + ss[1] + ss[2] + ss[3]) / (float)(U * 512) + eps);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        h[u][2 * j] = rbf(h[u][2 * j] * rinv * lo_bf(nr[u][j]));
        h[u][2 * j + 1] = rbf(h[u][2 * j + 1] * rinv * hi_bf(nr[u][j]));
      }
  }
};

// h = bf16(RMSNorm(xn) * norm_w), xn = x + bf16(the sum of P slices of o_proj's f32 sums) (oproj_slices.h); xn is what the layer continues with: block 0
// writes it to x_out, another vector than x, which other blocks still read.  U = 2.  The block reads the slices once, a wave a quarter of the columns, and
// shares xn through LDS: every wave for itself would be 4 P KB more per wave.
template <int P>
struct RowSlicesPro {
  static constexpr int K = 1024;
  const bf16_t *x, *w;
  const float* parts;   // (P, K)
  bf16_t* x_out;
  float eps;
  int bid;
  float* xs;   // LDS, K + 4 floats
  uint2 xr;
  float4 pr[P];
  u32x4_t nr[2];
  __device__ __forceinline__ void request() {
    const int lane = threadIdx.x & 63, k = threadIdx.x * 4;
    xr = *reinterpret_cast<const uint2*>(x + k);
#pragma unroll
    for (int p = 0; p < P; ++p) pr[p] = *reinterpret_cast<const float4*>(parts + p * K + k);
#pragma unroll
    for (int u = 0; u < 2; ++u) nr[u] = ld16(w + u * 512 + lane * 8);
  }
  __device__ __forceinline__ void make(float (&h)[2][8]) {
    const int lane = threadIdx.x & 63, k = threadIdx.x * 4;
    float4 s = pr[0];
#pragma unroll
    for (int p = 1; p < P; ++p) { s.x += pr[p].x; s.y += pr[p].y; s.z += pr[p].z; s.w += pr[p].w; }
    uint2 o;
    o.x = pack_bf(lo_bf(xr.x) + rbf(s.x), hi_bf(xr.x) + rbf(s.y));
    o.y = pack_bf(lo_bf(xr.y) + rbf(s.z), hi_bf(xr.y) + rbf(s.w));
    const float4 v = make_float4(lo_bf(o.x), hi_bf(o.x), lo_bf(o.y), hi_bf(o.y));
    *reinterpret_cast<float4*>(xs + xs_index(k)) = v;
    const float ss = wave_sum((v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w));
    if (lane == 0) xs[K + (threadIdx.x >> 6)] = ss;
    if (bid == 0) *reinterpret_cast<uint2*>(x_out + k) = o;
    __syncthreads();
    const float4 q = *reinterpret_cast<const float4*>(xs + K);
    const float rinv = 1.0f / sqrtf(((q.x + q.y) + (q.z + q.w)) / (float)K + eps);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float4 lo = *reinterpret_cast<const float4*>(xs + xs_index(u * 512 + lane * 8)), hi = *reinterpret_cast<const float4*>(xs + xs_index(u * 512 + lane * 8 + 4));
      const float f[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        h[u][2 * j] = rbf(f[2 * j] * rinv * lo_bf(nr[u][j]));
        h[u][2 * j + 1] = rbf(f[2 * j + 1] * rinv * hi_bf(nr[u][j]));
      }
    }
  }
};

// h = (x - mean) / sqrt(var + eps) * w + b over `width` columns, x in 32 bits, w and b zero behind them; by every wave for itself as well
template <int U>
struct RowLayerNormPro {
  const float* x;
  const bf16_t *w, *b;
  float eps;
  int width;
  float4 s[U][2];
  u32x4_t wr[U], br[U];
  __device__ __forceinline__ void request() {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      s[u][0] = *reinterpret_cast<const float4*>(x + u * 512 + lane * 8);
      s[u][1] = *reinterpret_cast<const float4*>(x + u * 512 + lane * 8 + 4);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) wr[u] = ld16(w + u * 512 + lane * 8);
#pragma unroll
    for (int u = 0; u < U; ++u) br[u] = ld16(b + u * 512 + lane * 8);
  }
  __device__ __forceinline__ void make(float (&h)[U][8]) {
    const int lane = threadIdx.x & 63;
    float sum = 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i) sum += (s[u][i].x + s[u][i].y) + (s[u][i].z + s[u][i].w);   // (pad columns are zero)
    const float mean = wave_sum(sum) / (float)width;
    sum = 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int i = 0; i < 2; ++i) { h[u][4 * i] = s[u][i].x; h[u][4 * i + 1] = s[u][i].y; h[u][4 * i + 2] = s[u][i].z; h[u][4 * i + 3] = s[u][i].w; }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        h[u][i] = u * 512 + lane * 8 + i < width ? h[u][i] - mean : 0.f;
        sum += h[u][i] * h[u][i];
      }
    }
    const float rinv = 1.0f / sqrtf(wave_sum(sum) / (float)width + eps);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        h[u][2 * j] = fmaf(h[u][2 * j] * rinv, lo_bf(wr[u][j]), lo_bf(br[u][j]));
        h[u][2 * j + 1] = fmaf(h[u][2 * j + 1] * rinv, hi_bf(wr[u][j]), hi_bf(br[u][j]));
      }
  }
};

// aux: see GEMV_HOT_PARAMS.  Of `rest` only the outputs (and res_scale) are read, behind the first weights.
template <int R, int U, int EPI, class Pro>
__device__ __forceinline__ void gemv_row_body(const GemvArgs& rest, const void* W, const void* aux, unsigned long long* trace, const int N, const int bid, const int nblk, Pro& pro) {
  constexpr int NW = EPI == GEMV_SILU_MUL ? 2 : 1, KK = U * 512;
  using res_t = typename std::conditional<EPI == GEMV_AXPY_F32, float, bf16_t>::type;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool stamps = trace != nullptr && wave == 0 && (bid == 0 || bid == 255 || bid == nblk - 1);
  auto stamp = [&](int k) {
    if (stamps && lane == 0) trace[(bid == 0 ? 0 : bid == 255 ? 1 : 2) * 6 + k] = wall_clock64();
  };
  stamp(0);
  pro.request();
  u32x4_t bufA[NW][R][U], bufB[NW][R][U];
  res_t resA[R], resB[R];
  auto issue = [&](int tile, u32x4_t (&buf)[NW][R][U], res_t (&resv)[R]) {
    const int row0 = (tile * GEMV_WAVES + wave) * R;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int row = min(row0 + r, N - 1);   // (rows past the end are computed and not stored)
      if (EPI == GEMV_RESIDUAL || EPI == GEMV_AXPY_F32) resv[r] = ((const res_t*)aux)[row];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int row = min(row0 + r, N - 1);
      const bf16_t *p0 = (const bf16_t*)W + (int64_t)row * KK, *p1 = nullptr;
      if (NW == 2) {
        if (aux != nullptr) {   // separate gate / up matrices
          p1 = (const bf16_t*)aux + (int64_t)row * KK;
        } else {                // 16-row blocks alternating gate / up
          p0 = (const bf16_t*)W + (int64_t)((row >> 4) * 32 + (row & 15)) * KK;
          p1 = p0 + 16 * KK;
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if constexpr (gemv_mapped<Pro>::value) {
          const bf16_t* p = pro.ptr(row, u);
          buf[0][r][u] = ld_nt16(p);
          if (NW == 2) buf[NW - 1][r][u] = ld_nt16(p + 16 * KK);
          continue;
        }
        buf[0][r][u] = ld_nt16(p0 + u * 512 + lane * 8);
        if (NW == 2) buf[NW - 1][r][u] = ld_nt16(p1 + u * 512 + lane * 8);
      }
    }
  };
  __builtin_amdgcn_sched_barrier(0);
  issue(bid, bufA, resA);
  __builtin_amdgcn_sched_barrier(0);
  stamp(1);
  float h[U][8];
  pro.make(h);
  stamp(2);
  auto consume = [&](int tile, u32x4_t (&buf)[NW][R][U], res_t (&resv)[R]) {
    float acc[NW][R];
#pragma unroll
    for (int m = 0; m < NW; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r) acc[m][r] = 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < NW; ++m) {
          float s = acc[m][r];   // (the activation first: gemv_body.h)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            s = fmaf(h[u][2 * j], lo_bf(buf[m][r][u][j]), s);
            s = fmaf(h[u][2 * j + 1], hi_bf(buf[m][r][u][j]), s);
          }
          acc[m][r] = s;
        }
#pragma unroll
    for (int m = 0; m < NW; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r) acc[m][r] = wave_sum(acc[m][r]);
    if constexpr (gemv_mapped<Pro>::value && EPI == GEMV_SILU_MUL) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float s = pro.scale(min((tile * GEMV_WAVES + wave) * R + r, N - 1));
#pragma unroll
        for (int m = 0; m < NW; ++m) acc[m][r] *= s;
      }
    }
    if (lane == 0) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int row = (tile * GEMV_WAVES + wave) * R + r;
        if (row >= N) continue;
        const float lin = rbf(acc[0][r]);
        if constexpr (EPI == GEMV_AXPY_F32) rest.y_f32[row] = fmaf(rest.res_scale, resv[r], acc[0][r]);
        else if constexpr (EPI == GEMV_PARTIAL_F32) rest.y_f32[row] = acc[0][r];
        else if constexpr (EPI == GEMV_STORE) ((bf16_t*)rest.y)[row] = f2bf(lin);
        else if constexpr (EPI == GEMV_RESIDUAL) ((bf16_t*)rest.y)[row] = f2bf(bf2f(resv[r]) + lin);
        else ((bf16_t*)rest.y)[row] = f2bf(rbf(silu_f(lin)) * rbf(acc[NW - 1][r]));
      }
    }
  };
  const int ntiles = (N + GEMV_WAVES * R - 1) / (GEMV_WAVES * R);
  int t = bid;
  for (; t + 2 * nblk < ntiles; t += 2 * nblk) {   // (both refills unconditional, as gemv_body's FAST form)
    __builtin_amdgcn_sched_barrier(0);
    issue(t + nblk, bufB, resB);
    __builtin_amdgcn_sched_barrier(0);
    consume(t, bufA, resA);
    __builtin_amdgcn_sched_barrier(0);
    issue(t + 2 * nblk, bufA, resA);
    __builtin_amdgcn_sched_barrier(0);
    consume(t + nblk, bufB, resB);
  }
  if (t + nblk < ntiles) {
    __builtin_amdgcn_sched_barrier(0);
    issue(t + nblk, bufB, resB);
    __builtin_amdgcn_sched_barrier(0);
    consume(t, bufA, resA);
    consume(t + nblk, bufB, resB);
  } else {
    consume(t, bufA, resA);
  }
  stamp(4);
}

}  // namespace aha
