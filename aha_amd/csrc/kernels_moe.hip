// Routed experts of the layer-list decoders: scores s = sigmoid(router logits), the `top` largest per token; a chosen expert computes
//   down (silu(s gate h) * (s up h))      (the score multiplies the expert's input; gate and up are linear, so it is applied to their outputs)
//   moe_topk_kernel     scores, the largest, tokens per expert
//   moe_slots_kernel    slots: an expert's (token, choice) pairs one after the other; tiles of `bm` slots of one expert
//   moe_gemm_kernel     bf16, 128 x 128 tiles (many tokens per expert), rows gathered by slot
//   moe_gemm256_kernel  bf16, 256 x 256 tiles (kernels_moe256.hip)
//   moe_gemm_few_kernel  bf16, up to 32 slots x 16 or 48 weight rows, whole K (few tokens per expert)
//   moe_gemm_f32_kernel   the 32-bit mode
#include <math.h>

#include <algorithm>

#include <type_traits>

#include "attn_common.h"
#include "kernels_prenorm.h"
#include "rows_common.h"
#include "skinny_body.h"

namespace aha {

namespace {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* glb_ptr_t;
constexpr int MAX_EXPERTS = 1024;
constexpr float LOG2E = 1.4426950408889634f;

// One wave per row, `per` rows per wave.  Ordering by the logits (the sigmoid is monotonic), ties to the lower index.
template <int NJ>   // experts <= NJ * 64
__global__ __launch_bounds__(256) void moe_topk_kernel(const float* __restrict__ z, int64_t ldz, int rows, int experts, int top, int per, MoeRouting r) {
  __shared__ int hist[NJ * 64];
  for (int i = threadIdx.x; i < experts; i += 256) hist[i] = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63, row0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * per;
  for (int row = row0; row < min(row0 + per, rows); ++row) {
    const float* zr = z + (int64_t)row * ldz;
    float v[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) v[j] = j * 64 + lane < experts ? zr[j * 64 + lane] : -INFINITY;
    for (int k = 0; k < top; ++k) {
      float best = -INFINITY;
      int bi = 1 << 30;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
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
      for (int j = 0; j < NJ; ++j)
        if (j * 64 + lane == bi) v[j] = -INFINITY;
      if (lane == 0) {
        r.sel[row * top + k] = bi;
        r.sel_w[row * top + k] = 1.0f / (1.0f + expf(-m));
        atomicAdd(&hist[bi], 1);
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < experts; i += 256)
    if (hist[i]) atomicAdd(r.counts + i, hist[i]);
}

// Every block scans the counts, reserves runs of its pairs' slots and fills them in; block 0 lists the tiles.  (The order of an expert's slots
// depends on the blocks' order; no result does.)
__global__ __launch_bounds__(1024) void moe_slots_kernel(int rows, int experts, int top, int bm, MoeRouting r) {
  __shared__ int cnt[MAX_EXPERTS], start[MAX_EXPERTS], base[MAX_EXPERTS], wsum[2][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int total = tid < experts ? r.counts[tid] : 0;
  const int mine = tid < experts ? (total + bm - 1) / bm : 0;
  int s = total, t = mine;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int x = __shfl_up(s, o, 64), y = __shfl_up(t, o, 64);
    if (lane >= o) {
      s += x;
      t += y;
    }
  }
  if (lane == 63) {
    wsum[0][wave] = s;
    wsum[1][wave] = t;
  }
  cnt[tid] = 0;
  __syncthreads();
  for (int w = 0; w < wave; ++w) {
    s += wsum[0][w];
    t += wsum[1][w];
  }
  start[tid] = s - total;
  if (blockIdx.x == 0 && tid < experts) {
    for (int i = 0; i < mine; ++i) {
      int32_t* o = r.tiles + (int64_t)(t - mine + i) * 3;
      o[0] = tid;
      o[1] = s - total + i * bm;
      o[2] = min(bm, total - i * bm);
    }
    if (tid == experts - 1) *r.n_tiles = t;
  }
  __syncthreads();
  const int i = blockIdx.x * 1024 + tid, n = rows * top;
  int e = 0, at = 0;
  if (i < n) {
    e = r.sel[i];
    at = atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  if (tid < experts && cnt[tid]) base[tid] = atomicAdd(r.cursor + tid, cnt[tid]);
  __syncthreads();
  if (i < n) {
    const int slot = start[e] + base[e] + at;
    r.slot_of[i] = slot;
    r.slot_row[slot] = i / top;
    r.slot_w[slot] = r.sel_w[i];
  }
}

__device__ __forceinline__ float silu_fast(float x) { return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-LOG2E * x)); }

// ---- 128 x 128 x 64 tiles, four waves of 64 x 64 (staging and swizzle: kernels_gemm.hip gemm_glds_kernel), two LDS stages ----------------------
constexpr int TM = 128, TN = 128, TK = 64, OPB = 128 * TK * 2;
__device__ __forceinline__ int tswz(int row, int slot) { return row * 128 + ((slot ^ ((row >> 1) & 7)) << 4); }

template <bool GATHER, bool PAIRS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void moe_gemm_kernel(MoeGemmArgs a, MoeRouting r, int ntn, int parts) {   // parts: 128-row pieces of a listed tile
  extern __shared__ __attribute__((aligned(16))) char smem[];   // 2 x [A | W]
  const int nt = *r.n_tiles * parts;
  // an XCD's blocks take consecutive tiles: the column tiles of one expert's slots share its rows, the slot tiles its weights
  const int per_t = (nt * ntn + 7) >> 3, idx = ((int)blockIdx.x & 7) * per_t + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= per_t || idx >= nt * ntn) return;
  const int mt = idx / ntn, n0 = (idx - mt * ntn) * TN;
  const int32_t* tl = r.tiles + mt / parts * 3;
  const int part = mt % parts, ex = tl[0], s0 = tl[1] + part * TM, ns = min(TM, tl[2] - part * TM);
  if (ns <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, G = lane >> 4, c = lane & 15, wm = wave >> 1, wn = wave & 1;
  const bf16_t* W = (const bf16_t*)a.W + (int64_t)ex * a.n * a.k;
  const bf16_t *ga[4], *gw[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = (j * 4 + wave) * 8 + (lane >> 3), s = (lane & 7) ^ ((row >> 1) & 7);
    const int slot = s0 + min(row, ns - 1);
    ga[j] = (const bf16_t*)a.A + (int64_t)(GATHER ? r.slot_row[slot] : slot) * a.lda + s * 8;
    gw[j] = W + (int64_t)min(n0 + row, a.n - 1) * a.k + s * 8;
  }
  f32x4_t acc[4][4];   // [ni][mi]
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int nk = a.k / TK;
  auto stage = [&](int kt) {
    char* sa = smem + (kt & 1) * (2 * OPB);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(ga[j] + kt * TK), (lds_ptr_t)(sa + (j * 4 + wave) * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(gw[j] + kt * TK), (lds_ptr_t)(sa + OPB + (j * 4 + wave) * 1024), 16, 0, 0);
    }
  };
  stage(0);
  for (int kt = 0; kt < nk; ++kt) {
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    if (kt + 1 < nk) stage(kt + 1);
    const char *sa = smem + (kt & 1) * (2 * OPB), *sw = sa + OPB;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8_t af[4], wf[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        af[i] = as_frag(*reinterpret_cast<const u32x4_t*>(sa + tswz(wm * 64 + i * 16 + c, ks * 4 + G)));
        wf[i] = as_frag(*reinterpret_cast<const u32x4_t*>(sw + tswz(wn * 64 + i * 16 + c, ks * 4 + G)));
      }
#pragma unroll
      for (int ni = 0; ni < 4; ++ni)
#pragma unroll
        for (int mi = 0; mi < 4; ++mi) acc[ni][mi] = mfma16(wf[ni], af[mi], acc[ni][mi]);
    }
  }
#pragma unroll
  for (int mi = 0; mi < 4; ++mi) {
    const int row = wm * 64 + mi * 16 + c;
    if (row >= ns) continue;
    bf16_t* o = (bf16_t*)a.C + (int64_t)(s0 + row) * a.ldc;
    if constexpr (PAIRS) {
      const float w = r.slot_w[s0 + row];
#pragma unroll
      for (int ni = 0; ni < 4; ni += 2) {
        const int n = n0 + wn * 64 + ni * 16;
        if (n >= a.n) continue;
        float f[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) f[q] = silu_fast(w * acc[ni][mi][q]) * (w * acc[ni + 1][mi][q]);
        *reinterpret_cast<uint2*>(o + n / 2 + G * 4) = make_uint2(pack_bf(f[0], f[1]), pack_bf(f[2], f[3]));
      }
    } else {
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) {
        const int n = n0 + wn * 64 + ni * 16;
        if (n < a.n) *reinterpret_cast<uint2*>(o + n + G * 4) = make_uint2(pack_bf(acc[ni][mi][0], acc[ni][mi][1]), pack_bf(acc[ni][mi][2], acc[ni][mi][3]));
      }
    }
  }
}

// ---- few slots per expert: up to 32 of them against R8 * 8 weight rows, whole K (skinny_body.h) ---------------------------------------------------
// Bound by the chosen experts' weights.  Tiles of 32 slots, so that an expert with 17 to 32 of them still reads its weights once; the ring has the
// activation rows a tile needs (8, 16 or 32).  MI355X, 32 tokens x 2 of 32 experts at the 8B sizes: gate + up (1.4 GB) 348 -> 212 us, down
// (0.7 GB) 160 -> 107 us (6.6 TB/s) against 16 x 64 tiles that loaded fragments to registers (16 rows x 64 bytes per request).
constexpr int MOE_FEW = 32;

template <int R8, int M8, bool GATHER, bool PAIRS>
__device__ __forceinline__ void moe_few_body(const MoeGemmArgs& a, const MoeRouting& r, int n_blk, int ex, int s0, int ns, char* smem) {
  constexpr int MT = (M8 + 1) / 2;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), G = lane >> 4, c = lane & 15;
  const char* W = (const char*)((const bf16_t*)a.W + (int64_t)ex * a.n * a.k);
  const char* src[R8 + M8];
#pragma unroll
  for (int q = 0; q < R8 + M8; ++q) {
    const int local = (q < R8 ? q : q - R8) * 8 + (lane >> 3), piece = skinny_piece(local, lane);
    if (q >= R8) {
      const int slot = s0 + min(local, ns - 1);
      src[q] = (const char*)a.A + (int64_t)(GATHER ? r.slot_row[slot] : slot) * a.lda * 2 + piece;
    } else if (PAIRS) {   // eight gate rows, then the eight up rows of the same columns
      const int col = (n_blk * (R8 / 2) + q / 2) * 8 + (lane >> 3);
      src[q] = W + (int64_t)min((col >> 4) * 32 + (q & 1) * 16 + (col & 15), a.n - 1) * a.k * 2 + piece;
    } else {
      src[q] = W + (int64_t)min(n_blk * (R8 * 8) + local, a.n - 1) * a.k * 2 + piece;
    }
  }
  skinny_sums<R8, M8>(src, a.k / 64, skinny_first(n_blk * (R8 * 8), a.k / 64), smem, wave, lane);
  for (int i = wave; i < (R8 / 2) * MT; i += SKINNY_WAVES) {
    const int f = i / MT, row = (i - f * MT) * 16 + c;
    if (row >= ns) continue;
    bf16_t* o = (bf16_t*)a.C + (int64_t)(s0 + row) * a.ldc;
    if constexpr (PAIRS) {
      const int col = (n_blk * (R8 / 2) + f) * 8 + G * 4;
      if (G >= 2 || col >= a.n / 2) continue;
      const float w = r.slot_w[s0 + row];
      const f32x4_t g = skinny_total<R8, M8>(smem, i, lane), u = skinny_total<R8, M8>(smem, i, lane + 32);
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = silu_fast(w * g[q]) * (w * u[q]);
      *reinterpret_cast<uint2*>(o + col) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
    } else {
      const int n = n_blk * (R8 * 8) + f * 16 + G * 4;
      if (n >= a.n) continue;
      const f32x4_t v = skinny_total<R8, M8>(smem, i, lane);
      *reinterpret_cast<uint2*>(o + n) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
    }
  }
}

template <int R8, bool GATHER, bool PAIRS>
__global__ __launch_bounds__(SKINNY_WAVES * 64) void moe_gemm_few_kernel(MoeGemmArgs a, MoeRouting r, int ntn) {
  static_assert(R8 % 2 == 0, "whole fragments");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int mt = blockIdx.x / ntn, n_blk = (int)blockIdx.x - mt * ntn;
  if (mt >= *r.n_tiles) return;
  const int ex = r.tiles[mt * 3], s0 = r.tiles[mt * 3 + 1], ns = r.tiles[mt * 3 + 2];
  if (ns <= 8) moe_few_body<R8, 1, GATHER, PAIRS>(a, r, n_blk, ex, s0, ns, smem);
  else if (ns <= 16) moe_few_body<R8, 2, GATHER, PAIRS>(a, r, n_blk, ex, s0, ns, smem);
  else moe_few_body<R8, 4, GATHER, PAIRS>(a, r, n_blk, ex, s0, ns, smem);
}

// ---- 32-bit mode: 64 x 64 tiles on v_mfma_f32_16x16x4_f32 (kernels_gemm_f32.hip gemm_f32_any_kernel with gathered rows) --------------------------------
constexpr int FBK = 32, FPITCH = FBK + 1;
template <bool GATHER>
__global__ __launch_bounds__(256) void moe_gemm_f32_kernel(MoeGemmArgs a, MoeRouting r) {
  __shared__ float as[64 * FPITCH], ws[64 * FPITCH];
  if ((int)blockIdx.y >= *r.n_tiles) return;
  const int ex = r.tiles[blockIdx.y * 3], s0 = r.tiles[blockIdx.y * 3 + 1], ns = r.tiles[blockIdx.y * 3 + 2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, G = lane >> 4, n0 = blockIdx.x * 64;
  const bf16_t* W = (const bf16_t*)a.W + (int64_t)ex * a.n * a.k;
  f32x4_t acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < a.k; k0 += FBK) {
#pragma unroll
    for (int i = 0; i < 64 * FBK / 4 / 256; ++i) {
      const int p = tid + i * 256, row = p >> 3, kk = (p & 7) * 4;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f), w = v;
      if (row < ns) v = *reinterpret_cast<const float4*>((const float*)a.A + (int64_t)(GATHER ? r.slot_row[s0 + row] : s0 + row) * a.lda + k0 + kk);
      if (n0 + row < a.n) w = wbf4(W, (int64_t)(n0 + row) * a.k + k0 + kk);
      float *da = as + row * FPITCH + kk, *dw = ws + row * FPITCH + kk;
      da[0] = v.x; da[1] = v.y; da[2] = v.z; da[3] = v.w;
      dw[0] = w.x; dw[1] = w.y; dw[2] = w.z; dw[3] = w.w;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < FBK; k += 4) {
      const float av = as[(wave * 16 + c) * FPITCH + k + G];
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, ws[(j * 16 + c) * FPITCH + k + G], acc[j], 0, 0, 0);
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + j * 16 + c;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int m = wave * 16 + G * 4 + q;
      if (m < ns && n < a.n) ((float*)a.C)[(int64_t)(s0 + m) * a.ldc + n] = acc[j][q];
    }
  }
}

}  // namespace

int moe_max_tiles(int rows, int top, int experts, int bm) { return (rows * top + bm - 1) / bm + std::min(experts, rows * top); }

int moe_tile_rows(int slots, int experts, bool f32) { return f32 ? 64 : slots <= 24 * experts ? MOE_FEW : slots >= 96 * experts ? 2 * TM : TM; }

void launch_moe_route(const float* z, int64_t ldz, int rows, int experts, int top, int bm, const MoeRouting& r, hipStream_t st) {
  if (rows <= 0) return;
  const int per = rows >= 4096 ? 4 : 1;
  auto topk = [&](auto k) { hipLaunchKernelGGL(k, dim3((unsigned)((rows + 4 * per - 1) / (4 * per))), dim3(256), 0, st, z, ldz, rows, experts, top, per, r); };
  if (experts <= 64) topk(moe_topk_kernel<1>);
  else if (experts <= 256) topk(moe_topk_kernel<4>);
  else topk(moe_topk_kernel<16>);
  hipLaunchKernelGGL(moe_slots_kernel, dim3((unsigned)((rows * top + 1023) / 1024)), dim3(1024), 0, st, rows, experts, top, bm, r);
}

void launch_moe_gemm(const MoeGemmArgs& a, const MoeRouting& r, int bm, bool f32, hipStream_t st) {
  if (a.slots <= 0) return;
  const int mt = (a.slots + bm - 1) / bm + std::min(a.experts, a.slots);
  if (f32) {
    const dim3 grid((unsigned)((a.n + 63) / 64), (unsigned)mt);
    if (a.gather) hipLaunchKernelGGL(moe_gemm_f32_kernel<true>, grid, dim3(256), 0, st, a, r);
    else hipLaunchKernelGGL(moe_gemm_f32_kernel<false>, grid, dim3(256), 0, st, a, r);
    return;
  }
  // 256-row tiles where they fill the chip, the k loop is long enough for one block per CU, and a gathered row's offset fits the loads' 1 GiB
  if (bm == 2 * TM && a.k >= 512 && (int64_t)a.slots * a.lda < (1 << 28) && (int64_t)(a.slots / bm) * ((a.n + 255) / 256) >= 192) {
    launch_moe_gemm256(a, r, mt, st);
    return;
  }
  auto go = [&](auto ga, auto pa) {
    constexpr bool GA = decltype(ga)::value, PA = decltype(pa)::value;
    if (bm == MOE_FEW) {
      // 48 weight rows per block; 16 where the tiles (at most one per expert while slots are few) would leave CUs without a block
      auto few = [&](auto r8) {
        constexpr int R8 = decltype(r8)::value, lds = std::max({skinny_lds(R8, 1), skinny_lds(R8, 2), skinny_lds(R8, 4)});
        const int ntn = (a.n + R8 * 8 - 1) / (R8 * 8);
        if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(moe_gemm_few_kernel<R8, GA, PA>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        hipLaunchKernelGGL((moe_gemm_few_kernel<R8, GA, PA>), dim3((unsigned)(mt * ntn)), dim3(SKINNY_WAVES * 64), lds, st, a, r, ntn);
      };
      if (std::min(a.experts, a.slots) * ((a.n + 47) / 48) >= 512) few(std::integral_constant<int, 6>{});
      else few(std::integral_constant<int, 2>{});
    } else {
      const int ntn = (a.n + TN - 1) / TN, parts = bm / TM;
      const unsigned nb = (unsigned)((mt * parts * ntn + 7) / 8 * 8);
      hipLaunchKernelGGL((moe_gemm_kernel<GA, PA>), dim3(nb), dim3(256), 4 * OPB, st, a, r, ntn, parts);
    }
  };
  if (a.gather) {
    if (a.pairs) go(std::true_type{}, std::true_type{});
    else go(std::true_type{}, std::false_type{});
  } else {
    if (a.pairs) go(std::false_type{}, std::true_type{});
    else go(std::false_type{}, std::false_type{});
  }
}

}  // namespace aha
