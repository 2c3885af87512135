// Latent attention of the layer-list decoders: a token's cache row is one latent c and one rotated key part shared by all heads; head h's key
// is [W_uk_h c | key part], its value W_uv_h c; position i sees the last `window` positions up to itself.
//   latent_post_kernel      rotation of the queries, norm of the latent, rotation of the key part, append
//   prompts, bf16:          keys and values of the visible positions expanded by a GEMM, latent_prefill_kernel on them
//   one token each, bf16:   latent_query_kernel takes the queries into the latent space (W_uk_h^T q_h) and appends the token's cache row,
//                           latent_decode_kernel reads every cached row once per 16 heads, latent_merge_kernel joins the splits and applies W_uv
//   any sizes, 32-bit mode: latent_rows_kernel, also in the latent space
// Scores, maxima, exponentials and sums are f32; P feeds the matrix cores as bf16.
#include <math.h>

#include <algorithm>

#include <type_traits>

#include "attn_common.h"
#include "kernels_prenorm.h"
#include "rows_common.h"

namespace aha {

namespace {

typedef short __attribute__((ext_vector_type(4))) tr4_t;
typedef __attribute__((address_space(3))) tr4_t* lds_tr_t;
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* glb_ptr_t;
constexpr float LOG2E = 1.4426950408889634f;

// cached row of position `pos`
template <typename T>
__device__ __forceinline__ T* cache_row(const LatentCache& c, const LatentDims& d, int slot, int pos) {
  return reinterpret_cast<T*>(c.tab[(int64_t)slot * c.ld + pos / KV_PAGE_TOKENS] + c.off) + (int64_t)(pos % KV_PAGE_TOKENS) * d.ldc();
}

// the token's cache row: latent normed, key part rotated (256 threads; red: 4 floats, not reused before the next barrier).  All that a row of up to 1024 and
// 256 columns takes is requested before its sum.
template <typename TI, typename T>
__device__ __forceinline__ void append_row(const LatentPostArgs& a, const SeqEntry& e, int r, int pos, const float2* cs, float* red) {
  constexpr int NV = 4;
  const int tid = threadIdx.x, half = a.d.rot >> 1;
  const TI* kv = (const TI*)a.in + (int64_t)r * a.ld + a.kv_off;
  const bf16_t* nw = (const bf16_t*)a.norm_w;
  float v[NV], w[NV], u0 = 0.f, u1 = 0.f;
  float2 t0 = make_float2(0.f, 0.f);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    v[j] = w[j] = 0.f;
    if (j * 256 < a.d.rank) {
      const int i = min(tid + j * 256, a.d.rank - 1);
      v[j] = Act<TI>::ld(kv + i);
      w[j] = bf2f(nw[i]);
    }
  }
  auto key_part = [&](int i, float& x0, float& x1, float2& t) {
    const int k = i < half ? i : i - half;
    x0 = Act<TI>::ld(kv + a.d.rp + k);
    x1 = Act<TI>::ld(kv + a.d.rp + k + half);
    t = cs[k];
  };
  if (tid < a.d.rot) key_part(tid, u0, u1, t0);
  T* out = cache_row<T>(a.c, a.d, e.slot, pos);
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j)
    if (tid + j * 256 < a.d.rank) s = fmaf(v[j], v[j], s);
  for (int i = tid + NV * 256; i < a.d.rank; i += 256) {
    const float x = Act<TI>::ld(kv + i);
    s = fmaf(x, x, s);
  }
  const float rinv = 1.0f / sqrtf(block_sum_n<256>(s, red) / (float)a.d.rank + a.eps);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = tid + j * 256;
    if (i < a.d.rp) Act<T>::st(out + i, i < a.d.rank ? v[j] * rinv * w[j] : 0.f);
  }
  for (int i = tid + NV * 256; i < a.d.rp; i += 256) Act<T>::st(out + i, i < a.d.rank ? Act<TI>::ld(kv + i) * rinv * bf2f(nw[i]) : 0.f);
  for (int i = tid; i < a.d.tp; i += 256) {
    if (i >= 256 && i < a.d.rot) key_part(i, u0, u1, t0);
    Act<T>::st(out + a.d.rp + i, i >= a.d.rot ? 0.f : i < half ? u0 * t0.x - u1 * t0.y : u1 * t0.x + u0 * t0.y);
  }
}

template <typename TI, typename T>
__global__ __launch_bounds__(256) void latent_post_kernel(LatentPostArgs a, SeqBatch b) {
  __shared__ float red[4];
  const int r = blockIdx.x, tid = threadIdx.x, half = a.d.rot >> 1, qd = a.d.qd();
  const SeqEntry e = seq_entry_at(b, entry_of_row(b, r));
  const int pos = e.pos0 + r - e.row0;
  const TI* in = (const TI*)a.in + (int64_t)r * a.ld;
  T* q = (T*)a.q + (int64_t)r * a.ldq;
  const float2* cs = reinterpret_cast<const float2*>(a.rope) + (int64_t)r * half;
  for (int i = tid; i < a.d.heads * half; i += 256) {
    const int h = i / half, k = i - h * half, j = h * qd + a.d.dp + k;
    const float u = Act<TI>::ld(in + j), v = Act<TI>::ld(in + j + half);
    const float2 t = cs[k];
    Act<T>::st(q + j, u * t.x - v * t.y);
    Act<T>::st(q + j + half, v * t.x + u * t.y);
  }
  if (a.kv_off >= 0) append_row<TI, T>(a, e, r, pos, cs, red);
}

// One token per sequence: blocks (64 latent dims, head, 16 sequences) as heads_gemm_kernel, a head's blocks rotate its queries between them; the blocks
// behind the last head append the cache rows, one each.  A chain of waits at these sizes: the rotation's inputs are requested in front of the product, and
// what the first requests take is in the leading arguments (0.6B widths, one sequence: 4.1 -> 3.9 us; 8B,
// 32 sequences: 7.0 -> 5.0).
template <typename TI>
__global__ __launch_bounds__(256) void latent_query_kernel(const TI* in, const bf16_t* w_ukt, const float2* rope, int ld, int heads, int rp, int dp, int tp, int rot, int rows, LatentQueryArgs a, SeqBatch b) {
  __shared__ float red[4];
  const int tid = threadIdx.x, h = blockIdx.y, m0 = blockIdx.z * 16, half = rot >> 1, nx = rp >> 6;
  if (h >= heads) {
    const int r = m0 + (h - heads) * nx + blockIdx.x;
    if (r >= min(m0 + 16, rows)) return;
    const SeqEntry e = seq_entry_at(b, r);
    append_row<TI, bf16_t>(a.p, e, r, e.pos0, rope + (int64_t)r * half, red);
    return;
  }
  in += (int64_t)h * (dp + tp);
  const int lane = tid & 63, wave = tid >> 6, G = lane >> 4, c = lane & 15, n0 = blockIdx.x * 64 + wave * 16;
  const bf16_t* w = w_ukt + ((int64_t)h * rp + n0 + c) * dp + G * 8;
  const TI* x = in + (int64_t)min(m0 + c, rows - 1) * ld + G * 8;
  float u = 0.f, v = 0.f;
  float2 t = make_float2(0.f, 0.f);
  auto request = [&](int i) {
    const int rr = (unsigned)i / (unsigned)tp, j = i - rr * tp, r = m0 + rr;
    if (j < rot) {
      const int k = j < half ? j : j - half;
      const TI* q = in + (int64_t)r * ld + dp;
      u = Act<TI>::ld(q + k);
      v = Act<TI>::ld(q + k + half);
      t = rope[(int64_t)r * half + k];
    }
  };
  const int turns = min(16, rows - m0) * tp;
  int i = blockIdx.x * 256 + tid;
  if (i < turns) request(i);
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < dp; k += 32) {
    const float4 lo = Act<TI>::ld4(x + k), hi = Act<TI>::ld4(x + k + 4);
    acc = mfma16(as_frag(ld16(w + k)), as_frag(u32x4_t{pack_bf(lo.x, lo.y), pack_bf(lo.z, lo.w), pack_bf(hi.x, hi.y), pack_bf(hi.z, hi.w)}), acc);
  }
  if (m0 + c < rows) *reinterpret_cast<uint2*>((bf16_t*)a.qa + ((int64_t)(m0 + c) * heads + h) * rp + n0 + G * 4) = make_uint2(pack_bf(acc[0], acc[1]), pack_bf(acc[2], acc[3]));
  for (; i < turns; i += nx * 256) {
    if (i >= nx * 256) request(i);
    const int rr = (unsigned)i / (unsigned)tp, j = i - rr * tp;
    ((bf16_t*)a.qr)[((int64_t)(m0 + rr) * heads + h) * tp + j] = f2bf(j >= rot ? 0.f : j < half ? u * t.x - v * t.y : v * t.x + u * t.y);
  }
}

// ---- every head's own product: four waves of 16 output columns, MT x 16 rows -------------------------------------------------------------
template <int MT>
__global__ __launch_bounds__(256) void heads_gemm_kernel(HeadsGemmArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, G = lane >> 4, c = lane & 15, h = blockIdx.y;
  const int n0 = blockIdx.x * 64 + wave * 16, m0 = blockIdx.z * (MT * 16);
  if (n0 >= a.n) return;
  const bf16_t* w = (const bf16_t*)a.W + ((int64_t)h * a.n + n0 + c) * a.k + G * 8;
  const bf16_t* x[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) x[i] = (const bf16_t*)a.A + (int64_t)min(m0 + i * 16 + c, a.rows - 1) * a.lda + h * a.sa + G * 8;
  f32x4_t acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < a.k; k += 32) {
    const bf16x8_t wf = as_frag(ld16(w + k));
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = mfma16(wf, as_frag(ld16(x[i] + k)), acc[i]);
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int r = m0 + i * 16 + c;
    if (r < a.rows)
      *reinterpret_cast<uint2*>((bf16_t*)a.C + (int64_t)r * a.ldc + h * a.sc + n0 + G * 4) = make_uint2(pack_bf(acc[i][0], acc[i][1]), pack_bf(acc[i][2], acc[i][3]));
  }
}

// ---- any sizes: one wave per (row, head), 64 positions at a time, lane = position for the scores, lanes = latent dims for the sum ------------
constexpr int ROWS_MAX_RANK = 1024;
template <typename T>
__global__ __launch_bounds__(64) void latent_rows_kernel(LatentRowsArgs a, SeqBatch b) {
  extern __shared__ __attribute__((aligned(16))) float sh[];   // query (rp + tp), then 64 probabilities
  const int r = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, rp = a.d.rp, tp = a.d.tp;
  const SeqEntry e = seq_entry_at(b, entry_of_row(b, r));
  const int pos = e.pos0 + r - e.row0, lo = a.d.first(pos);
  float* ps = sh + rp + tp;
  const T *qa = (const T*)a.qa + ((int64_t)r * a.d.heads + h) * rp, *qr = (const T*)a.q + (int64_t)r * a.ldq + h * a.d.qd() + a.d.dp;
  for (int i = lane; i < rp; i += 64) sh[i] = Act<T>::ld(qa + i);
  for (int i = lane; i < tp; i += 64) sh[rp + i] = i < a.d.rot ? Act<T>::ld(qr + i) : 0.f;
  __syncthreads();
  float m = -INFINITY, l = 0.f, o[ROWS_MAX_RANK / 64];
#pragma unroll
  for (int i = 0; i < ROWS_MAX_RANK / 64; ++i) o[i] = 0.f;
  for (int pg = lo / KV_PAGE_TOKENS; pg <= pos / KV_PAGE_TOKENS; ++pg) {
    const T* base = cache_row<T>(a.c, a.d, e.slot, pg * KV_PAGE_TOKENS);
    const int t = pg * KV_PAGE_TOKENS + lane;
    float s = -INFINITY;
    if (t >= lo && t <= pos) {
      const T* row = base + (int64_t)lane * a.d.ldc();
      float dot = 0.f;
      for (int i = 0; i < rp + tp; i += 4) {
        const float4 k = Act<T>::ld4(row + i), q = *reinterpret_cast<const float4*>(sh + i);
        dot = fmaf(q.x, k.x, fmaf(q.y, k.y, fmaf(q.z, k.z, fmaf(q.w, k.w, dot))));
      }
      s = dot * a.d.scale;
    }
    const float m_new = fmaxf(m, wave_max(s));   // (a visited page holds at least one visible position)
    const float al = expf(m - m_new), p = expf(s - m_new);
    l = l * al + wave_sum(p);
    m = m_new;
    ps[lane] = p;
    __syncthreads();
    const int k0 = max(0, lo - pg * KV_PAGE_TOKENS), k1 = min(KV_PAGE_TOKENS - 1, pos - pg * KV_PAGE_TOKENS);
#pragma unroll
    for (int i = 0; i < ROWS_MAX_RANK / 64; ++i) {
      if (i * 64 >= rp) break;   // (rp is a multiple of 64)
      float acc = o[i] * al;
      for (int k = k0; k <= k1; ++k) acc = fmaf(ps[k], Act<T>::ld(base + (int64_t)k * a.d.ldc() + i * 64 + lane), acc);
      o[i] = acc;
    }
    __syncthreads();
  }
  const float inv = 1.0f / l;
  T* op = (T*)a.o + ((int64_t)r * a.d.heads + h) * rp;
#pragma unroll
  for (int i = 0; i < ROWS_MAX_RANK / 64; ++i)
    if (i * 64 < rp) Act<T>::st(op + i * 64 + lane, o[i] * inv);
}

// ---- prompts ------------------------------------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void latent_gather_kernel(LatentDims d, LatentCache c, const int32_t* ext0, T* out, SeqBatch b) {
  const SeqEntry e = seq_entry_at(b, blockIdx.y);
  constexpr int EP = 16 / sizeof(T);
  const int lo = d.first(e.pos0) & ~(KV_PAGE_TOKENS - 1), n = e.pos0 + e.len - lo, np = (int)(d.ldc() / EP);
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int r = (int)(i / np), p = (int)(i - (int64_t)r * np);
  if (r >= n) return;
  const int pos = lo + r;
  const uint64_t src = (uint64_t)cache_row<T>(c, d, e.slot, pos) + p * 16;
  *reinterpret_cast<u32x4_t*>(out + ((int64_t)ext0[blockIdx.y] + r) * d.ldc() + p * EP) = ld16_global(src);
}

// NWV waves x 16 query rows of one head; tiles of 64 positions, K and V staged by LDS-DMA (two stages) as 1-KB fragment blocks -- 16 positions x
// 32 dims, 16-byte piece l = position l & 15, dims (l >> 4) * 8 .. -- gathered from token-major rows by per-lane source addresses: unrotated key
// dims and values from the expanded rows, the rotated part from the cache rows.  V^T fragments are transposed reads (ds_read_b64_tr_b16).
// S^T = K . Q^T, so that the probabilities are the next product's operand in place.
template <int DQK, int DV, int NWV>
__global__ __launch_bounds__(NWV * 64) __attribute__((amdgpu_waves_per_eu(DV > 128 || DQK + DV > 320 ? 2 : NWV == 4 && (DV == 128 || DQK == 256) ? 3 : 4, 4))) void latent_prefill_kernel(LatentPrefillArgs a, SeqBatch b, int nqb) {
  constexpr int KS = DQK / 32, VS = DV / 32, DS = DV / 16, KB = KS * 4, VB = VS * 4, STAGE = (KB + VB) * 1024;
  constexpr int RING = DV >= 128 ? 3 : DQK >= 128 ? 6 : 4, KRING = RING < KB ? RING : KB, VRING = DQK + DV >= 320 ? 2 : DV >= 128 ? 3 : 4 < 2 * DS ? 4 : 2 * DS;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), G = lane >> 4, c = lane & 15;
  int head, qblk;
  {   // heads dealt to the XCDs, an XCD's blocks in order of (head, query block): its L2 holds the keys and values they share
    const int id = blockIdx.x, nh = a.d.heads;
    if (nh % 8 == 0) {
      const int slot = id >> 3;
      head = (id & 7) * (nh >> 3) + slot / nqb;
      qblk = nqb - 1 - slot % nqb;
    } else {
      head = id / nqb;
      qblk = nqb - 1 - id % nqb;
    }
  }
  const SeqEntry e = seq_entry_at(b, blockIdx.y);
  const int qb = qblk * (16 * NWV), q0 = qb + wave * 16;
  if (qb >= e.len) return;   // (uniform over the block)
  const int lo = a.d.first(e.pos0) & ~(KV_PAGE_TOKENS - 1), W = a.d.window > 0 ? a.d.window : 1 << 30;
  const int qpos = e.pos0 + min(q0 + c, e.len - 1), qpos0 = e.pos0 + min(q0, e.len - 1), qpos1 = e.pos0 + min(q0 + 15, e.len - 1);   // of the lane's, the wave's first and last rows
  const int64_t ldkv = (int64_t)a.d.heads * (a.d.dp + a.d.vp), ldc = a.d.ldc();
  const int64_t ext = a.ext0[blockIdx.y];
  const int nrow = e.pos0 + e.len - lo;   // gathered rows of the entry; tile t holds rows t * 64 .., position lo + row
  const bf16_t* kvb = (const bf16_t*)a.kv + ext * ldkv;
  const bf16_t* latb = (const bf16_t*)a.lat + ext * ldc + a.d.rp;
  const int dpk = a.d.dp >> 5;
  bf16x8_t qf[KS];
  {
    const bf16_t* qp = (const bf16_t*)a.q + (int64_t)(e.row0 + min(q0 + c, e.len - 1)) * a.ldq + (int64_t)head * DQK + G * 8;
#pragma unroll
    for (int k4 = 0; k4 < KS; ++k4) qf[k4] = as_frag(ld16(qp + k4 * 32));
  }
  auto stage = [&](int tile) __attribute__((always_inline)) {
    char* dst = smem + (tile & 1) * STAGE;
#pragma unroll
    for (int i = 0; i < (KB + NWV - 1) / NWV; ++i) {
      const int blk = wave + i * NWV;
      if (KB % NWV == 0 || blk < KB) {
        const int sub = blk / KS, k4 = blk - sub * KS, row = min(tile * 64 + sub * 16 + c, nrow - 1);
        const bf16_t* src = k4 < dpk ? kvb + row * ldkv + head * a.d.dp + k4 * 32 + G * 8 : latb + row * ldc + (k4 - dpk) * 32 + G * 8;
        __builtin_amdgcn_global_load_lds((glb_ptr_t)src, (lds_ptr_t)(dst + blk * 1024), 16, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < (VB + NWV - 1) / NWV; ++i) {
      const int blk = wave + i * NWV;
      if (VB % NWV == 0 || blk < VB) {
        const int sub = blk / VS, k4 = blk - sub * VS, row = min(tile * 64 + sub * 16 + c, nrow - 1);
        const bf16_t* src = kvb + row * ldkv + a.d.heads * a.d.dp + head * DV + k4 * 32 + G * 8;
        __builtin_amdgcn_global_load_lds((glb_ptr_t)src, (lds_ptr_t)(dst + (KB + blk) * 1024), 16, 0, 0);
      }
    }
  };
  const int tile0 = (a.d.first(e.pos0 + qb) - lo) >> 6, ntiles = ((e.pos0 + min(qb + 16 * NWV, e.len) - 1 - lo) >> 6) + 1;
  float m = -INFINITY, l = 0.f;
  f32x4_t o[DS];
#pragma unroll
  for (int i = 0; i < DS; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  stage(tile0);
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
  __syncthreads();
  const int tr_row = G * 4 + (c >> 2), tr_col = (c & 3) * 4;
  for (int tile = tile0; tile < ntiles; ++tile) {
    stage(tile + 1);   // (behind the last tile: the clamped last row, nobody reads it)
    const int t0 = lo + tile * 64;
    if (t0 <= qpos1 && t0 + 63 > qpos0 - W) {   // wave-uniform: some row of the wave sees some position of the tile
      const char* ks = smem + (tile & 1) * STAGE;
      const char* vs = ks + KB * 1024;
      f32x4_t st[4];
#pragma unroll
      for (int sub = 0; sub < 4; ++sub) st[sub] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      {
        auto kread = [&](int f) { return *reinterpret_cast<const u32x4_t*>(ks + (((f & 3) * KS + (f >> 2)) * 64 + lane) * 16); };   // fragment (k4, sub) = (f / 4, f % 4)
        u32x4_t ring[KRING];
#pragma unroll
        for (int f = 0; f < KRING; ++f) ring[f] = kread(f);
#pragma unroll
        for (int f = 0; f < KB; ++f) {
          st[f & 3] = mfma16(as_frag(ring[f % KRING]), qf[f >> 2], st[f & 3]);
          if (f + KRING < KB) ring[f % KRING] = kread(f + KRING);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      float alpha, m2;
      if (t0 + 63 <= qpos0 && t0 > qpos1 - W) softmax_scores<3>(st, a.d.scale, [](int) { return true; }, G, m, alpha, m2);
      else softmax_scores<3>(st, a.d.scale, [&](int tk) { return t0 + tk <= qpos && t0 + tk > qpos - W; }, G, m, alpha, m2);
      auto vread = [&](int f) {   // V^T fragment f = (kk, ds) = (f / DS, f % DS)
        const int n = (f % DS) * 16 + tr_col;
        const char* p = vs + ((((f / DS) * 2 * VS + (n >> 5)) * 64 + ((n >> 3) & 3) * 16 + tr_row) * 16) + (n & 7) * 2;
        union { tr4_t t[2]; u32x4_t u; } x;
        x.t[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)p);
        x.t[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(p + VS * 1024));
        return x.u;
      };
      u32x4_t vring[VRING];
#pragma unroll
      for (int f = 0; f < VRING; ++f) vring[f] = vread(f);
      __builtin_amdgcn_sched_barrier(0);
      bf16x8_t pf[2];
      softmax_probs<true>(st, m2, alpha, l, pf, a.d.scale * LOG2E);
      if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) o[ds] *= alpha;
      }
#pragma unroll
      for (int f = 0; f < 2 * DS; ++f) {
        o[f % DS] = mfma16(as_frag(vring[f % VRING]), pf[f / DS], o[f % DS]);
        if (f + VRING < 2 * DS) vring[f % VRING] = vread(f + VRING);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);   // this wave's share of the next tile has landed
    __syncthreads();
  }
  const float inv = 1.0f / group_sum(l);
  if (q0 + c < e.len) {
    bf16_t* op = (bf16_t*)a.o + (int64_t)(e.row0 + q0 + c) * a.ldo + head * DV + G * 4;
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) *reinterpret_cast<uint2*>(op + ds * 16) = make_uint2(pack_bf(o[ds][0] * inv, o[ds][1] * inv), pack_bf(o[ds][2] * inv, o[ds][3] * inv));
  }
}

// ---- one token per sequence, in the latent space ---------------------------------------------------------------------------------------------
// Block (split, 16 heads, sequence), four waves; tiles of 32 positions in two LDS stages, fragment blocks as above.  Scores: wave w takes positions
// (w & 1) * 16 .. and half w >> 1 of the dims, the halves meet in LDS; every wave then does the (small) softmax of all 16 x 32 scores and the
// sum for its quarter of the latent dims.
constexpr int LD_NT = 256;
__host__ __device__ inline int latent_decode_lds(const LatentDims& d) { return (int)((d.ldc() / 32) * 1024 * 5 + 4 * 256 * 4); }
template <int NDS>   // 16-dim tiles of the latent per wave
__global__ __launch_bounds__(LD_NT) void latent_decode_kernel(LatentDecodeArgs a, SeqBatch b) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), G = lane >> 4, c = lane & 15;
  const int KS = (int)(a.d.ldc() >> 5), RS = a.d.rp >> 5, split = blockIdx.x, hg = blockIdx.y, heads = a.d.heads;
  char* const Qs = smem;                                   // [KS] fragments
  char* const Ks = Qs + KS * 1024;                         // 2 stages x [2][KS] fragments
  float* const ps = reinterpret_cast<float*>(Ks + KS * 4096);   // [4 waves][16 heads][16 positions]
  const int stage_bytes = KS * 2048;
  const SeqEntry e = seq_entry_at(b, blockIdx.z);
  const int pos = e.pos0, lo = a.d.first(pos), tl0 = lo >> 5, nt = (pos >> 5) - tl0 + 1, per = (nt + a.nsplit - 1) / a.nsplit;
  const int ta = tl0 + min(split * per, nt), tb = tl0 + min((split + 1) * per, nt);
  const int head = min(hg * 16 + c, heads - 1);
  auto stage = [&](int tile) {   // wave w: position half w & 1, every other dim block
    const uint64_t base = a.c.tab[(int64_t)e.slot * a.c.ld + (tile >> 1)] + a.c.off;
    const int row = (tile & 1) * 32 + (wave & 1) * 16 + c, p = min((tile >> 1) * 64 + row, pos) & 63;   // (positions behind the newest: its row)
    const uint64_t src = base + ((uint64_t)p * a.d.ldc() + G * 8) * 2;
    char* dst = Ks + (tile & 1) * stage_bytes + (wave & 1) * KS * 1024;
    for (int k4 = wave >> 1; k4 < KS; k4 += 2) __builtin_amdgcn_global_load_lds((glb_ptr_t)(src + k4 * 64), (lds_ptr_t)(dst + k4 * 1024), 16, 0, 0);
  };
  f32x4_t o[NDS];
#pragma unroll
  for (int i = 0; i < NDS; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  if (ta < tb) {
    stage(ta);
    const bf16_t *qa = (const bf16_t*)a.qa + ((int64_t)blockIdx.z * heads + head) * a.d.rp, *qr = (const bf16_t*)a.qr + ((int64_t)blockIdx.z * heads + head) * a.d.tp;
    for (int k4 = wave; k4 < KS; k4 += 4)
      *reinterpret_cast<u32x4_t*>(Qs + (k4 * 64 + lane) * 16) = ld16(k4 < RS ? qa + k4 * 32 + G * 8 : qr + (k4 - RS) * 32 + G * 8);
  }
  const int tr_row = G * 4 + (c >> 2), tr_col = (c & 3) * 4;
  const int kh = (KS + 1) >> 1, ka = (wave >> 1) * kh, kb = min(KS, ka + kh);
  for (int tile = ta; tile < tb; ++tile) {
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();   // the tile is whole; everyone is past the stage the next one goes to
    if (tile + 1 < tb) stage(tile + 1);
    const char* ks = Ks + (tile & 1) * stage_bytes;
    f32x4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k4 = ka; k4 < kb; ++k4)
      s = mfma16(as_frag(*reinterpret_cast<const u32x4_t*>(ks + (((wave & 1) * KS + k4) * 64 + lane) * 16)), as_frag(*reinterpret_cast<const u32x4_t*>(Qs + (k4 * 64 + lane) * 16)), s);
    *reinterpret_cast<f32x4_t*>(ps + (wave * 16 + c) * 16 + G * 4) = s;
    __syncthreads();
    float sc[8];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const f32x4_t x = *reinterpret_cast<const f32x4_t*>(ps + (u * 16 + c) * 16 + G * 4) + *reinterpret_cast<const f32x4_t*>(ps + ((u + 2) * 16 + c) * 16 + G * 4);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int p = tile * 32 + u * 16 + G * 4 + r;
        sc[u * 4 + r] = p >= lo && p <= pos ? x[r] * (a.d.scale * LOG2E) : -INFINITY;
      }
    }
    float tm = sc[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) tm = fmaxf(tm, sc[j]);
    tm = group_max(tm);                          // (a tile of the range holds at least one visible position)
    const float mn = fmaxf(m, tm), al = __builtin_amdgcn_exp2f(m - mn);
    float p[8], sum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      p[j] = __builtin_amdgcn_exp2f(sc[j] - mn);
      sum += p[j];
    }
    l = l * al + sum;
    m = mn;
    const bf16x8_t pf = as_frag(u32x4_t{pack_bf(p[0], p[1]), pack_bf(p[2], p[3]), pack_bf(p[4], p[5]), pack_bf(p[6], p[7])});
#pragma unroll
    for (int i = 0; i < NDS; ++i) {
      const int ds = i * 4 + wave;
      if (ds * 16 < a.d.rp) {
        const int n = ds * 16 + tr_col;
        const char* q = ks + (((n >> 5) * 64 + ((n >> 3) & 3) * 16 + tr_row) * 16) + (n & 7) * 2;
        union { tr4_t t[2]; u32x4_t u; } x;
        x.t[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)q);
        x.t[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(q + KS * 1024));
        o[i] = mfma16(as_frag(x.u), pf, o[i] * al);
      }
    }
  }
  l = group_sum(l);
  if (hg * 16 + c >= heads) return;
  const int64_t at = ((int64_t)blockIdx.z * a.nsplit + split) * heads + head;
#pragma unroll
  for (int i = 0; i < NDS; ++i) {
    const int ds = i * 4 + wave;
    if (ds * 16 < a.d.rp) *reinterpret_cast<f32x4_t*>(a.part_o + at * a.d.rp + ds * 16 + G * 4) = o[i];
  }
  if (wave == 0 && G == 0) *reinterpret_cast<float2*>(a.part_ml + at * 2) = make_float2(m, l);
}

// The same for rp of 128, 256 or 512 and tp of 32 or 64, where a tile's keys and its sums fit one wave: every wave takes tiles of its own, requested at once
// -- no barrier, no exchange of scores and no wait of one tile for another until the four waves' sums meet in LDS.  (Four waves on one tile at a time,
// 4096 positions at rp 256: 8.9 us, 7.1 now; 32 sequences of 100 at rp 512: 10.6, 10.5.)
// ONE: one sequence, its places in the leading arguments, which are in registers before the first instruction; else from the batch's table.
__host__ __device__ inline bool latent_waves_ok(const LatentDims& d) { return (d.rp == 128 || d.rp == 256 || d.rp == 512) && (d.tp == 32 || d.tp == 64); }
__host__ __device__ constexpr int latent_waves_lds(int ldc) { return ldc / 32 * 1024 * 2 * 4 + 4 * 16 * 8; }   // (the sums: rp / 4 KB, fewer)
template <int RS, int TS, bool ONE>   // 32-dim blocks of the latent and of the key part
__global__ __launch_bounds__(LD_NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void latent_waves_kernel(const bf16_t* qa, const bf16_t* qr, const uint64_t* tab, uint64_t off, int heads, int pos, int lo,
                                                                                                        int nsplit, float scale, LatentDecodeArgs a, SeqBatch b) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int KS = RS + TS, rp = RS * 32, tp = TS * 32, ldc = rp + tp;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), G = lane >> 4, c = lane & 15;
  const int split = blockIdx.x, hg = blockIdx.y, seq = ONE ? 0 : blockIdx.z, head = min(hg * 16 + c, heads - 1);
  if constexpr (!ONE) {
    const SeqEntry e = seq_entry_at(b, seq);
    tab += (int64_t)e.slot * a.c.ld;
    pos = e.pos0;
    lo = a.d.first(pos);
    qa += (int64_t)seq * heads * rp;
    qr += (int64_t)seq * heads * tp;
  }
  const int tl0 = lo >> 5, nt = (pos >> 5) - tl0 + 1, per = (nt + nsplit - 1) / nsplit;
  const int ta = tl0 + min(split * per, nt), tb = tl0 + min((split + 1) * per, nt);
  char* const ks = smem + wave * (KS * 2048);   // [2 halves of 16 positions][KS] fragments
  const int own = ta + wave;
  uint64_t base = own < tb ? tab[own >> 1] + off : 0;
  qa += (int64_t)head * rp + G * 8;
  qr += (int64_t)head * tp + G * 8;
  f32x4_t o[RS * 2];
#pragma unroll
  for (int i = 0; i < RS * 2; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const int tr_row = G * 4 + (c >> 2), tr_col = (c & 3) * 4;
  for (int tile = own; tile < tb; tile += 4) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the stage's reads are done)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int p = min((tile >> 1) * 64 + (tile & 1) * 32 + u * 16 + c, pos) & 63;   // (positions behind the newest: its row)
      const uint64_t src = base + (uint32_t)(p * ldc + G * 8) * 2u;
#pragma unroll
      for (int k4 = 0; k4 < KS; ++k4) __builtin_amdgcn_global_load_lds((glb_ptr_t)(src + k4 * 64), (lds_ptr_t)(ks + (u * KS + k4) * 1024), 16, 0, 0);
    }
    bf16x8_t q[KS];   // (for every tile again: 512 dims of them and of the sums are more registers than a wave has)
#pragma unroll
    for (int k4 = 0; k4 < KS; ++k4) q[k4] = as_frag(ld16(k4 < RS ? qa + k4 * 32 : qr + (k4 - RS) * 32));
    if (tile + 4 < tb) base = tab[(tile + 4) >> 1] + off;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    f32x4_t x[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int k4 = 0; k4 < KS; ++k4)
#pragma unroll
      for (int u = 0; u < 2; ++u) x[u] = mfma16(as_frag(*reinterpret_cast<const u32x4_t*>(ks + ((u * KS + k4) * 64 + lane) * 16)), q[k4], x[u]);
    float sc[8];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int p = tile * 32 + u * 16 + G * 4 + r;
        sc[u * 4 + r] = p >= lo && p <= pos ? x[u][r] * (scale * LOG2E) : -INFINITY;
      }
    float tm = sc[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) tm = fmaxf(tm, sc[j]);
    tm = group_max(tm);                          // (a tile of the range holds at least one visible position)
    const float mn = fmaxf(m, tm), al = __builtin_amdgcn_exp2f(m - mn);
    float p[8], sum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      p[j] = __builtin_amdgcn_exp2f(sc[j] - mn);
      sum += p[j];
    }
    l = l * al + sum;
    m = mn;
    const bf16x8_t pf = as_frag(u32x4_t{pack_bf(p[0], p[1]), pack_bf(p[2], p[3]), pack_bf(p[4], p[5]), pack_bf(p[6], p[7])});
#pragma unroll
    for (int i = 0; i < RS * 2; ++i) {
      const int n = i * 16 + tr_col;
      const char* at = ks + (((n >> 5) * 64 + ((n >> 3) & 3) * 16 + tr_row) * 16) + (n & 7) * 2;
      union { tr4_t t[2]; u32x4_t u; } v;
      v.t[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)at);
      v.t[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(at + KS * 1024));
      o[i] = mfma16(as_frag(v.u), pf, o[i] * al);
    }
  }
  l = group_sum(l);
  // the waves' sums over the stages: [wave][16-dim tile][lane]
  float2* const ml = reinterpret_cast<float2*>(smem + KS * 8192);
  if (G == 0) ml[wave * 16 + c] = make_float2(m, l);
  __syncthreads();   // everyone is past its stage
  float M = -INFINITY, L = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) M = fmaxf(M, ml[w * 16 + c].x);
  const float from = M == -INFINITY ? 0.f : M;   // (waves without a tile: exp2(-inf) of nothing)
#pragma unroll
  for (int w = 0; w < 4; ++w) L = fmaf(ml[w * 16 + c].y, __builtin_amdgcn_exp2f(ml[w * 16 + c].x - from), L);
  const float f = __builtin_amdgcn_exp2f(m - from);
#pragma unroll
  for (int i = 0; i < RS * 2; ++i) *reinterpret_cast<f32x4_t*>(smem + ((wave * RS * 2 + i) * 64 + lane) * 16) = o[i] * f;
  __syncthreads();
  if (hg * 16 + c >= heads) return;
  const int64_t at = ((int64_t)seq * nsplit + split) * heads + head;
#pragma unroll
  for (int j = 0; j < RS / 2; ++j) {
    const int i = j * 4 + wave;
    f32x4_t v = *reinterpret_cast<const f32x4_t*>(smem + (i * 64 + lane) * 16);
#pragma unroll
    for (int w = 1; w < 4; ++w) v += *reinterpret_cast<const f32x4_t*>(smem + ((w * RS * 2 + i) * 64 + lane) * 16);
    *reinterpret_cast<f32x4_t*>(a.part_o + at * rp + i * 16 + G * 4) = v;
  }
  if (wave == 0 && G == 0) *reinterpret_cast<float2*>(a.part_ml + at * 2) = make_float2(M, L);
}

// Block (head, 32 rows of its W_uv, sequence): the splits' latent sums joined into LDS, then eight rows per wave.  wuv null: the joined sums
template <int RQ>   // rp / 256, rounded up
__global__ __launch_bounds__(256) void latent_merge_kernel(const float* part_o, const float* part_ml, const bf16_t* wuv, int nsplit, int heads, int rp, int vp, LatentMergeArgs a) {
  __shared__ float lat[RQ * 256], wt[LATENT_MAX_SPLIT];
  const int h = blockIdx.x, n = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t at = (int64_t)n * nsplit * heads + h;
  const int row0 = blockIdx.y * 32 + wave * 8;
  constexpr int RC = (RQ + 1) / 2;   // 16-byte pieces of a W_uv row per lane
  float2 ml = make_float2(-INFINITY, 0.f);
  if (tid < nsplit) ml = *reinterpret_cast<const float2*>(part_ml + (at + (int64_t)tid * heads) * 2);   // (nsplit <= 64: wave 0)
  // The splits' sums, up to 64 of them requested at once and ahead of the weights that join them (one after the other behind the weights' barrier, the 64 of
  // a 4096-position window made the launch 8.8 us, 32 at a time 5.7; 4.4 now, in 43 splits).  Eight at a time are skipped behind the end; the last one again within.
  constexpr int NB = RQ == 1 ? 64 : RQ == 2 ? 32 : 16;
  const char* part = reinterpret_cast<const char*>(part_o + at * rp);
  uint32_t col[RQ];   // (byte offsets: LATENT_MAX_SPLIT x heads x rp floats, latent_decode_ok)
  float v[RQ][NB];
  auto request = [&](int s0) {
#pragma unroll
    for (int j8 = 0; j8 < NB; j8 += 8) {
      if (s0 + j8 >= nsplit) break;
#pragma unroll
      for (int j = j8; j < j8 + 8; ++j)
#pragma unroll
        for (int q = 0; q < RQ; ++q) v[q][j] = *reinterpret_cast<const float*>(part + (col[q] + (uint32_t)(min(s0 + j, nsplit - 1) * heads * rp) * 4u));
    }
  };
#pragma unroll
  for (int q = 0; q < RQ; ++q) col[q] = (uint32_t)min(q * 256 + tid, rp - 1) * 4u;
  request(0);
  u32x4_t w[8][RC];
  if (wuv) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int q = 0; q < RC; ++q) w[j][q] = ld16(wuv + ((int64_t)h * vp + row0 + j) * rp + min((q * 64 + lane) * 8, rp - 8));
  }
  if (tid < 64) {
    const float M = wave_max(ml.x), e = ml.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml.x - M), s = wave_sum(e * ml.y);
    wt[lane] = e / s;
  }
  __syncthreads();
  float sum[RQ];
#pragma unroll
  for (int q = 0; q < RQ; ++q) sum[q] = 0.f;
  for (int s0 = 0; s0 < nsplit; s0 += NB) {
    if (s0 > 0) request(s0);
#pragma unroll
    for (int j8 = 0; j8 < NB; j8 += 8) {
      if (s0 + j8 >= nsplit) break;
#pragma unroll
      for (int j = j8; j < j8 + 8; ++j)
#pragma unroll
        for (int q = 0; q < RQ; ++q) sum[q] = s0 + j < nsplit ? fmaf(wt[s0 + j], v[q][j], sum[q]) : sum[q];
    }
  }
#pragma unroll
  for (int q = 0; q < RQ; ++q) lat[q * 256 + tid] = q * 256 + tid < rp ? sum[q] : 0.f;
  if (!wuv) {
    for (int d = tid; d < rp; d += 256) ((bf16_t*)a.o)[((int64_t)n * heads + h) * rp + d] = f2bf(lat[d]);   // (own elements)
    return;
  }
  __syncthreads();
  float acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = 0.f;
#pragma unroll
  for (int q = 0; q < RC; ++q) {
    const int k = (q * 64 + lane) * 8;
    if (k < rp) {
      const float4 x0 = *reinterpret_cast<const float4*>(lat + k), x1 = *reinterpret_cast<const float4*>(lat + k + 4);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const u32x4_t v = w[j][q];
        acc[j] = fmaf(x0.x, lo_bf(v[0]), fmaf(x0.y, hi_bf(v[0]), fmaf(x0.z, lo_bf(v[1]), fmaf(x0.w, hi_bf(v[1]), acc[j]))));
        acc[j] = fmaf(x1.x, lo_bf(v[2]), fmaf(x1.y, hi_bf(v[2]), fmaf(x1.z, lo_bf(v[3]), fmaf(x1.w, hi_bf(v[3]), acc[j]))));
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = wave_sum(acc[j]);
  if (lane == 0) {
    u32x4_t v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = pack_bf(acc[2 * j], acc[2 * j + 1]);
    *reinterpret_cast<u32x4_t*>((bf16_t*)a.o + (int64_t)n * a.ldo + h * vp + row0) = v;
  }
}

int pad_to(int d, const int* opts, int n) {
  for (int i = 0; i < n; ++i)
    if (d <= opts[i]) return opts[i];
  return 0;
}

template <class F>
void by_qk_v(int dqk, int dv, F&& f) {
  using std::integral_constant;
  auto inner = [&](auto q) {
    if (dv == 32) f(q, integral_constant<int, 32>{});
    else if (dv == 64) f(q, integral_constant<int, 64>{});
    else if (dv == 128) f(q, integral_constant<int, 128>{});
    else f(q, integral_constant<int, 256>{});
  };
  if (dqk == 64) inner(integral_constant<int, 64>{});
  else if (dqk == 96) inner(integral_constant<int, 96>{});
  else if (dqk == 128) inner(integral_constant<int, 128>{});
  else if (dqk == 192) inner(integral_constant<int, 192>{});
  else inner(integral_constant<int, 256>{});
}

}  // namespace

bool latent_prefill_dims(int dim, int rot, int vdim, int* dp, int* tp, int* vp) {
  static const int qk[] = {64, 96, 128, 192, 256}, v[] = {32, 64, 128, 256};
  *tp = (rot + 31) / 32 * 32;
  const int dqk = pad_to((dim + 31) / 32 * 32 + *tp, qk, 5);
  *dp = dqk - *tp;
  *vp = pad_to(vdim, v, 4);
  if (dqk && *vp) return true;
  *dp = (dim + 31) / 32 * 32;
  *vp = (vdim + 31) / 32 * 32;
  return false;
}

void launch_latent_post(const LatentPostArgs& a, const SeqBatch& b, bool f32, hipStream_t st) {
  if (b.rows <= 0) return;
  const dim3 grid((unsigned)b.rows), block(256);
  if (f32) hipLaunchKernelGGL((latent_post_kernel<float, float>), grid, block, 0, st, a, b);
  else hipLaunchKernelGGL((latent_post_kernel<bf16_t, bf16_t>), grid, block, 0, st, a, b);
}

void launch_latent_query(const LatentQueryArgs& a, const SeqBatch& b, hipStream_t st) {
  if (b.n <= 0) return;
  const LatentDims& d = a.p.d;
  const int nx = d.rp / 64, append = a.p.kv_off >= 0 ? (std::min(b.n, 16) + nx - 1) / nx : 0;
  const dim3 grid((unsigned)nx, (unsigned)(d.heads + append), (unsigned)((b.n + 15) / 16)), block(256);
  auto go = [&](auto ti) {
    using TI = decltype(ti);
    hipLaunchKernelGGL(latent_query_kernel<TI>, grid, block, 0, st, (const TI*)a.p.in, (const bf16_t*)a.w_ukt, (const float2*)a.p.rope, (int)a.p.ld, d.heads, d.rp, d.dp, d.tp, d.rot, b.n, a, b);
  };
  if (a.p.in_f32) go(float{});
  else go(bf16_t{});
}

void launch_heads_gemm(const HeadsGemmArgs& a, bool f32, hipStream_t st) {
  if (a.rows <= 0) return;
  if (f32) {
    launch_gemm_f32((const float*)a.A, a.lda, a.W, a.k, (float*)a.C, a.ldc, a.rows, a.n, a.k, st, a.heads, a.sa, (int64_t)a.n * a.k, a.sc);
    return;
  }
  auto go = [&](auto mt) {
    constexpr int MT = decltype(mt)::value;
    hipLaunchKernelGGL(heads_gemm_kernel<MT>, dim3((unsigned)((a.n + 63) / 64), (unsigned)a.heads, (unsigned)((a.rows + MT * 16 - 1) / (MT * 16))), dim3(256), 0, st, a);
  };
  if (a.rows <= 16) go(std::integral_constant<int, 1>{});
  else go(std::integral_constant<int, 4>{});
}

void launch_latent_rows(const LatentRowsArgs& a, const SeqBatch& b, bool f32, hipStream_t st) {
  if (b.rows <= 0) return;
  const dim3 grid((unsigned)b.rows, (unsigned)a.d.heads), block(64);
  const size_t lds = (size_t)(a.d.rp + a.d.tp + 64) * 4;
  if (f32) hipLaunchKernelGGL(latent_rows_kernel<float>, grid, block, lds, st, a, b);
  else hipLaunchKernelGGL(latent_rows_kernel<bf16_t>, grid, block, lds, st, a, b);
}

void launch_latent_gather(const LatentDims& d, const LatentCache& c, const int32_t* ext0, void* out, const SeqBatch& b, int max_rows, bool f32, hipStream_t st) {
  if (b.rows <= 0 || max_rows <= 0) return;
  const int64_t pieces = (int64_t)max_rows * (d.ldc() / (f32 ? 4 : 8));
  const dim3 grid((unsigned)((pieces + 255) / 256), (unsigned)b.n), block(256);
  if (f32) hipLaunchKernelGGL(latent_gather_kernel<float>, grid, block, 0, st, d, c, ext0, (float*)out, b);
  else hipLaunchKernelGGL(latent_gather_kernel<bf16_t>, grid, block, 0, st, d, c, ext0, (bf16_t*)out, b);
}

void launch_latent_prefill(const LatentPrefillArgs& a, const SeqBatch& b, hipStream_t st) {
  if (b.rows <= 0) return;
  const bool wide = (int64_t)((b.max_len + 127) / 128) * a.d.heads * b.n >= 512;
  by_qk_v(a.d.qd(), a.d.vp, [&](auto q, auto v) {
    constexpr int DQK = decltype(q)::value, DV = decltype(v)::value, lds = 2 * 64 * (DQK + DV) * 2;
    auto go = [&](auto nw) {
      constexpr int NWV = decltype(nw)::value;
      const int nqb = (b.max_len + 16 * NWV - 1) / (16 * NWV);
      auto k = latent_prefill_kernel<DQK, DV, NWV>;
      if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      hipLaunchKernelGGL(k, dim3((unsigned)(nqb * a.d.heads), (unsigned)b.n), dim3(NWV * 64), lds, st, a, b, nqb);
    };
    if (wide) go(std::integral_constant<int, 8>{});
    else go(std::integral_constant<int, 4>{});
  });
}

int latent_decode_blocks_per_cu(const LatentDims& d) { return std::max(1, std::min(2, 160 * 1024 / (latent_waves_ok(d) ? latent_waves_lds((int)d.ldc()) : latent_decode_lds(d)))); }
bool latent_decode_ok(const LatentDims& d) { return d.rp <= 1024 && (int64_t)d.heads * d.rp < 1 << 24 && latent_decode_lds(d) <= 160 * 1024 && d.scale > 0.f; }

void launch_latent_decode(const LatentDecodeArgs& a, const SeqBatch& b, hipStream_t st) {
  if (b.n <= 0) return;
  const bool waves = latent_waves_ok(a.d);
  const int lds = waves ? latent_waves_lds((int)a.d.ldc()) : latent_decode_lds(a.d);
  const dim3 grid((unsigned)a.nsplit, (unsigned)((a.d.heads + 15) / 16), (unsigned)b.n);
  auto allow = [&](auto k) {
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    return k;
  };
  if (waves) {
    auto go = [&](auto rs, auto ts, auto one) {
      constexpr bool ONE = decltype(one)::value;
      auto k = allow(latent_waves_kernel<decltype(rs)::value, decltype(ts)::value, ONE>);
      const int pos = b.one.pos0;
      hipLaunchKernelGGL(k, grid, dim3(LD_NT), lds, st, (const bf16_t*)a.qa, (const bf16_t*)a.qr, a.c.tab + (ONE ? (int64_t)b.one.slot * a.c.ld : 0), a.c.off, a.d.heads, pos, a.d.first(pos),
                         a.nsplit, a.d.scale, a, b);
    };
    auto by_rank = [&](auto ts, auto one) {
      if (a.d.rp == 128) go(std::integral_constant<int, 4>{}, ts, one);
      else if (a.d.rp == 256) go(std::integral_constant<int, 8>{}, ts, one);
      else go(std::integral_constant<int, 16>{}, ts, one);
    };
    auto by_key = [&](auto one) {
      if (a.d.tp == 32) by_rank(std::integral_constant<int, 1>{}, one);
      else by_rank(std::integral_constant<int, 2>{}, one);
    };
    if (b.has_one) by_key(std::true_type{});
    else by_key(std::false_type{});
    return;
  }
  auto go = [&](auto nds) { hipLaunchKernelGGL(allow(latent_decode_kernel<decltype(nds)::value>), grid, dim3(LD_NT), lds, st, a, b); };
  if (a.d.rp <= 128) go(std::integral_constant<int, 2>{});
  else if (a.d.rp <= 256) go(std::integral_constant<int, 4>{});
  else if (a.d.rp <= 512) go(std::integral_constant<int, 8>{});
  else go(std::integral_constant<int, 16>{});
}

void launch_latent_merge(const LatentMergeArgs& a, hipStream_t st) {
  if (a.n <= 0) return;
  const dim3 grid((unsigned)a.d.heads, (unsigned)(a.wuv ? a.d.vp / 32 : 1), (unsigned)a.n), block(256);
  auto go = [&](auto rq) {
    hipLaunchKernelGGL(latent_merge_kernel<decltype(rq)::value>, grid, block, 0, st, a.part_o, a.part_ml, (const bf16_t*)a.wuv, a.nsplit, a.d.heads, a.d.rp, a.d.vp, a);
  };
  if (a.d.rp <= 256) go(std::integral_constant<int, 1>{});
  else if (a.d.rp <= 512) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 4>{});
}

}  // namespace aha
