// Attention over several sequences with a chunked causal mask and a sink (layered.hip): query position i sees the keys
// floor(i / chunk) * chunk .. i of its own sequence; a sink adds a key of score 0 without a value, i.e. one to the softmax's denominator.
//   prompt rows:   attn_prefill_kernel<.., CHUNK = 1> (attn_prefill_body.h) on fragment-major bf16 pages
//   one token each: attn_chunk_decode_kernel: q / k norm + rotation + value mixing + KV append + split-KV attention + merge, one launch
//   the 32-bit mode, heads of 64 or 128 dims: attn_chunk_f32_kernel on token-major pages, one token each: attn_chunk_f32_decode_kernel
//   any head dims: attn_chunk_rows_kernel on token-major pages
// q head h reads kv head h / (heads / kv heads).  Scores, maxima, exponentials and sums are f32; P feeds the MFMA as bf16.
#include <algorithm>

#include <type_traits>

#include "attn_prefill_body.h"

namespace aha {

namespace {

// ---- decode ----------------------------------------------------------------------------------------------------------------------
// Block (split, kv head, sequence), four waves; wave w of split s is unit s * 4 + w and takes the chunk's pages unit, unit + units, ...
// Every block redoes the small per-token work (sums of squares over the whole q / k projections, norm + rotation of its g query heads and of
// the new key, the new value); split 0 appends the new key and value to the page, unit 0 owns the sink, the last
// unit begins with the new token from LDS.
// Partials: one un-normalised (max, sum, O) per split and head, written through to memory; the split block that arrives last at the kv head's
// counter merges them, writes the output and resets the counter.
// What bounds it is the work in front of and behind the pages: 14.6 us at 8 sequences of ~260 positions (32 / 8 heads x 128) with the sums read by
// elements, the last page requested twice, the new token scored behind unit 0's pages and the waves merged by dwords; 11.4 us as it is.
// TI: type of the qkv row (float behind the decode matvec, bf16 behind a GEMM).
constexpr int CD_NW = 4, CD_NT = CD_NW * 64;
template <int DQK, int DV>
constexpr int chunk_decode_lds() { return (16 * DQK + DQK + DV) * 2 + CD_NW * DV * 16 * 4 + 2 * CD_NW * 16 * 4; }

template <typename TI>
__device__ __forceinline__ float ld_in(const void* p, int i);
template <>
__device__ __forceinline__ float ld_in<float>(const void* p, int i) { return ((const float*)p)[i]; }
template <>
__device__ __forceinline__ float ld_in<bf16_t>(const void* p, int i) { return bf2f(((const bf16_t*)p)[i]); }

// LEAN (launch_chunk_attn_decode): whole heads of 128 dims, all of them rotated, q | k | v without gaps, up to 4096 query and 2048 key columns, up to
// seven query heads per kv head.  Row i of the step is sequence i, so the row, the norms, the angles and the values are requested before the sequence's
// entry is there, the page table behind them, the pages behind that -- three round trips where the loops below make one per group of columns and head --
// and the pages go through a descriptor that is empty for a unit without any (attn_decode_body.h): 11.4 -> 9.5 us
// at 8 sequences of ~260 positions.
template <int DQK, int DV, typename TI, bool LEAN = false, bool BIAS = false>
__global__ __launch_bounds__(CD_NT) void attn_chunk_decode_kernel(const void* qkv_, const float* bias_, const void* q_norm_, const void* k_norm_, const SeqEntry* entries_, const uint64_t* tab_,
                                                                  int ld_, int g_kvh_nsplit, ChunkDecodeArgs a, SeqBatch b) {
  // (what the first requests need: in scalar registers at the start, gemv_body.h)
  a.p.qkv = qkv_;
  a.p.bias = bias_;
  a.p.q_norm = q_norm_;
  a.p.k_norm = k_norm_;
  b.entries = entries_;
  a.p.kv.tab = tab_;
  a.p.ld = ld_;
  a.nsplit = g_kvh_nsplit & 0xff;
  if (LEAN) {
    a.p.kvh = g_kvh_nsplit >> 8 & 0xfff;
    a.p.heads = (g_kvh_nsplit >> 20) * a.p.kvh;
  }
  constexpr int KS = DQK / 32, DS = DV / 16;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  bf16_t* qs = reinterpret_cast<bf16_t*>(smem);    // [16][DQK]
  bf16_t* ksn = qs + 16 * DQK;                     // [DQK]
  bf16_t* vsn = ksn + DQK;                         // [DV]
  float* mo = reinterpret_cast<float*>(vsn + DV);  // per wave O [CD_NW][16][DV]
  float* mm = mo + CD_NW * DV * 16;                // [CD_NW][16]
  float* mlz = mm + CD_NW * 16;                    // [CD_NW][16]
  __shared__ float red[2][CD_NW];
  __shared__ int s_last;
  const int tid = (int)threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, G = lane >> 4, c = lane & 15;
  const int split = blockIdx.x, kvhd = blockIdx.y, ent = blockIdx.z, nsplit = a.nsplit;
  const QkvPostArgs& p = a.p;
  const int g = LEAN ? g_kvh_nsplit >> 20 : p.heads / p.kvh;
  // (LEAN: the requests that need no entry, in the order their data is needed)
  constexpr int PER8 = std::is_same<TI, float>::value ? 2 : 1;   // 16-byte requests per eight columns
  u32x4_t rq8[2][PER8], rk8[PER8];
  f32x4_t bq8[2][2], bk8[2];
  float hx[2][2], hb[2][2];
  bf16_t hw[2][2];
  float vraw = 0.f, vbias = 0.f;
  if constexpr (LEAN) {
    const int nq = g * p.kvh * 128, nk = p.kvh * 128;
    const TI* row = (const TI*)p.qkv + (int64_t)ent * p.ld;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = min(tid * 8 + j * 2048, nq - 8);
#pragma unroll
      for (int k = 0; k < PER8; ++k) rq8[j][k] = ld16(row + i + k * 4);
      if (BIAS) bq8[j][0] = *reinterpret_cast<const f32x4_t*>(p.bias + i), bq8[j][1] = *reinterpret_cast<const f32x4_t*>(p.bias + i + 4);
    }
    const int ik = nq + min(tid * 8, nk - 8);
#pragma unroll
    for (int k = 0; k < PER8; ++k) rk8[k] = ld16(row + ik + k * 4);
    if (BIAS) bk8[0] = *reinterpret_cast<const f32x4_t*>(p.bias + ik), bk8[1] = *reinterpret_cast<const f32x4_t*>(p.bias + ik + 4);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int hs = min(wave + j * CD_NW, g), w0 = (hs == g ? kvhd : kvhd * g + hs) * 128, off = (hs == g ? nq : 0) + w0;
      const bf16_t* w = (const bf16_t*)(hs == g ? p.k_norm : p.q_norm) + w0;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        hx[j][k] = ld_in<TI>(row, off + lane + k * 64);
        if (BIAS) hb[j][k] = p.bias[off + lane + k * 64];
        hw[j][k] = w[lane + k * 64];
      }
    }
    vraw = ld_in<TI>(row, nq + nk + kvhd * 128 + (tid & 127));
    if (BIAS) vbias = p.bias[nq + nk + kvhd * 128 + (tid & 127)];
  }
  const SeqEntry e = seq_entry_at(b, ent);
  const int pos = e.pos0;
  const int lo = a.chunk > 0 ? pos / a.chunk * a.chunk : 0;   // first visible position; the new token's own is pos
  const int page0 = lo / KV_PAGE_TOKENS, npages = pos > lo ? (pos - 1) / KV_PAGE_TOKENS - page0 + 1 : 0;   // pages of the OLD tokens
  const int nunits = nsplit * CD_NW, unit = split * CD_NW + wave;
  const uint64_t* tab = p.kv.tab + (int64_t)e.slot * p.kv.ld;

  typedef const __attribute__((address_space(1))) char* gchar_t;
  const uint32_t l_off = (uint32_t)lane * 16;
  u32x4_t kf[4][KS], vf[DS][2];
  uint64_t my_pages = 0;   // LEAN: lane i: this unit's i-th page, lane 63: the new token's
  auto page_of = [&](int it) {
    const uint32_t x = __builtin_amdgcn_readlane((uint32_t)my_pages, it), y = __builtin_amdgcn_readlane((uint32_t)(my_pages >> 32), it);
    return (uint64_t)y << 32 | x;
  };
  auto page_base = [&](int i) {
    if (LEAN && (i - unit) / nunits < 63) return page_of((i - unit) / nunits);
    return (uint64_t)(tab[page0 + i] + p.kv.layer_off);
  };
  auto load_k = [&](uint64_t base, bool have = true) {
    if constexpr (LEAN) {
      const auto rs = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(base), 0, have ? p.kvh * KV_PAGE_TOKENS * (DQK + DV) * 2 : 0, 0x00020000);
#pragma unroll
      for (int sub = 0; sub < 4; ++sub)
#pragma unroll
        for (int k4 = 0; k4 < KS; ++k4)
          kf[sub][k4] = __builtin_amdgcn_raw_buffer_load_b128(rs, l_off + (sub * KS + k4) % 4 * 1024, kvhd * (KV_PAGE_TOKENS * DQK * 2) + (sub * KS + k4) / 4 * 4096, 2 /* nt */);
      return;
    }
    gchar_t kb = reinterpret_cast<gchar_t>(base + (uint64_t)kvhd * (KV_PAGE_TOKENS * DQK * 2));
#pragma unroll
    for (int sub = 0; sub < 4; ++sub)
#pragma unroll
      for (int k4 = 0; k4 < KS; ++k4) kf[sub][k4] = __builtin_nontemporal_load(reinterpret_cast<gptr16_t>(kb + (sub * KS + k4) * 1024 + l_off));
  };
  auto load_v = [&](uint64_t base, bool have = true) {
    if constexpr (LEAN) {
      const auto rs = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(base), 0, have ? p.kvh * KV_PAGE_TOKENS * (DQK + DV) * 2 : 0, 0x00020000);
#pragma unroll
      for (int ds = 0; ds < DS; ++ds)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
          vf[ds][kk] = __builtin_amdgcn_raw_buffer_load_b128(rs, l_off + (ds * 2 + kk) % 4 * 1024, p.kvh * (KV_PAGE_TOKENS * DQK * 2) + kvhd * (DV * KV_PAGE_TOKENS * 2) + (ds * 2 + kk) / 4 * 4096, 2 /* nt */);
      return;
    }
    gchar_t vb = reinterpret_cast<gchar_t>(base + (uint64_t)p.kvh * (KV_PAGE_TOKENS * DQK * 2) + (uint64_t)kvhd * (DV * KV_PAGE_TOKENS * 2));
#pragma unroll
    for (int ds = 0; ds < DS; ++ds)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) vf[ds][kk] = __builtin_nontemporal_load(reinterpret_cast<gptr16_t>(vb + (ds * 2 + kk) * 1024 + l_off));
  };

  // ---- the new token: sums of squares, norm + rotation of the block's heads, value ------------------------------------------------
  // Requests in the order their data is needed (returns are in order within a wave): the whole q / k row for the sums, this wave's first head
  // and its norm weights and angles, the value, then the unit's first page; the arithmetic runs under the page fetch.
  if constexpr (LEAN) {
    const int nq = g * p.kvh * 128, nk = p.kvh * 128;
    const float2 cs = reinterpret_cast<const float2*>(p.rope)[ent * 64 + lane];
    const int64_t vf_at = ((int64_t)ent * p.kvh + kvhd) * 128 + (tid & 127);
    const float vold = *(p.v_use ? p.v_first + vf_at : p.rope);
    my_pages = tab[lane == 63 ? pos / KV_PAGE_TOKENS : min(page0 + unit + lane * nunits, pos / KV_PAGE_TOKENS)] + p.kv.layer_off;
    const uint64_t b0 = page_of(0);
    __builtin_amdgcn_sched_barrier(0);
    load_k(b0, unit < npages);
    __builtin_amdgcn_sched_barrier(0);
    load_v(b0, unit < npages);
    __builtin_amdgcn_sched_barrier(0);
    auto sq8 = [&](const u32x4_t (&r)[PER8], const f32x4_t (&bi)[2], float s) {
      float v[8];
      if constexpr (PER8 == 2) {
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = __uint_as_float(r[k >> 2][k & 3]);
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) { v[2 * k] = lo_bf(r[0][k]); v[2 * k + 1] = hi_bf(r[0][k]); }
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float x = BIAS ? v[k] + bi[k >> 2][k & 3] : v[k];
        s = fmaf(x, x, s);
      }
      return s;
    };
    float sq = 0.f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float s = sq8(rq8[j], bq8[j], sq);
      sq = tid * 8 + j * 2048 < nq ? s : sq;
    }
    float sk = sq8(rk8, bk8, 0.f);
    sk = tid * 8 < nk ? sk : 0.f;
    sq = wave_sum(sq);
    sk = wave_sum(sk);
    if (lane == 0) { red[0][wave] = sq; red[1][wave] = sk; }
    __syncthreads();
    sq = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
    sk = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    const float rq = 1.0f / sqrtf(sq / (float)nq + p.eps), rk = 1.0f / sqrtf(sk / (float)nk + p.eps);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int hs = wave + j * CD_NW;
      const float rinv = hs == g ? rk : rq;
      const float x = (BIAS ? hx[j][0] + hb[j][0] : hx[j][0]) * rinv * bf2f(hw[j][0]), z = (BIAS ? hx[j][1] + hb[j][1] : hx[j][1]) * rinv * bf2f(hw[j][1]);
      if (hs <= g) {
        const int dst = hs == g ? 16 * DQK : hs * DQK;
        qs[dst + lane] = f2bf(fmaf(x, cs.x, -z * cs.y));
        qs[dst + lane + 64] = f2bf(fmaf(z, cs.x, x * cs.y));
      }
    }
    if (tid < 128) {
      float v = BIAS ? vraw + vbias : vraw;
      if (p.v_store && split == 0) p.v_first[vf_at] = v;
      if (p.v_use) v = fmaf(p.lambda, vold, (1.f - p.lambda) * v);
      vsn[tid] = f2bf(v);
    }
  } else {
    constexpr int ND = (DQK + 63) / 64, NVD = (DV + CD_NT - 1) / CD_NT;
    const char* row = (const char*)p.qkv + (int64_t)e.row0 * p.ld * (int64_t)sizeof(TI);
    const int nq = p.heads * p.dim, nk = p.kvh * p.dim, nv = p.kvh * p.vdim, half = p.rope_dims / 2;
    const float2* cs = reinterpret_cast<const float2*>(p.rope) + (int64_t)e.row0 * half;
    auto col = [&](int i) { return ld_in<TI>(row, i) + (p.bias ? p.bias[i] : 0.f); };
    uint64_t b0 = 0;
    if (unit < npages) b0 = page_base(unit);
    float sq = 0.f, sk = 0.f;
    constexpr int BQ = 8;   // columns of the row requested together
    // the row in 16-byte pieces where it lies so (every head dim that is a multiple of 8 does)
    const bool wide = p.ld % 8 == 0 && p.k_off % 8 == 0 && nq % 8 == 0 && nk % 8 == 0 && (((uintptr_t)p.qkv | (uintptr_t)p.bias) & 15) == 0;
    auto sumsq = [&](int off, int n) {
      float s = 0.f;
      if (wide) {
        for (int i0 = tid * 8; i0 < n; i0 += CD_NT * 16) {
          float v[2][8];
          f32x4_t bi[2][2];
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int i = off + min(i0 + j * CD_NT * 8, n - 8);
            if constexpr (std::is_same<TI, float>::value) {
              *reinterpret_cast<f32x4_t*>(v[j]) = *reinterpret_cast<const f32x4_t*>((const float*)row + i);
              *reinterpret_cast<f32x4_t*>(v[j] + 4) = *reinterpret_cast<const f32x4_t*>((const float*)row + i + 4);
            } else {
              const u32x4_t w = ld16((const bf16_t*)row + i);
#pragma unroll
              for (int k = 0; k < 4; ++k) { v[j][2 * k] = lo_bf(w[k]); v[j][2 * k + 1] = hi_bf(w[k]); }
            }
#pragma unroll
            for (int k = 0; k < 2; ++k) bi[j][k] = p.bias ? *reinterpret_cast<const f32x4_t*>(p.bias + i + 4 * k) : f32x4_t{0.f, 0.f, 0.f, 0.f};
          }
#pragma unroll
          for (int j = 0; j < 2; ++j)
            if (i0 + j * CD_NT * 8 < n) {
#pragma unroll
              for (int k = 0; k < 8; ++k) {
                const float x = v[j][k] + bi[j][k >> 2][k & 3];
                s = fmaf(x, x, s);
              }
            }
        }
        return s;
      }
      for (int i0 = tid; i0 < n; i0 += CD_NT * BQ) {
        float v[BQ];
#pragma unroll
        for (int j = 0; j < BQ; ++j) {
          const int i = i0 + j * CD_NT;
          v[j] = col(off + min(i, n - 1));
          if (i >= n) v[j] = 0.f;
        }
#pragma unroll
        for (int j = 0; j < BQ; ++j) s = fmaf(v[j], v[j], s);
      }
      return s;
    };
    struct Head { float x[ND], z[ND], wx[ND], wz[ND]; float2 t[ND]; };
    auto fetch = [&](int hs, Head& h) {   // hs < g: query head kvhd * g + hs, hs == g: the key
      const bool is_k = hs == g;
      const int w0 = (is_k ? kvhd : kvhd * g + hs) * p.dim, off = is_k ? p.k_off : 0;
      const bf16_t* w = (const bf16_t*)(is_k ? p.k_norm : p.q_norm);
#pragma unroll
      for (int k = 0; k < ND; ++k) {
        const int d = min(lane + k * 64, p.dim - 1), pd = d >= p.rope_dims ? d : d < half ? d + half : d - half;
        h.x[k] = col(off + w0 + d);
        h.z[k] = col(off + w0 + pd);
        h.wx[k] = bf2f(w[w0 + d]);
        h.wz[k] = bf2f(w[w0 + pd]);
        h.t[k] = d < p.rope_dims ? cs[d < half ? d : d - half] : make_float2(1.f, 0.f);
      }
    };
    auto finish = [&](int hs, const Head& h, float rinv) {
      const int dst = hs == g ? 16 * DQK : hs * DQK;
#pragma unroll
      for (int k = 0; k < ND; ++k) {
        const int d = lane + k * 64;
        if (DQK % 64 != 0 && d >= DQK) continue;
        const float y = h.x[k] * rinv * h.wx[k], z = h.z[k] * rinv * h.wz[k];
        const float o = fmaf(y, h.t[k].x, (d < half ? -z : z) * h.t[k].y);
        qs[dst + d] = f2bf(d < p.dim ? o : 0.f);
      }
    };
    sq = sumsq(0, nq);
    sk = sumsq(p.k_off, nk);
    Head first;
    fetch(min(wave, g), first);
    float vnew[NVD], vold[NVD];
#pragma unroll
    for (int k = 0; k < NVD; ++k) {
      const int d = min(tid + k * CD_NT, p.vdim - 1);
      vnew[k] = col(p.v_off + kvhd * p.vdim + d);
      vold[k] = p.v_use ? p.v_first[(int64_t)e.row0 * nv + kvhd * p.vdim + d] : 0.f;
    }
    if (unit < npages) {
      __builtin_amdgcn_sched_barrier(0);
      load_k(b0);
      __builtin_amdgcn_sched_barrier(0);
      load_v(b0);
      __builtin_amdgcn_sched_barrier(0);
    }
    sq = wave_sum(sq);
    sk = wave_sum(sk);
    if (lane == 0) { red[0][wave] = sq; red[1][wave] = sk; }
    __syncthreads();
    sq = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
    sk = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    const float rq = 1.0f / sqrtf(sq / (float)nq + p.eps), rk = 1.0f / sqrtf(sk / (float)nk + p.eps);
    if (wave <= g) finish(wave, first, wave == g ? rk : rq);
    for (int hs = wave + CD_NW; hs <= g; hs += CD_NW) {   // more heads than waves
      Head h;
      fetch(hs, h);
      finish(hs, h, hs == g ? rk : rq);
    }
#pragma unroll
    for (int k = 0; k < NVD; ++k) {
      const int d = tid + k * CD_NT;
      if (d >= DV) continue;
      float v = vnew[k];
      if (d < p.vdim && p.v_store && split == 0) p.v_first[(int64_t)e.row0 * nv + kvhd * p.vdim + d] = v;
      if (p.v_use) v = fmaf(p.lambda, vold[k], (1.f - p.lambda) * v);
      vsn[d] = f2bf(d < p.vdim ? v : 0.f);
    }
  }
  __syncthreads();
  if (split == 0) {   // append for the following steps
    typedef __attribute__((address_space(1))) bf16_t* gbf_t;
    const int t = pos % KV_PAGE_TOKENS;
    const uint64_t base = LEAN ? page_of(63) : (uint64_t)(tab[pos / KV_PAGE_TOKENS] + p.kv.layer_off);
    gbf_t kd = reinterpret_cast<gbf_t>(base) + (int64_t)kvhd * KV_PAGE_TOKENS * DQK;
    gbf_t vd = reinterpret_cast<gbf_t>(base) + (int64_t)p.kvh * KV_PAGE_TOKENS * DQK + (int64_t)kvhd * DV * KV_PAGE_TOKENS;
    for (int i = tid; i < DQK; i += CD_NT) kd[kpage_elem(t, i, KS)] = ksn[i];
    for (int i = tid; i < DV; i += CD_NT) vd[vpage_elem(t, i)] = vsn[i];
  }
  bf16x8_t qf[KS];
#pragma unroll
  for (int k4 = 0; k4 < KS; ++k4) {
    u32x4_t v = *reinterpret_cast<const u32x4_t*>(qs + min(c, g - 1) * DQK + k4 * 32 + G * 8);
    if (c >= g) v = u32x4_t{0u, 0u, 0u, 0u};
    qf[k4] = as_frag(v);
  }
  float m = -INFINITY, l = 0.f;
  if (unit == 0 && a.sink) {
    m = 0.f;
    l = G == 0 ? 1.f : 0.f;
  }
  f32x4_t o[DS];
#pragma unroll
  for (int i = 0; i < DS; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (unit == nunits - 1) {   // the new token, from LDS: this unit's running state begins with it, under its page fetch
    float d4[4] = {0.f, 0.f, 0.f, 0.f};
    const u32x4_t* qr = reinterpret_cast<const u32x4_t*>(qs + min(c, g - 1) * DQK + G * (DQK / 4));
    const u32x4_t* kr = reinterpret_cast<const u32x4_t*>(ksn + G * (DQK / 4));
#pragma unroll
    for (int j = 0; j < DQK / 32; ++j) {
      const u32x4_t qv = qr[j], kv = kr[j];
#pragma unroll
      for (int x = 0; x < 4; ++x) d4[x] = fmaf(hi_bf(qv[x]), hi_bf(kv[x]), fmaf(lo_bf(qv[x]), lo_bf(kv[x]), d4[x]));
    }
    m = group_sum((d4[0] + d4[1]) + (d4[2] + d4[3])) * a.scale;
    l = G == 0 ? 1.f : 0.f;
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) {
      const uint2 v = *reinterpret_cast<const uint2*>(vsn + ds * 16 + G * 4);
      o[ds] = f32x4_t{lo_bf(v.x), hi_bf(v.x), lo_bf(v.y), hi_bf(v.y)};
    }
  }
  int page = unit;
  auto do_page = [&](auto more_tag) {   // MORE: the unit has another page after this one, requested as soon as the registers are free
    constexpr bool MORE = decltype(more_tag)::value;
    uint64_t nb = 0;
    if (MORE) nb = page_base(page + nunits);
    f32x4_t st[4];
#pragma unroll
    for (int sub = 0; sub < 4; ++sub) {
      st[sub] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k4 = 0; k4 < KS; ++k4) st[sub] = mfma16(as_frag(kf[sub][k4]), qf[k4], st[sub]);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (MORE) load_k(nb);
    __builtin_amdgcn_sched_barrier(0);
    float alpha;
    bf16x8_t pf[2];
    const int t0 = (page0 + page) * KV_PAGE_TOKENS;
    softmax_tile(st, a.scale, [&](int t) { return t0 + t >= lo && t0 + t < pos; }, G, m, l, alpha, pf);
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) {
      o[ds] *= alpha;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) o[ds] = mfma16(as_frag(vf[ds][kk]), pf[kk], o[ds]);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (MORE) load_v(nb);
    __builtin_amdgcn_sched_barrier(0);
    page += nunits;
  };
  if (page < npages) {
    while (page + nunits < npages) do_page(std::true_type{});
    do_page(std::false_type{});
  }
  l = group_sum(l);

  // ---- merge the four waves through LDS ---------------------------------------------------------------------------------------------
  {
    float* wo = mo + wave * (DV * 16);
    if (c < g) {
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) *reinterpret_cast<f32x4_t*>(wo + c * DV + ds * 16 + G * 4) = o[ds];
    }
    if (G == 0) {
      mm[wave * 16 + c] = m;
      mlz[wave * 16 + c] = l;
    }
  }
  __syncthreads();
  const bool single = nsplit == 1;
  const int64_t hrow = (int64_t)ent * p.heads;   // output rows of this sequence: (sequence, head)
  bf16_t* out = (bf16_t*)a.o + (hrow + kvhd * g) * DV;
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(a.part_o + (int64_t)ent * nsplit * p.heads * DV, 0, (int)((size_t)nsplit * p.heads * DV * 4), 0x00020000);
  float* ml = a.part_ml + (int64_t)ent * nsplit * p.heads * 2;
  for (int item = tid; item < g * (DV / 4); item += CD_NT) {
    const int q = item / (DV / 4), d0 = (item % (DV / 4)) * 4;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < CD_NW; ++w) M = fmaxf(M, mm[w * 16 + q]);
    float acc[4] = {0.f, 0.f, 0.f, 0.f}, ls = 0.f;
#pragma unroll
    for (int w = 0; w < CD_NW; ++w) {
      const float mw = mm[w * 16 + q];
      const float wt = (mw == -INFINITY) ? 0.f : __expf(mw - M);
      const f32x4_t ow = *reinterpret_cast<const f32x4_t*>(mo + w * (DV * 16) + q * DV + d0);
#pragma unroll
      for (int x = 0; x < 4; ++x) acc[x] = fmaf(wt, ow[x], acc[x]);
      ls = fmaf(wt, mlz[w * 16 + q], ls);
    }
    if (single) {
      const float inv = 1.0f / ls;
      *reinterpret_cast<uint2*>(out + q * DV + d0) = make_uint2(pack_bf(acc[0] * inv, acc[1] * inv), pack_bf(acc[2] * inv, acc[3] * inv));
    } else {
      const int head = kvhd * g + q;
      const u32x4_t v = {__float_as_uint(acc[0]), __float_as_uint(acc[1]), __float_as_uint(acc[2]), __float_as_uint(acc[3])};
      __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, (uint32_t)((split * p.heads + head) * DV + d0) * 4, 0, 16 /* sc1 */);
      if (d0 == 0) {
        const unsigned long long mlp = ((unsigned long long)__float_as_uint(ls) << 32) | __float_as_uint(M);
        __hip_atomic_store(reinterpret_cast<unsigned long long*>(ml + ((int64_t)split * p.heads + head) * 2), mlp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (single) return;
  // write-through stores above: wait for their acknowledgement, then one relaxed atomic per block decides who is last
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    unsigned* ctr = a.ctr + ((int64_t)ent * p.kvh + kvhd) * 32;
    const unsigned prev = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = prev + 1u == (unsigned)nsplit;
    if (s_last) __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // every block of this head has arrived
  }
  __syncthreads();
  if (!s_last) return;
  float* w_lds = mo;             // [g][nsplit] weights, then [g] 1 / sum   (nsplit <= 32, g <= 16)
  float* inv_lds = mo + 16 * CHUNK_DECODE_MAX_SPLIT;
  for (int q = wave; q < g; q += CD_NW) {
    float2 v = make_float2(-INFINITY, 0.f);
    if (lane < nsplit) v = act_ldf2<true>(ml + ((int64_t)lane * p.heads + kvhd * g + q) * 2);
    const float M = wave_max(v.x);
    const float wgt = (v.x == -INFINITY) ? 0.f : __expf(v.x - M);
    const float ls = wave_sum(wgt * v.y);
    if (lane < nsplit) w_lds[q * nsplit + lane] = wgt;
    if (lane == 0) inv_lds[q] = 1.0f / ls;
  }
  __syncthreads();
  for (int item = tid; item < g * (DV / 4); item += CD_NT) {
    const int q = item / (DV / 4), d0 = (item % (DV / 4)) * 4;
    const uint32_t off = (uint32_t)((kvhd * g + q) * DV + d0) * 4, stride = (uint32_t)p.heads * DV * 4;
    f32x4_t f = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < nsplit; s0 += 8) {
      u32x4_t v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off + (uint32_t)min(s0 + j, nsplit - 1) * stride, 0, 16 /* sc1 */);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float wgt = s0 + j < nsplit ? w_lds[q * nsplit + s0 + j] : 0.f;
#pragma unroll
        for (int x = 0; x < 4; ++x) f[x] = fmaf(wgt, __uint_as_float(v[j][x]), f[x]);
      }
    }
    const float inv = inv_lds[q];
    *reinterpret_cast<uint2*>(out + q * DV + d0) = make_uint2(pack_bf(f[0] * inv, f[1] * inv), pack_bf(f[2] * inv, f[3] * inv));
  }
}

// ---- any dims, token-major pages: a block per (row, head) ------------------------------------------------------------------------------
// 64 keys at a time, lane = key for the scores, lanes = value dims for P.V.  What bounds it is the chain load -> score -> softmax -> load -> sum of
// one page: the four waves take the row's pages in turn and join (max, sum, O) in LDS, a lane's key row comes in 16-byte pieces and the values of
// eight keys are requested at once.  (One wave per row with scalar loads: 125 us per launch at 2 x 150 positions of 16 heads x 128 in 32 bits;
// 32 us here.)
constexpr int ROWS_MAX_DV = 1024, ROWS_NW = 4;
template <typename T, int NV>   // vdim <= NV * 64
__global__ __launch_bounds__(ROWS_NW * 64) void attn_chunk_rows_kernel(ChunkAttnArgs a, SeqBatch b) {
  extern __shared__ __attribute__((aligned(16))) float sh[];   // q (dim, padded to 4), then per wave O (NV * 64), max and sum
  typedef const __attribute__((address_space(1))) T* gptr_t;
  typedef T __attribute__((ext_vector_type(4))) t4;
  typedef const __attribute__((address_space(1))) t4* g4_t;
  auto widen = [](T v) {
    if constexpr (std::is_same<T, float>::value) return v;
    else return bf2f(v);
  };
  const int r = blockIdx.x, head = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const SeqEntry e = seq_entry_at(b, b.has_one ? 0 : b.row_entry[r]);
  const int pos = e.pos0 + r - e.row0, lo = a.chunk > 0 ? pos / a.chunk * a.chunk : 0;
  const int kvhd = head / (a.heads / a.kv.kvh), dim4 = (a.dim + 3) & ~3;
  float *os = sh + dim4, *ml = os + ROWS_NW * NV * 64;
  const T* q = (const T*)a.q + ((int64_t)r * a.heads + head) * a.kv.dq;
  for (int d = tid; d < dim4; d += ROWS_NW * 64) sh[d] = d < a.dim ? widen(q[d]) : 0.f;
  __syncthreads();
  const bool vec = ((a.dim | a.kv.dq) & 3) == 0;   // whole aligned groups of four
  float m = a.sink && wave == 0 ? 0.f : -INFINITY, l = a.sink && wave == 0 ? 1.f : 0.f, o[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) o[i] = 0.f;
  for (int pg = lo / KV_PAGE_TOKENS + wave; pg <= pos / KV_PAGE_TOKENS; pg += ROWS_NW) {
    const gptr_t kp = reinterpret_cast<gptr_t>(a.kv.tab[(int64_t)e.slot * a.kv.ld + pg] + a.kv.layer_off);
    const gptr_t vp = kp + (int64_t)a.kv.kvh * KV_PAGE_TOKENS * a.kv.dq + (int64_t)kvhd * KV_PAGE_TOKENS * a.kv.dv;
    const gptr_t kr = kp + ((int64_t)kvhd * KV_PAGE_TOKENS + lane) * a.kv.dq;
    const int t = pg * KV_PAGE_TOKENS + lane;
    float dot;
    if (vec) {
      f32x4_t d4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
      for (int d = 0; d < a.dim; d += 4) {
        const t4 k4 = *reinterpret_cast<g4_t>(kr + d);
        const f32x4_t q4 = *reinterpret_cast<const f32x4_t*>(sh + d);
#pragma unroll
        for (int i = 0; i < 4; ++i) d4[i] = fmaf(q4[i], widen(k4[i]), d4[i]);
      }
      dot = (d4[0] + d4[1]) + (d4[2] + d4[3]);
    } else {
      dot = 0.f;
      for (int d = 0; d < a.dim; ++d) dot = fmaf(sh[d], widen(kr[d]), dot);
    }
    const float s = t >= lo && t <= pos ? dot * a.scale : -INFINITY;
    const float m_new = fmaxf(m, wave_max(s));   // (a visited page holds at least one visible key)
    const float al = m == -INFINITY ? 0.f : expf(m - m_new), p = s == -INFINITY ? 0.f : expf(s - m_new);
    l = l * al + wave_sum(p);
    m = m_new;
#pragma unroll
    for (int i = 0; i < NV; ++i) o[i] *= al;
    const int k0 = max(0, lo - pg * KV_PAGE_TOKENS), k1 = min(KV_PAGE_TOKENS - 1, pos - pg * KV_PAGE_TOKENS);
#pragma unroll 8
    for (int k = k0; k <= k1; ++k) {
      const float pk = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(p), k));
#pragma unroll
      for (int i = 0; i < NV; ++i) o[i] = fmaf(pk, widen(vp[(int64_t)k * a.kv.dv + min(lane + i * 64, a.vdim - 1)]), o[i]);   // (surplus lanes repeat the last dim)
    }
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) os[(wave * NV + i) * 64 + lane] = o[i];
  if (lane == 0) {
    ml[wave] = m;
    ml[ROWS_NW + wave] = l;
  }
  __syncthreads();
  float mx = ml[0], f[ROWS_NW], z = 0.f;
#pragma unroll
  for (int w = 1; w < ROWS_NW; ++w) mx = fmaxf(mx, ml[w]);
#pragma unroll
  for (int w = 0; w < ROWS_NW; ++w) {
    f[w] = ml[w] == -INFINITY ? 0.f : expf(ml[w] - mx);
    z = fmaf(ml[ROWS_NW + w], f[w], z);
  }
  const float inv = 1.0f / z;
  T* op = (T*)a.o + (int64_t)r * a.ldo + (int64_t)head * a.dvo;
  for (int d = tid; d < a.vdim; d += ROWS_NW * 64) {
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < ROWS_NW; ++w) v = fmaf(os[w * NV * 64 + d], f[w], v);
    if constexpr (std::is_same<T, float>::value) op[d] = v * inv;
    else op[d] = f2bf(v * inv);
  }
}

// ---- 32 bits, heads of D = 64 or 128 dims, token-major pages: 16 (row, head) pairs per block -------------------------------------------------
// Block (16 / GQ rows of a sequence, kv head or head, sequence): the GQ query heads of a kv head share its keys and values (GQ = 1 where the group does
// not divide 16).  The eight waves take 16 keys each in turn and join (max, sum, O) in LDS.  Both products on v_mfma_f32_16x16x4_f32: S^T = K Q^T with
// lane (c, G) holding dims 16 t + 4 G + i of key c and of pair c, so both operands come in 16-byte pieces; S^T leaves lane (c, G) with keys 4 G + i of
// pair c, which is the operand layout of O^T = V^T P^T, its k index i running over those keys; V rows come in 16-byte pieces too, lane c taking value dims
// 64 b + 4 c + x, so row 4 G + i of accumulator (b, x) is value dim 64 b + 16 G + 4 i + x.
// What bounds it is a chain of round trips (entry, page, keys) and, for long prompts, the f32 matrix rate.  2 x 150 positions, 16 / 8 heads x 128, before (attn_chunk_rows_kernel: every
// row read its keys and values again) and with it: prompt 96 -> 22 us, one token each 20.7 -> 11.8.
constexpr int F32A_NW = 8;
typedef float fv4 __attribute__((ext_vector_type(4)));
template <int D>
constexpr int f32a_lds() { return F32A_NW * 16 * (D + 2) * 4; }
template <int D>
__global__ __launch_bounds__(F32A_NW * 64) void attn_chunk_f32_kernel(const float* qp, float* op, const uint64_t* tab, int heads_kvh, int gq, SeqBatch b, ChunkAttnArgs a) {
  constexpr int NT16 = D / 16, NB = D / 64;
  extern __shared__ __attribute__((aligned(16))) float os[];   // O [wave][16][D], max [wave][16], sum [wave][16]
  float *mls = os + F32A_NW * 16 * D, *lls = mls + F32A_NW * 16;
  typedef const __attribute__((address_space(1))) fv4* g4_t;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, G = lane >> 4;
  const int heads = heads_kvh >> 16, kvh = heads_kvh & 0xffff;
  const int nrow = 16 / gq, head0 = blockIdx.y * gq, kvhd = gq > 1 ? blockIdx.y : head0 / (heads / kvh);
  const SeqEntry e = seq_entry_at(b, blockIdx.z);
  const int i0 = blockIdx.x * nrow;   // first row inside the entry
  if (i0 >= e.len) return;
  const int ic = min(i0 + c / gq, e.len - 1), pos = e.pos0 + ic, lo = a.chunk > 0 ? pos / a.chunk * a.chunk : 0;   // this lane's pair (c): surplus pairs repeat the last row
  const int p_first = e.pos0 + i0, p_last = e.pos0 + min(i0 + nrow, e.len) - 1, lo_first = a.chunk > 0 ? p_first / a.chunk * a.chunk : 0;
  const float* q = qp + ((int64_t)(e.row0 + ic) * heads + head0 + c % gq) * D + G * 4;
  fv4 qf[NT16];
#pragma unroll
  for (int t = 0; t < NT16; ++t) qf[t] = *reinterpret_cast<const fv4*>(q + t * 16);
  float m = a.sink && wave == 0 ? 0.f : -INFINITY, l = a.sink && wave == 0 ? 1.f : 0.f;
  f32x4_t o[NB][4];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int x = 0; x < 4; ++x) o[i][x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int u = lo_first / 16 + wave; u <= p_last / 16; u += F32A_NW) {   // keys 16 u .. 16 u + 15
    const int k16 = u * 16 % KV_PAGE_TOKENS;
    const uint64_t base = tab[(int64_t)e.slot * a.kv.ld + u * 16 / KV_PAGE_TOKENS] + a.kv.layer_off;
    const uint64_t kb = base + ((uint64_t)kvhd * KV_PAGE_TOKENS + k16 + c) * (D * 4) + G * 16;
    const uint64_t vrow = base + ((uint64_t)(kvh + kvhd) * KV_PAGE_TOKENS + k16) * (D * 4), vb = vrow + G * 4 * (D * 4) + c * 16;
    fv4 kf[NT16], vf[4][NB];
#pragma unroll
    for (int t = 0; t < NT16; ++t) kf[t] = *reinterpret_cast<g4_t>(kb + t * 64);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) vf[i][nb] = *reinterpret_cast<g4_t>(vb + (i * D + nb * 64) * 4);
    __builtin_amdgcn_sched_barrier(0);
    f32x4_t s2[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};   // two chains: a product's result is not waited for by the next
#pragma unroll
    for (int t = 0; t < NT16; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) s2[i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t][i], qf[t][i], s2[i & 1], 0, 0, 0);
    f32x4_t st;
    const int t0 = u * 16 + G * 4;
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      st[i] = t0 + i >= lo && t0 + i <= pos ? (s2[0][i] + s2[1][i]) * a.scale : -INFINITY;
      mx = fmaxf(mx, st[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    const float m_new = fmaxf(m, fmaxf(mx, __shfl_xor(mx, 32, 64)));
    const float al = m == -INFINITY ? 0.f : expf(m - m_new);
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      st[i] = st[i] == -INFINITY ? 0.f : expf(st[i] - m_new);
      ps += st[i];
    }
    l = l * al + group_sum(ps);
    m = m_new;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int x = 0; x < 4; ++x) o[nb][x] *= al;
    // A value is multiplied by the zero weight of a pair that does not see its key.  Where that could leave a NaN (a value that is not finite: behind the
    // sequence's end in a page used before, or a later row's own), the keys go one by one, each to the pairs that see it.
    float bad = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int x = 0; x < 4; ++x) bad = fmaf(vf[i][nb][x], 0.f, bad);
    if (__any(bad != 0.f)) {
#pragma unroll 1
      for (int k = 0; k < 16; ++k) {
        const float w01 = k & 1 ? st[1] : st[0], w23 = k & 1 ? st[3] : st[2];
        const float w = __shfl(k & 2 ? w23 : w01, (k >> 2) * 16 + c, 64);
        if (u * 16 + k < lo || u * 16 + k > pos) continue;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const fv4 v = *reinterpret_cast<g4_t>(vrow + (k * D + nb * 64 + G * 16 + i * 4) * 4);
#pragma unroll
            for (int x = 0; x < 4; ++x) o[nb][x][i] = fmaf(w, v[x], o[nb][x][i]);
          }
      }
      continue;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int x = 0; x < 4; ++x) o[nb][x] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][nb][x], st[i], o[nb][x], 0, 0, 0);
  }
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<fv4*>(os + (wave * 16 + c) * D + nb * 64 + G * 16 + i * 4) = fv4{o[nb][0][i], o[nb][1][i], o[nb][2][i], o[nb][3][i]};
  if (G == 0) {
    mls[wave * 16 + c] = m;
    lls[wave * 16 + c] = l;
  }
  __syncthreads();
  for (int it = threadIdx.x; it < 16 * (D / 4); it += F32A_NW * 64) {
    const int j = it / (D / 4), d = it % (D / 4) * 4, ir = i0 + j / gq;
    if (ir >= e.len) continue;
    float M = mls[j], z = 0.f;
#pragma unroll
    for (int w = 1; w < F32A_NW; ++w) M = fmaxf(M, mls[w * 16 + j]);
    fv4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < F32A_NW; ++w) {
      const float f = mls[w * 16 + j] == -INFINITY ? 0.f : expf(mls[w * 16 + j] - M);
      z = fmaf(lls[w * 16 + j], f, z);
      const fv4 ow = *reinterpret_cast<const fv4*>(os + (w * 16 + j) * D + d);
#pragma unroll
      for (int x = 0; x < 4; ++x) v[x] = fmaf(ow[x], f, v[x]);
    }
    const float inv = 1.0f / z;
    float* dst = op + (int64_t)(e.row0 + ir) * a.ldo + (int64_t)(head0 + j % gq) * a.dvo + d;
#pragma unroll
    for (int x = 0; x < 4; ++x) dst[x] = v[x] * inv;
  }
}

// ---- 32 bits, one token per sequence, heads of D = 64 or 128 dims: q / k norm + rotation + value mixing + KV append + attention, one launch ----------
// Block (kv head, sequence), eight to sixteen waves; wave w takes 16 keys in turn, requested as soon as their page is known and before the
// block redoes the per-token work (sums of squares over the whole q / k projections, its GQ query heads, its key and value).  Lane (c, G) holds dims
// 16 t + 4 G + i of key c and value dims 64 b + 4 c + x of keys 4 G + i, as in attn_chunk_f32_kernel, but the products are plain f32 fma: of the matrix
// cores' sixteen columns a token has GQ, and their f32 rate (256 flops a cycle and CU) leaves nothing over for the rest.  The new token joins from LDS.
// A chain of round trips all the same: 2 x 150 positions, 16 / 8 heads x 128,
// 11.1 us for the 13.6 + 5.0 of attn_chunk_f32_kernel and qkv_post_f32_kernel.
constexpr int f32d_waves(int d, int gq) { return d * gq > 256 ? 8 : d * gq > 128 ? 12 : 16; }   // (the heads' sums and a unit of keys in registers)
constexpr int F32D_COLUMNS = 8192;   // of q and k
template <int D, int GQ>   // GQ: query heads per kv head, at most
constexpr int f32d_lds() {
  constexpr int NW = f32d_waves(D, GQ);
  return (2 * (GQ + 2) * D + NW * GQ * (D + 2 + 16) + GQ + 2 * NW) * 4;
}
template <int D, int GQ>
__global__ __launch_bounds__(f32d_waves(D, GQ) * 64) void attn_chunk_f32_decode_kernel(const float* qkv, const float* bias, const SeqEntry* entries, const uint64_t* tab, int ld, int heads_kvh, int slot, int pos, QkvPostArgs a,
                                                                           ChunkAttnArgs t) {
  constexpr int NW = f32d_waves(D, GQ), NTH = NW * 64, NT16 = D / 16, NB = D / 64, NC = (F32D_COLUMNS + 4 * NTH - 1) / (4 * NTH);
  extern __shared__ __attribute__((aligned(16))) float sm[];
  float *raw = sm, *qs = raw + (GQ + 2) * D, *ks = qs + GQ * D, *vs = ks + D;   // raw: the heads' q, k; then with norm and rotation
  float *os = vs + D, *ml = os + NW * GQ * D, *ll = ml + NW * GQ, *ps = ll + NW * GQ, *fresh = ps + NW * GQ * 16, *red = fresh + GQ;
  typedef const __attribute__((address_space(1))) fv4* g4_t;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, G = lane >> 4;
  const int heads = heads_kvh >> 16, kvh = heads_kvh & 0xffff, g = heads / kvh, kv = blockIdx.x, r = blockIdx.y, head0 = kv * g;
  const int k_off = a.k_off, v_off = a.v_off, rope_dims = a.rope_dims, v_use = a.v_use, v_store = a.v_store, chunk = t.chunk;
  const bf16_t *q_norm = (const bf16_t*)a.q_norm, *k_norm = (const bf16_t*)a.k_norm;
  const float* rope = a.rope;
  float* v_first = a.v_first;
  const int64_t tab_ld = a.kv.ld;
  const uint64_t layer_off = a.kv.layer_off;
  const float lambda = a.lambda, eps = a.eps;
  const int nq = heads * D, nk = kvh * D, half = rope_dims >> 1;
  if (entries) {   // (one sequence: its place comes with the launch)
    typedef const __attribute__((address_space(1))) int32_t* gint_t;
    const gint_t p = (gint_t)(uintptr_t)(entries + r);
    pos = p[2];
    slot = p[3];
  }
  const int lo = chunk > 0 ? pos / chunk * chunk : 0;
  tab += (int64_t)slot * tab_ld;
  // the row
  float4 x[NC], bi[NC];
  const float* row = qkv + (int64_t)r * ld;
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    x[j] = bi[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (j * NTH * 4 >= nq + nk) continue;
    const int i = min((tid + j * NTH) * 4, nq + nk - 4), at = i < nq ? i : i - nq + k_off;
    x[j] = *reinterpret_cast<const float4*>(row + at);
    if (bias) bi[j] = *reinterpret_cast<const float4*>(bias + at);
  }
  // this thread's four value columns; its piece of a head: dims d .. d + 3 with their partners half a rotation further, or four behind the rotated ones
  const bool val = tid >= NTH - D / 4;
  const int vd = (tid - (NTH - D / 4)) * 4, hp = half >> 2, per = (D >> 2) - hp, np = (g + 1) * per;
  float4 xv = make_float4(0.f, 0.f, 0.f, 0.f), bv = xv, first = xv;
  if (val) {
    xv = *reinterpret_cast<const float4*>(row + v_off + kv * D + vd);
    if (bias) bv = *reinterpret_cast<const float4*>(bias + v_off + kv * D + vd);
    if (v_use && !v_store) first = *reinterpret_cast<const float4*>(v_first + ((int64_t)r * kvh + kv) * D + vd);
  }
  const int hd = min(tid, np - 1) / per, pc = min(tid, np - 1) - hd * per, pd = pc < hp ? pc * 4 : rope_dims + (pc - hp) * 4;
  uint2 wx = make_uint2(0u, 0u), wy = wx;
  float4 cs0 = make_float4(1.f, 0.f, 1.f, 0.f), cs1 = cs0;
  if (tid < np) {
    const bf16_t* w = hd < g ? q_norm + (head0 + hd) * D : k_norm + kv * D;
    wx = *reinterpret_cast<const uint2*>(w + pd);
    wy = *reinterpret_cast<const uint2*>(w + (pc < hp ? pd + half : pd));
    if (hp > 0) {
      const float4* at = reinterpret_cast<const float4*>(rope + ((int64_t)r * half + (pc < hp ? pd : 0)) * 2);
      cs0 = at[0];
      cs1 = at[1];
    }
  }
  fv4 kf[NT16], vf[4][NB];
  uint64_t at_k = 0;   // this lane's piece of the unit's first key
  auto request_keys = [&](int u) {   // 16 u .. 16 u + 15
    at_k = tab[u * 16 / KV_PAGE_TOKENS] + layer_off + ((uint64_t)kv * KV_PAGE_TOKENS + u * 16 % KV_PAGE_TOKENS) * (D * 4);
    const uint64_t kb = at_k + c * (D * 4) + G * 16;
#pragma unroll
    for (int i = 0; i < NT16; ++i) kf[i] = *reinterpret_cast<g4_t>(kb + i * 64);
  };
  auto request_values = [&] {   // of the same keys
    const uint64_t vb = at_k + (uint64_t)kvh * KV_PAGE_TOKENS * (D * 4) + G * 4 * (D * 4) + c * 16;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) vf[i][nb] = *reinterpret_cast<g4_t>(vb + (i * D + nb * 64) * 4);
  };
  const int u0 = lo / 16 + wave, last = pos / 16;
  const uint64_t new_page = tab[pos / KV_PAGE_TOKENS] + layer_off;
  request_keys(min(u0, last));   // (waves without keys too: behind a branch nothing requested before is waited for by itself)
  // sums of squares; the heads' own columns to LDS
  float sq = 0.f, sk = 0.f;
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int i = (tid + j * NTH) * 4;
    if (i >= nq + nk) continue;
    const float4 y = make_float4(x[j].x + bi[j].x, x[j].y + bi[j].y, x[j].z + bi[j].z, x[j].w + bi[j].w);
    (i < nq ? sq : sk) += (y.x * y.x + y.y * y.y) + (y.z * y.z + y.w * y.w);
    const int own = i < nq ? i - head0 * D : i - nq - kv * D;
    if (own >= 0 && own < (i < nq ? g * D : D)) *reinterpret_cast<float4*>(raw + (i < nq ? 0 : GQ * D) + own) = y;
  }
  sq = wave_sum(sq);
  sk = wave_sum(sk);
  if (lane == 0) {
    red[wave] = sq;
    red[NW + wave] = sk;
  }
  __syncthreads();
  request_values();
  float tq = 0.f, tk = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    tq += red[w];
    tk += red[NW + w];
  }
  const float rq = 1.0f / sqrtf(tq / (float)nq + eps), rk = 1.0f / sqrtf(tk / (float)nk + eps);
  const int tok = pos % KV_PAGE_TOKENS;
  typedef __attribute__((address_space(1))) fv4* s4_t;
  const uint64_t kpage = new_page + ((uint64_t)kv * KV_PAGE_TOKENS + tok) * (D * 4), vpage = kpage + (uint64_t)kvh * KV_PAGE_TOKENS * (D * 4);
  if (tid < np) {
    const float rinv = hd < g ? rq : rk;
    float* dst = hd < g ? qs + hd * D : ks;
    const float* src = raw + (hd < g ? hd : GQ) * D;
    const float4 s4 = *reinterpret_cast<const float4*>(src + pd);
    const float4 y0 = make_float4(s4.x * rinv * lo_bf(wx.x), s4.y * rinv * hi_bf(wx.x), s4.z * rinv * lo_bf(wx.y), s4.w * rinv * hi_bf(wx.y));
    float4 out0 = y0, out1 = y0;
    if (pc < hp) {
      const float4 t4 = *reinterpret_cast<const float4*>(src + pd + half);
      const float4 y1 = make_float4(t4.x * rinv * lo_bf(wy.x), t4.y * rinv * hi_bf(wy.x), t4.z * rinv * lo_bf(wy.y), t4.w * rinv * hi_bf(wy.y));
      out0 = make_float4(y0.x * cs0.x - y1.x * cs0.y, y0.y * cs0.z - y1.y * cs0.w, y0.z * cs1.x - y1.z * cs1.y, y0.w * cs1.z - y1.w * cs1.w);
      out1 = make_float4(y1.x * cs0.x + y0.x * cs0.y, y1.y * cs0.z + y0.y * cs0.w, y1.z * cs1.x + y0.z * cs1.y, y1.w * cs1.z + y0.w * cs1.w);
    }
    const int pd1 = pc < hp ? pd + half : pd;
    *reinterpret_cast<float4*>(dst + pd) = out0;
    *reinterpret_cast<float4*>(dst + pd1) = out1;
    if (hd == g) {
      *reinterpret_cast<s4_t>(kpage + pd * 4) = fv4{out0.x, out0.y, out0.z, out0.w};
      *reinterpret_cast<s4_t>(kpage + pd1 * 4) = fv4{out1.x, out1.y, out1.z, out1.w};
    }
  }
  if (val) {
    const float4 y = make_float4(xv.x + bv.x, xv.y + bv.y, xv.z + bv.z, xv.w + bv.w);
    if (v_store) *reinterpret_cast<float4*>(v_first + ((int64_t)r * kvh + kv) * D + vd) = y;
    const float4 f = v_store ? y : first;   // (stored and used at once: the value itself)
    const float k0 = 1.f - lambda, k1 = lambda;
    const float4 o = v_use ? make_float4(k0 * y.x + k1 * f.x, k0 * y.y + k1 * f.y, k0 * y.z + k1 * f.z, k0 * y.w + k1 * f.w) : y;
    *reinterpret_cast<float4*>(vs + vd) = o;
    *reinterpret_cast<s4_t>(vpage + vd * 4) = fv4{o.x, o.y, o.z, o.w};
  }
  __syncthreads();
  if (wave < g) {   // the new token's score for head `wave`
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NB; ++i) s = fmaf(qs[wave * D + i * 64 + lane], ks[i * 64 + lane], s);
    s = wave_sum(s) * t.scale;
    if (lane == 0) fresh[wave] = s;
  }
  float m[GQ], l[GQ];
  f32x4_t o[GQ][NB];
#pragma unroll
  for (int h = 0; h < GQ; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) o[h][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  for (int u = u0; u <= last; u += NW) {
    const bool key = u * 16 + c >= lo && u * 16 + c < pos;
#pragma unroll
    for (int h = 0; h < GQ; ++h) {
      if (h >= g) continue;
      float s2[2] = {0.f, 0.f};
#pragma unroll
      for (int i = 0; i < NT16; ++i) {
        const fv4 q = *reinterpret_cast<const fv4*>(qs + h * D + i * 16 + G * 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) s2[j & 1] = fmaf(kf[i][j], q[j], s2[j & 1]);
      }
      const float s = key ? rows_sum(s2[0] + s2[1]) * t.scale : -INFINITY;
      const float mn = fmaxf(m[h], row_max(s)), from = mn == -INFINITY ? 0.f : mn;   // (nothing of this unit or before is visible)
      const float al = expf(m[h] - from), p = expf(s - from);
      l[h] = l[h] * al + p;
      m[h] = mn;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) o[h][nb] *= al;
      ps[(wave * GQ + h) * 16 + c] = p;   // (the four lanes of one key: the same)
    }
    // a value whose key is not visible may be anything: it must not meet its zero weight
    const int k0 = u * 16 + G * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int j = 0; j < 4; ++j) vf[i][nb][j] = k0 + i >= lo && k0 + i < pos ? vf[i][nb][j] : 0.f;
#pragma unroll
    for (int h = 0; h < GQ; ++h) {
      if (h >= g) continue;
      const fv4 p = *reinterpret_cast<const fv4*>(ps + (wave * GQ + h) * 16 + G * 4);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[h][nb][j] = fmaf(p[i], vf[i][nb][j], o[h][nb][j]);
    }
    if (u + NW <= last) {
      request_keys(u + NW);
      request_values();
    }
  }
#pragma unroll
  for (int h = 0; h < GQ; ++h) {
    if (h >= g) continue;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      f32x4_t v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = rows_sum(o[h][nb][j]);
      if (G == 0) *reinterpret_cast<f32x4_t*>(os + (wave * GQ + h) * D + nb * 64 + c * 4) = v;
    }
    const float z = row_sum(l[h]);
    if (lane == 0) {
      ml[wave * GQ + h] = m[h];
      ll[wave * GQ + h] = z;
    }
  }
  __syncthreads();
  if (wave == 0 && G < g) {   // sixteen lanes a head: the waves' factors, then the new token's and 1 / sum
    const float mine = fresh[G], mw = c < NW ? ml[c * GQ + G] : -INFINITY, M = fmaxf(t.sink ? fmaxf(mine, 0.f) : mine, row_max(mw));
    const float f = expf(mw - M), f0 = expf(mine - M), z = row_sum(c < NW ? ll[c * GQ + G] * f : 0.f) + f0 + (t.sink ? expf(-M) : 0.f);
    ps[G * 20 + c] = f;
    if (c == 0) {
      ps[G * 20 + 16] = f0;
      ps[G * 20 + 17] = 1.0f / z;
    }
  }
  __syncthreads();
  for (int it = tid; it < g * D; it += NTH) {
    const int h = it / D, d = it - h * D;
    float v = ps[h * 20 + 16] * vs[d];
#pragma unroll
    for (int w = 0; w < NW; ++w) v = fmaf(os[(w * GQ + h) * D + d], ps[h * 20 + w], v);
    ((float*)t.o)[(int64_t)r * t.ldo + (int64_t)(head0 + h) * t.dvo + d] = v * ps[h * 20 + 17];
  }
}

int pad_dim(int d) { return d <= 32 ? 32 : d <= 64 ? 64 : d <= 128 ? 128 : d <= 256 ? 256 : 0; }

template <class F>
void dispatch_dims(int dq, int dv, F&& f) {
  auto inner = [&](auto q) {
    if (dv == 32) f(q, std::integral_constant<int, 32>{});
    else if (dv == 64) f(q, std::integral_constant<int, 64>{});
    else if (dv == 128) f(q, std::integral_constant<int, 128>{});
    else f(q, std::integral_constant<int, 256>{});
  };
  if (dq == 32) inner(std::integral_constant<int, 32>{});
  else if (dq == 64) inner(std::integral_constant<int, 64>{});
  else if (dq == 128) inner(std::integral_constant<int, 128>{});
  else inner(std::integral_constant<int, 256>{});
}

template <int DQK, int DV>
void launch_seqs(AttnPrefillArgs a, int n, int max_len, hipStream_t st) {
  const int nwv = (int64_t)((max_len + 127) / 128) * a.nh * n >= 512 ? 8 : 4;
  const int nqb = (max_len + 16 * nwv - 1) / (16 * nwv);
  const bool xcd_order = a.kvh % 8 == 0;
  a.nqb = xcd_order ? nqb : 0;
  const dim3 grid = xcd_order ? dim3((unsigned)(nqb * a.nh), (unsigned)n) : dim3((unsigned)nqb, (unsigned)n, (unsigned)a.nh), block(nwv * 64);
  const size_t stage = (size_t)2 * KV_PAGE_TOKENS * 2 * (DQK + DV), epi = a.epi_rows ? (size_t)nwv * 16 * (DV * 2 + 16) : 0;
  const size_t lds = std::max(stage, epi);
  auto go = [&](auto nw) {
    constexpr int NW = decltype(nw)::value;
    auto k = attn_prefill_kernel<DQK, DV, 1, NW, false, 0, 3, 1>;
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(k, grid, block, lds, st, a, nullptr);
  };
  if (nwv == 8) go(std::integral_constant<int, 8>{});
  else go(std::integral_constant<int, 4>{});
}

}  // namespace

bool chunk_attn_dims_ok(int dim, int vdim, int* dq, int* dv) {
  *dq = pad_dim(dim);
  *dv = pad_dim(vdim);
  return *dq > 0 && *dv > 0;
}

void launch_chunk_attn_prefill(const ChunkAttnArgs& c, const SeqBatch& b, hipStream_t st) {
  if (b.rows <= 0) return;
  AttnPrefillArgs a{};
  a.q = c.q;
  a.o = c.o;
  a.kv.page_ptrs = c.kv.tab; a.kv.layer_off = c.kv.layer_off; a.kv.kvh = c.kv.kvh; a.kv.d = c.kv.dq;
  a.S = b.max_len; a.nh = c.heads; a.kvh = c.kv.kvh; a.d = c.dvo;
  a.causal = 1;
  a.scale = c.scale;
  a.seqs = b.entries; a.seq_tab_ld = c.kv.ld; a.chunk = c.chunk; a.sink = c.sink;
  a.epi_rows = a.d % 8 == 0 && a.d <= 128 && ((uintptr_t)a.o & 15) == 0;
  dispatch_dims(c.kv.dq, c.kv.dv, [&](auto q, auto v) { launch_seqs<decltype(q)::value, decltype(v)::value>(a, b.n, b.max_len, st); });
}

// the Qwen3 stack's head dims, q heads raw or rotated (AttnPrefillArgs::q_norm_w)
void launch_attn_prefill_seqs(const AttnPrefillArgs& a_in, int n, int max_len, hipStream_t st) {
  if (n <= 0) return;
  AttnPrefillArgs a = a_in;
  a.epi_rows = ((uintptr_t)a.o & 15) == 0;
  launch_seqs<128, 128>(a, n, max_len, st);
}

void launch_chunk_attn_decode(const ChunkDecodeArgs& a, const SeqBatch& b, hipStream_t st) {
  if (b.n <= 0) return;
  const dim3 grid((unsigned)a.nsplit, (unsigned)a.p.kvh, (unsigned)b.n), block(CD_NT);
  dispatch_dims(a.p.kv.dq, a.p.kv.dv, [&](auto q, auto v) {
    constexpr int DQK = decltype(q)::value, DV = decltype(v)::value;
    const size_t lds = chunk_decode_lds<DQK, DV>();
    auto go = [&](auto k) {
      if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      hipLaunchKernelGGL(k, grid, block, lds, st, a.p.qkv, a.p.bias, a.p.q_norm, a.p.k_norm, b.entries, a.p.kv.tab, (int)a.p.ld,
                         (int)((unsigned)(a.p.heads / a.p.kvh) << 20 | (unsigned)a.p.kvh << 8 | (unsigned)a.nsplit), a, b);
    };
    if constexpr (DQK == 128 && DV == 128) {
      const QkvPostArgs& p = a.p;
      const int nq = p.heads * 128, nk = p.kvh * 128;
      const bool lean = p.dim == 128 && p.vdim == 128 && p.rope_dims == 128 && p.k_off == nq && p.v_off == nq + nk && nq <= 4096 && nk <= 2048 && p.heads % p.kvh == 0 && p.heads / p.kvh <= 7 &&
                        p.ld % 8 == 0 && (((uintptr_t)p.qkv | (uintptr_t)p.bias) & 15) == 0 && b.max_len == 1;
      if (lean) {
        if (a.qkv_f32) p.bias ? go(attn_chunk_decode_kernel<DQK, DV, float, true, true>) : go(attn_chunk_decode_kernel<DQK, DV, float, true, false>);
        else p.bias ? go(attn_chunk_decode_kernel<DQK, DV, bf16_t, true, true>) : go(attn_chunk_decode_kernel<DQK, DV, bf16_t, true, false>);
        return;
      }
    }
    if (a.qkv_f32) go(attn_chunk_decode_kernel<DQK, DV, float>);
    else go(attn_chunk_decode_kernel<DQK, DV, bf16_t>);
  });
}

// Row i of the step is sequence i's only one; whole heads of 64 or 128 dims whose columns come in fours, up to four query heads per kv head and 8192 columns
// of q and k
bool chunk_attn_f32_decode_ok(const QkvPostArgs& a, const ChunkAttnArgs& t, const SeqBatch& b) {
  return b.max_len == 1 && b.rows == b.n && a.dim == a.vdim && (a.dim == 64 || a.dim == 128) && a.kv.dq == a.dim && a.kv.dv == a.dim && !a.kv.frag && a.heads % a.kvh == 0 && a.heads / a.kvh <= 4 &&
         a.heads < 32768 && (a.heads + a.kvh) * a.dim <= F32D_COLUMNS && ((a.k_off | a.v_off) & 3) == 0 && (a.ld & 3) == 0 && a.ld < (1 << 30) && a.rope_dims % 8 == 0 &&
         (((uintptr_t)a.qkv | (uintptr_t)a.bias | (uintptr_t)a.rope | (uintptr_t)a.q_norm | (uintptr_t)a.k_norm | (uintptr_t)a.v_first) & 15) == 0 && t.heads == a.heads && t.dim == a.dim;
}

void launch_chunk_attn_f32_decode(const QkvPostArgs& a, const ChunkAttnArgs& t, const SeqBatch& b, hipStream_t st) {
  if (b.n <= 0) return;
  auto go = [&](auto d, auto gq) {
    constexpr int D = decltype(d)::value, GQ = decltype(gq)::value, lds = f32d_lds<D, GQ>();
    auto k = attn_chunk_f32_decode_kernel<D, GQ>;
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    hipLaunchKernelGGL(k, dim3((unsigned)a.kvh, (unsigned)b.n), dim3(f32d_waves(D, GQ) * 64), lds, st, (const float*)a.qkv, a.bias, b.has_one ? nullptr : b.entries, a.kv.tab, (int)a.ld, a.heads << 16 | a.kvh, b.one.slot, b.one.pos0, a, t);
  };
  auto by_group = [&](auto d) {
    const int g = a.heads / a.kvh;
    if (g == 1) go(d, std::integral_constant<int, 1>{});
    else if (g == 2) go(d, std::integral_constant<int, 2>{});
    else go(d, std::integral_constant<int, 4>{});
  };
  if (a.dim == 128) by_group(std::integral_constant<int, 128>{});
  else by_group(std::integral_constant<int, 64>{});
}

void launch_chunk_attn_rows(const ChunkAttnArgs& a, const SeqBatch& b, bool f32, hipStream_t st) {
  if (b.rows <= 0) return;
  // (16-byte requests of q and of the pages' rows: whole heads of D dims lie so)
  if (f32 && a.dim == a.vdim && a.kv.dq == a.dim && a.kv.dv == a.dim && (a.dim == 64 || a.dim == 128) && ((uintptr_t)a.q & 15) == 0 && a.heads < 32768) {
    const int g = a.heads / a.kv.kvh, gq = g <= 16 && 16 % g == 0 ? g : 1, nrow = 16 / gq;
    const dim3 grid((unsigned)((b.max_len + nrow - 1) / nrow), (unsigned)(a.heads / gq), (unsigned)b.n), block(F32A_NW * 64);
    auto k = a.dim == 128 ? attn_chunk_f32_kernel<128> : attn_chunk_f32_kernel<64>;
    const int lds = a.dim == 128 ? f32a_lds<128>() : f32a_lds<64>();
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    hipLaunchKernelGGL(k, grid, block, lds, st, (const float*)a.q, (float*)a.o, a.kv.tab, a.heads << 16 | a.kv.kvh, gq, b, a);
    return;
  }
  auto go = [&](auto t, auto nv) {
    using T = decltype(t);
    constexpr int NV = decltype(nv)::value;
    const size_t lds = (size_t)(((a.dim + 3) & ~3) + ROWS_NW * NV * 64 + 2 * ROWS_NW) * 4;
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(attn_chunk_rows_kernel<T, NV>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL((attn_chunk_rows_kernel<T, NV>), dim3((unsigned)b.rows, (unsigned)a.heads), dim3(ROWS_NW * 64), lds, st, a, b);
  };
  auto dims = [&](auto t) {
    using std::integral_constant;
    if (a.vdim <= 64) go(t, integral_constant<int, 1>{});
    else if (a.vdim <= 128) go(t, integral_constant<int, 2>{});
    else if (a.vdim <= 256) go(t, integral_constant<int, 4>{});
    else go(t, integral_constant<int, ROWS_MAX_DV / 64>{});
  };
  if (f32) dims(float{});
  else dims(bf16_t{});
}

}  // namespace aha
