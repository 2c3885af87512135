// GQA attention over the paged KV cache: flash-style, no S x S score tensor, no repeat_kv
// copies, no mask tensor.  Reference semantics being reproduced (eager_attention_forward,
// /root/reference/src/models/common/modules.rs:757-813; repeat_kv /root/reference/src/utils/tensor_utils.rs:108-124;
// causal mask tensor_utils.rs:78-106):
//     scores = bf16(q . k^T) ; scores = bf16(scores * scale) ; (+ -inf above the diagonal) ; softmax ; P . v ; -> bf16
// q head i reads kv head i / g.  Softmax runs online in f32; P feeds the MFMA as bf16.  The two bf16 roundings of the scores are what
// the prefill kernel's score chains 0 / 1 reproduce (the bit-faithful forms, opt-in); the default chain of the prefill kernels since
// round 5 (SMX 3) and of the decode kernels since round 6 keeps the scores in f32 through scale, mask, maximum and exponential
// (attn_common.h; DESIGN.md section 2, deviation (iii)): one convention for a cache position, however it arrived.
//
// Fragment scheme (v_mfma_f32_16x16x32_bf16, wave64; G = lane>>4, c = lane&15):
//   S^T tile = K . Q^T :  A = K   (row = token c, k = dims G*8..+8  -> 16 B piece `lane` of a fragment-major K fragment)
//                         B = Q^T (col = q row c, k = dims G*8..+8  -> 16 B straight from a q row)
//                         C[reg] = S[token G*4+reg][q c]            -> softmax statistics are per lane column
//   O^T tile = V^T . P^T: A = V^T (row = dim c,  k = 8 token slots  -> 16 B piece `lane` of a fragment-major V fragment)
//                         B = P^T (col = q c,    k = the two S^T fragments of token sub-tiles 2kk, 2kk+1, in registers)
//                         C[reg] = O[q c][dim G*4+reg]
// so no operand ever needs a transpose or a cross-lane shuffle; page layout and the V slot permutation: common.h.
#include <algorithm>

#include <stdio.h>
#include <stdlib.h>

#include "attn_decode_body.h"
#include "oproj_slices.h"
#include "attn_prefill_body.h"

namespace aha {

namespace {

// ---- decode: one wave = one work unit striding over KV pages; K / V^T fragments straight from HBM --------------
// grid (kvh, nsplit), 4 waves per block => 4*nsplit units per kv head; unit u takes pages u, u + nunits, ...
// All g = nh/kvh q heads of the kv head ride along as MFMA columns, so every KV byte is read exactly once.
__global__ __launch_bounds__(256) void attn_decode_kernel(AttnDecodeArgs a) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, G = lane >> 4, c = lane & 15;
  const int kvhd = blockIdx.x;
  const int g = a.nh / a.kvh;
  const int nunits = gridDim.y * 4;
  const int unit = blockIdx.y * 4 + wave;
  const int L = *a.kv_len;
  const int npages = (L + KV_PAGE_TOKENS - 1) / KV_PAGE_TOKENS;

  bf16x8_t qf[4];
  {
    const bf16_t* qp = (const bf16_t*)a.q + (int64_t)(kvhd * g + min(c, g - 1)) * 128;
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4) {
      u32x4_t v = ld16(qp + k4 * 32 + G * 8);
      if (c >= g) v = u32x4_t{0u, 0u, 0u, 0u};
      qf[k4] = as_frag(v);
    }
  }
  float m = -INFINITY, l = 0.f;
  f32x4_t o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  for (int page = unit; page < npages; page += nunits) {
    const char* base = reinterpret_cast<const char*>(a.kv.page_ptrs[page] + a.kv.layer_off);
    const char* kb = base + (size_t)kvhd * KV_PAGE_TOKENS * 256;
    const char* vb = base + (size_t)a.kvh * KV_PAGE_TOKENS * 256 + (size_t)kvhd * 128 * (KV_PAGE_TOKENS * 2);
    u32x4_t kf[4][4], vf[8][2];
#pragma unroll
    for (int sub = 0; sub < 4; ++sub)
#pragma unroll
      for (int k4 = 0; k4 < 4; ++k4) kf[sub][k4] = ld_nt16(kb + ((sub * 4 + k4) * 64 + lane) * 16);   // fragment-major pages
#pragma unroll
    for (int ds = 0; ds < 8; ++ds)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) vf[ds][kk] = ld_nt16(vb + ((ds * 2 + kk) * 64 + lane) * 16);

    f32x4_t st[4];
#pragma unroll
    for (int sub = 0; sub < 4; ++sub) {
      st[sub] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k4 = 0; k4 < 4; ++k4) st[sub] = mfma16(as_frag(kf[sub][k4]), qf[k4], st[sub]);
    }
    float alpha;
    bf16x8_t pf[2];
    const int t0 = page * KV_PAGE_TOKENS;
    softmax_tile(st, a.scale, [&](int t) { return t0 + t < L; }, G, m, l, alpha, pf);
#pragma unroll
    for (int ds = 0; ds < 8; ++ds) {
      o[ds] *= alpha;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) o[ds] = mfma16(as_frag(vf[ds][kk]), pf[kk], o[ds]);
    }
  }
  l = group_sum(l);
  if (c < g) {
    const int head = kvhd * g + c;
    float* po = a.part_o + ((int64_t)unit * a.nh + head) * 128;
#pragma unroll
    for (int ds = 0; ds < 8; ++ds)
      *reinterpret_cast<float4*>(po + ds * 16 + G * 4) = make_float4(o[ds][0], o[ds][1], o[ds][2], o[ds][3]);
    if (G == 0) {
      a.part_ml[((int64_t)unit * a.nh + head) * 2 + 0] = m;
      a.part_ml[((int64_t)unit * a.nh + head) * 2 + 1] = l;
    }
  }
}

// merge the per-unit partials: o = sum_u e^{m_u - M} o_u / sum_u e^{m_u - M} l_u  -> bf16 (the P.V matmul output tensor)
// One block per head; nunits <= 256.  The per-unit weights e^{m_u - M} are computed once (one unit per thread) and
// shared through LDS; the weighted sum over units then runs 8 independent loads deep per thread.
__global__ __launch_bounds__(128) void attn_decode_combine_kernel(AttnDecodeArgs a, int nunits) {
  __shared__ float sw[256];
  __shared__ float red[4];
  const int head = blockIdx.x, d = threadIdx.x, lane = d & 63, wave = d >> 6;
  float mu[2], lu[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int u = d + i * 128;
    mu[i] = -INFINITY;
    lu[i] = 0.f;
    if (u < nunits) {
      const float2 ml = *reinterpret_cast<const float2*>(a.part_ml + ((int64_t)u * a.nh + head) * 2);
      mu[i] = ml.x;
      lu[i] = ml.y;
    }
  }
  float M = wave_max(fmaxf(mu[0], mu[1]));
  if (lane == 0) red[wave] = M;
  __syncthreads();
  M = fmaxf(red[0], red[1]);
  float lsum = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float w = (mu[i] == -INFINITY) ? 0.f : __expf(mu[i] - M);
    sw[d + i * 128] = w;
    lsum += w * lu[i];
  }
  lsum = wave_sum(lsum);
  if (lane == 0) red[2 + wave] = lsum;
  __syncthreads();
  lsum = red[2] + red[3];
  const float* po = a.part_o + (int64_t)head * 128 + d;
  const int64_t ustride = (int64_t)a.nh * 128;
  float acc = 0.f;
  int u = 0;
  for (; u + 8 <= nunits; u += 8) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = po[(u + j) * ustride];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc += sw[u + j] * v[j];
  }
  for (; u < nunits; ++u) acc += sw[u] * po[u * ustride];
  ((bf16_t*)a.o)[head * 128 + d] = f2bf(acc / lsum);
}

__global__ __launch_bounds__(256, 2) void attn_decode_fused_kernel(AttnDecodeFusedArgs a) {
  __shared__ __attribute__((aligned(16))) char smem[ATTN_DECODE_FUSED_LDS];
  attn_decode_fused_body<ATTN_DECODE_NW, false>(a, smem, (int)blockIdx.x, (int)blockIdx.y, (int)gridDim.y);
}
__global__ __launch_bounds__(256, 2) void attn_decode_defer_kernel(const void* qkv, const void* q_norm_w, const void* k_norm_w, const float* rope, const uint64_t* page_ptrs, int kv_len,
                                                                       int heads, int nsplit, unsigned page_stride, AttnDecodeFusedArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem_defer[];
  // (what the first requests need: in scalar registers at the start, gemv_body.h)
  a.qkv = qkv;
  a.q_norm_w = q_norm_w;
  a.k_norm_w = k_norm_w;
  a.rope = rope;
  a.kv.page_ptrs = page_ptrs;
  a.kv_len_v = kv_len;
  a.page_stride = page_stride;
  a.group = heads & 0x7fff;
  a.kvh = heads >> 16;
  a.nh = a.group * a.kvh;
  a.traced = heads >> 15 & 1;
  attn_decode_fused_body<ATTN_DECODE_NW, true>(a, smem_defer, (int)blockIdx.x, (int)blockIdx.y, nsplit);
}

// Short contexts: attention of one kv head (two query heads: 256 columns of W_o) and its share of 32 rows of o_proj, left as f32 for the next norm to add up.
// The 32 blocks of a kv head, all on one XCD, each do its attention: up to six pages that costs less than the launch of its own that o_proj
// takes elsewhere (attn_decode_slice_splits).  W_o's rows are requested behind the pages and arrive under the attention.  (Two kv heads and 16 rows per block of eight waves, half as
// many slices for the norm: 7.3 us + 4.3 of gate + up, here 5.4 + 5.2; attention, o_proj and gate + up in launches of their own 4.8 + 2.9 + 4.4; 19 positions.)
__global__ __launch_bounds__(256, 2) void attn_oproj_kernel(const void* qkv, const void* q_norm_w, const void* k_norm_w, const float* rope, const uint64_t* page_ptrs, const void* W,
                                                            int kvh_len, unsigned page_stride, AttnDecodeFusedArgs a, float* y, int n) {
  extern __shared__ __attribute__((aligned(16))) char smem_defer[];
  // (what the first requests need: in scalar registers at the start, gemv_body.h)
  a.qkv = qkv;
  a.q_norm_w = q_norm_w;
  a.k_norm_w = k_norm_w;
  a.rope = rope;
  a.kv.page_ptrs = page_ptrs;
  const int kvh = kvh_len >> 21;
  a.kv_len_v = kvh_len & 0xfffff;
  a.page_stride = page_stride;
  a.group = 2;
  a.kvh = kvh;
  a.nh = 2 * kvh;
  float* o = reinterpret_cast<float*>(smem_defer);
  const int kvhd = (int)blockIdx.x, slab = (int)blockIdx.y;
  a.traced = (kvh_len >> 20 & 1) && slab == 0;
  OprojRows<4, 256> rows;
  const int row0 = rows.row0(slab, ATTN_DECODE_NW);
  attn_decode_fused_body<ATTN_DECODE_NW, true, true>(a, smem_defer + 256 * 4, kvhd, 0, 1, o, slab == 0, [&] { rows.request((const bf16_t*)W, 256 * kvh, kvhd, row0); });
  __syncthreads();
  rows.multiply(o, y + kvhd * n, row0);
}

}  // namespace

void launch_attn_oproj(const AttnDecodeFusedArgs& a, const void* W, float* y, int n, hipStream_t st) {
  hipLaunchKernelGGL(attn_oproj_kernel, dim3(a.kvh, n / 32), dim3(256), 256 * 4 + ATTN_DEFER_LDS(2), st, a.qkv, a.q_norm_w, a.k_norm_w, a.rope, a.kv.page_ptrs, W,
                     a.kvh << 21 | (a.trace != nullptr) << 20 | a.kv_len_v, a.page_stride, a, y, n);
}

void launch_attn_decode_fused(const AttnDecodeFusedArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(attn_decode_fused_kernel, dim3(a.kvh, a.nsplit), dim3(256), 0, st, a);
}

// How many partials (0: the merge belongs inside the launch).  A CU streams ~56 bytes per ns here, half a microsecond per page of a kv head, so two
// pages per block while the partials last; every partial costs the o_proj matvec another 4 bytes per column and block from L2 (0.6B widths: +0.2 us
// for 4, +0.6 us for 8; 8B widths: +2.1 us for 4, so nothing is split there before a block has more than four pages).
// At six pages per block the launch that merges by itself is as fast.  Attention + o_proj before (merge by the last block) and with the deferred merge:
// 14.5 -> 10.5 us at 450 positions and 14.9 -> 13.7 at 2200 of 0.6B, 18.6 -> 18.0 at 900 of 8B; with the new token and the waves' sums as they are now
// (attn_decode_body.h) another 0.9 less.
int attn_decode_defer_splits(int npages, int nq) {
  if (nq > 4096) return 0;   // (the prologue holds the partials of 4096 columns in registers)
  const int most = nq <= 2048 ? 8 : 4;
  if (npages > 6 * most) return 0;
  return nq > 2048 && npages <= 4 ? 1 : std::min((npages + 1) / 2, most);
}
// 0.6B, us per token, merged by gemv_row_merge_kernel (beyond 48 pages inside the launch) / in slices: 20 positions 561 / 518, 200: 569 / 550, 300: 575 / 564, 400 (seven
// pages: every block of attn_oproj_kernel streams them all) 576 / 575, 470: 577 / 591; with splits of their own 470: 577 / 594, 900: 593 / 594, 1200: 602 / 596,
// 2000: 619 / 602, 4000: 713 / 625, 12000: 896 / 783.  In between the slices' extra bytes in front of gate + up cost what the merge saves.  (A unit has at most three
// pages, attn_decode_body.h: 192.)
int attn_decode_slice_splits(int npages) { return npages <= 6 ? -1 : npages <= 16 || npages > 192 ? 0 : std::min((npages + 1) / 2, 16); }
void launch_attn_decode_defer(const AttnDecodeFusedArgs& a, hipStream_t st) {
  const int lds = ATTN_DEFER_LDS(a.nh / a.kvh);
  hipLaunchKernelGGL(attn_decode_defer_kernel, dim3(a.kvh, a.nsplit), dim3(256), lds, st, a.qkv, a.q_norm_w, a.k_norm_w, a.rope, a.kv.page_ptrs, a.kv_len_v,
                     a.kvh << 16 | (a.trace != nullptr) << 15 | a.nh / a.kvh, a.nsplit, a.page_stride, a);
}

static int g_attn_smx_override = -1;
void set_attn_variant_override(int smx) { g_attn_smx_override = smx; }
static int g_attn_form_override = -1;
void set_attn_form_override(int form) { g_attn_form_override = form; }

// The kernel form launch_attn_prefill picks for these arguments: 0 = this file's 16-rows-per-wave kernel, 64 / 65 = kernels_attn64.hip
static int attn_prefill_form(const AttnPrefillArgs& a, int smx);
static int attn_prefill_smx(const AttnPrefillArgs& a);
static int attn_form_asked() {   // set_attn_form_override, else AHA_ATTN_FORM; -1 = automatic
  static const int form_env = [] { const char* e = getenv("AHA_ATTN_FORM"); return e ? atoi(e) : -1; }();
  return g_attn_form_override >= 0 ? g_attn_form_override : form_env;
}
static int attn_prefill_smx(const AttnPrefillArgs& a) {
  static const int smx_env = [] { const char* e = getenv("AHA_ATTN_SMX"); return e ? atoi(e) : 3; }();
  union { float f; uint32_t u; } sb;
  sb.f = a.scale;
  const uint32_t scale_bits = sb.u;
  int smx = g_attn_smx_override >= 0 ? g_attn_smx_override : smx_env;
  if (smx == 1 && (scale_bits & 0xffffu) != 0) smx = 0;
  if (smx == 3 && !(a.scale > 0.f)) smx = 0;   // the f32 chain keeps its running maximum in raw score units: needs a positive scale
  return smx;
}
static int attn_prefill_form(const AttnPrefillArgs& a, int smx) {
  // The kernel form.  AHA_ATTN_FORM / set_attn_form_override: 16 = this file's 16-rows-per-wave kernel, 64 = the one-wave-per-SIMD kernel
  // with 64 rows per wave (kernels_attn64.hip) with a tile's parts in program order, 65 = the same software-pipelined inside the wave;
  // unset = automatic: form 65 (f32 chain only) once its 256-row blocks fill the chip.
  const int form = attn_form_asked();
  if (smx != 3 || form == 16) return 0;
  const int64_t blocks64 = (a.rows_hint > 0 ? (int64_t)(a.rows_hint + 255) / 256 : (int64_t)((a.S + 255) / 256 + (a.S2 + 255) / 256)) * a.nh;
  // One 4-wave workgroup per CU: a full launch is rounds of 256 workgroups.  Same-box A/B against the 16-row kernel (scripts/attn64_ab.py,
  // 32 heads x head_dim 128, profiles/r06_attn_prefill.md): full attention 2048 / 3072 / 4096 / 8192 rows = 1 / 1.5 / 2 / 4 rounds:
  // 64 vs 75, 165 vs 160, 234 vs 273, 959 vs 1143 us -- ahead wherever the last round is at least ~80 % full; causal (long blocks first, the
  // rounds blur): 62 vs 55 us at 2048 rows, 95 vs 98 at 3072, 139 vs 154 at 4096, 0.51 vs 0.58 ms at 8192, 11.7 vs 13.5 ms at 40 980.
  const int64_t rounds64 = (blocks64 + 255) / 256;
  const bool fills = a.causal ? blocks64 >= 384 : (blocks64 >= 256 && blocks64 * 5 >= rounds64 * 256 * 4);
  const bool auto64 = fills && (a.d == 128 || a.d == 72);
  if (form == 64) return 64;
  if (form == 65 || (form < 0 && auto64)) return 65;
  return 0;
}
bool attn_prefill_takes_seqs(float scale) {
  AttnPrefillArgs a{};
  a.scale = scale;
  return attn_prefill_smx(a) == 3 && attn_form_asked() < 0;
}
bool attn_prefill_takes_qfuse(const AttnPrefillArgs& a) {
  static const bool on = [] { const char* e = getenv("AHA_ATTN_QFUSE"); return e ? atoi(e) != 0 : true; }();
  return on && a.d == 128 && attn_prefill_form(a, attn_prefill_smx(a)) == 0;
}

void launch_attn_prefill(const AttnPrefillArgs& a_in, hipStream_t st) {
  if (a_in.S <= 0) return;
  AttnPrefillArgs a = a_in;
  static const int nw_env = [] {
    const char* e = getenv("AHA_ATTN_WAVES");
    return e ? atoi(e) : 0;
  }();
  constexpr int qt = 1;  // 2 q sub-tiles per wave were measured slower (300 registers: one wave per SIMD)
  // 8 waves (128 q rows) per staged tile once that still fills the chip's 512 block slots (two 8-wave blocks per CU); below
  // that, 64-row blocks balance a causal launch better (S = 1542 x 32 heads: 44 vs 48 us; equal at 2048, 8 waves ahead from there)
  int nwv = (a.d != 64 && (int64_t)((a.S + 127) / 128 + (a.S2 + 127) / 128) * a.nh >= 512) ? 8 : 4;
  if (nw_env == 4 || (nw_env == 8 && a.d != 64)) nwv = nw_env;
  static const int sched_env = [] {
    const char* e = getenv("AHA_ATTN_SCHED");
    return e ? atoi(e) : 1;
  }();
  const bool xcd_order = sched_env && a.kvh % 8 == 0 && a.nh % a.kvh == 0;
  // AHA_ATTN_SEG2=0: a second segment always as its own launch (A/B)
  static const int seg2_env = [] { const char* e = getenv("AHA_ATTN_SEG2"); return e ? atoi(e) : 1; }();
  if (a.S2 > 0 && !(a.causal && xcd_order && seg2_env)) {
    AttnPrefillArgs b = a;
    b.S2 = 0;
    launch_attn_prefill(b, st);
    b.q = (const char*)a.q + (int64_t)a.S * (a.q_ld ? a.q_ld : (int64_t)a.nh * (a.d == 72 ? 96 : a.d)) * 2;
    b.o = (char*)a.o + (int64_t)a.S * a.nh * a.d * 2;
    if (a.q_rope_tab) b.q_rope_tab = (const char*)a.q_rope_tab + (int64_t)a.S * 128 * 2;   // the table rows travel with the q rows
    b.S = a.S2, b.kv_offset = a.kv_offset2, b.kv_total = a.kv_total2;
    launch_attn_prefill(b, st);
    return;
  }
  const int nqb = (a.S + 16 * qt * nwv - 1) / (16 * qt * nwv) + (a.S2 + 16 * qt * nwv - 1) / (16 * qt * nwv);
  a.nqb = xcd_order ? nqb : 0;
  dim3 grid = a.nqb ? dim3(nqb * a.nh) : dim3(nqb, a.nh), block(nwv * 64);
  // AHA_ATTN_SMX: the score chain.
  //   3 (default since round 5) = the f32 score chain: the scores stay the f32 QK^T accumulators through scale, mask, maximum and
  //       exponential; P is rounded to bf16 once for the P.V MFMA (attn_common.h softmax_scores<3>)
  //   0 = the reference's rounding chain bf16(bf16(q.k) * bf16(scale)) (modules.rs:782-783) in the vector ALU, 1 = the same bits with the
  //       scale multiply on the matrix pipe (needs a bf16-exact scale: every model path has one; an op-level caller with another scale
  //       gets 0) -- the bit-faithful forms, kept for A/B and for the parity tables of rounds 1-4
  const int smx = attn_prefill_smx(a);
  // (a caller that handed over raw q heads -- q_norm_w -- asked attn_prefill_takes_qfuse first; should the form have changed since, the
  // 16-row kernel below is the one that norms and rotates)
  const int form_pick = a.q_norm_w != nullptr ? 0 : attn_prefill_form(a, smx);
  if (form_pick != 0 && launch_attn_prefill64(a_in, st, form_pick == 64 ? 0 : 1)) return;
  // row-order epilogue stores (AHA_ATTN_EPI_ROWS=0: from the accumulator fragments): 16-byte pieces need head dims in multiples of 8
  // and 16-byte aligned output rows
  static const int epi_env = [] { const char* e = getenv("AHA_ATTN_EPI_ROWS"); return e ? atoi(e) : 1; }();
  a.epi_rows = epi_env && a.d % 8 == 0 && ((uintptr_t)a.o & 15) == 0;
#define ATTN_LAUNCH(DQK_, DV_)                                                                                                   \
  do {                                                                                                                           \
    if (nwv == 8) {                                                                                                              \
      if (smx == 3) hipLaunchKernelGGL((attn_prefill_kernel<DQK_, DV_, 1, 8, false, 0, 3>), grid, block, lds, st, a, nullptr); \
      else if (smx == 1) hipLaunchKernelGGL((attn_prefill_kernel<DQK_, DV_, 1, 8, false, 0, 1>), grid, block, lds, st, a, nullptr); \
      else hipLaunchKernelGGL((attn_prefill_kernel<DQK_, DV_, 1, 8>), grid, block, lds, st, a, nullptr);                         \
    } else {                                                                                                                     \
      if (smx == 3) hipLaunchKernelGGL((attn_prefill_kernel<DQK_, DV_, 1, 4, false, 0, 3>), grid, block, lds, st, a, nullptr); \
      else if (smx == 1) hipLaunchKernelGGL((attn_prefill_kernel<DQK_, DV_, 1, 4, false, 0, 1>), grid, block, lds, st, a, nullptr); \
      else hipLaunchKernelGGL((attn_prefill_kernel<DQK_, DV_, 1, 4>), grid, block, lds, st, a, nullptr);                         \
    }                                                                                                                            \
  } while (0)
  if (a.d == 128) {
    const size_t lds = 2 * KV_PAGE_TOKENS * 2 * (128 + 128);
#ifdef AHA_DEBUG_KERNELS   // per-part cycle trace and the ablation instantiations (results wrong by construction): debug builds only
    static const bool ptrace = [] { const char* e = getenv("AHA_ATTN_PTRACE"); return e && atoi(e) != 0; }();
    if (ptrace && nwv == 8) {   // debug: per-part cycle sums of two waves of the middle block
      static unsigned long long* d_tr = nullptr;
      if (!d_tr) (void)hipMalloc((void**)&d_tr, 16 * 8);
      (void)hipMemsetAsync(d_tr, 0, 16 * 8, st);
      hipLaunchKernelGGL((attn_prefill_kernel<128, 128, 1, 8, true>), grid, block, lds, st, a, d_tr);
      unsigned long long h[16];
      (void)hipMemcpyAsync(h, d_tr, sizeof(h), hipMemcpyDeviceToHost, st);
      (void)hipStreamSynchronize(st);
      static const char* names[7] = {"top", "QK^T", "scores", "probs", "P.V", "stage", "barriers"};
      for (int w = 0; w < 2; ++w) {
        fprintf(stderr, "[attn ptrace] wave %d, %llu tiles, cycles per tile:", w * 4, h[w * 8 + 7]);
        for (int k = 0; k < 7; ++k) fprintf(stderr, " %s %.0f", names[k], h[w * 8 + 7] ? (double)h[w * 8 + k] / (double)h[w * 8 + 7] : 0.0);
        fprintf(stderr, "\n");
      }
      return;
    }
    static const int abl = [] { const char* e = getenv("AHA_ATTN_ABL"); return e ? atoi(e) : 0; }();
    if (abl && nwv == 8) {
      if (abl == 2) hipLaunchKernelGGL((attn_prefill_kernel<128, 128, 1, 8, false, 2>), grid, block, lds, st, a, nullptr);
      if (abl == 3) hipLaunchKernelGGL((attn_prefill_kernel<128, 128, 1, 8, false, 3>), grid, block, lds, st, a, nullptr);
      if (abl == 4) hipLaunchKernelGGL((attn_prefill_kernel<128, 128, 1, 8, false, 4>), grid, block, lds, st, a, nullptr);
      return;
    }
#endif
    ATTN_LAUNCH(128, 128);
  } else if (a.d == 64) {  // Qwen3-ASR audio encoder
    const size_t lds = 2 * KV_PAGE_TOKENS * 2 * (64 + 64);
    if (smx == 3) hipLaunchKernelGGL((attn_prefill_kernel<64, 64, 1, 4, false, 0, 3>), grid, block, lds, st, a, nullptr);
    else if (smx == 1) hipLaunchKernelGGL((attn_prefill_kernel<64, 64, 1, 4, false, 0, 1>), grid, block, lds, st, a, nullptr);
    else hipLaunchKernelGGL((attn_prefill_kernel<64, 64, 1, 4>), grid, block, lds, st, a, nullptr);
  } else {  // head_dim 72 (Qwen3-VL ViT): Q/K rows padded to 96, V block to 80
    const size_t lds = 2 * KV_PAGE_TOKENS * 2 * (96 + 80);
    ATTN_LAUNCH(96, 80);
  }
#undef ATTN_LAUNCH
}

void launch_attn_decode(const AttnDecodeArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(attn_decode_kernel, dim3(a.kvh, a.nsplit), dim3(256), 0, st, a);
  hipLaunchKernelGGL(attn_decode_combine_kernel, dim3(a.nh), dim3(128), 0, st, a, a.nsplit * 4);
}

}  // namespace aha
