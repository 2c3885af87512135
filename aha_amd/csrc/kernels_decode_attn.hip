// The attention half of a layer of one decode step in ONE launch: norm, q k v, attention, o_proj, residual (4096 columns, 32 query and 8 kv heads of 128 dims, up to 64
// pages of positions).
//
// As three launches these took 24.1 us a layer for 84 MB of weights (13.3 at the rate HBM reaches): q k v 9.4, attention 5.5 with HBM idle, o_proj 9.3 of which 4 are
// its own start and the merge of the attention's splits in every block.  Here a block per CU has its part of both projections (196 KB and 131 KB, in the registers of four
// waves), and o_proj's weights come while four other waves exchange and attend.  XCD x = b % 8 has kv head x with its four query heads, block s = b / 8 there
//   24 of the head's 768 rows of q, k, v, shared inside the XCD;
//   the pages of attention unit s (16 units at most; a wave the scores of 16 tokens, then 32 dims of the sums), shared inside the XCD; beyond 24 pages (DIRECT) pages s and
//     s + 32, each a unit of its own, as the attention launch has it there;
//   from block 16 on: 32 of the head's 512 joined sums, which go to everybody (DIRECT: 16 by every block);
//   16 whole rows of o_proj.
// Of 19 us q k v take 8.5, the hand-off of q k v 1.2, norm and rotation 0.4, a page 1.0, the units' hand-off and the join 2.1, the joined sums' 2.5 (all 256 blocks ask for
// all of them), o_proj behind them 1.3.  us a layer of 8B with gate, up and down (49.6): 20 positions 71.4 -> 70.1, 900: 74.6 -> 70.4, 1550: 76.4 -> 70.5,
// 2200: 76.5 -> 71.2, 3900: 76.9 -> 72.5.
// Exchange and bounded waits: kernels_decode_stack.hip.
//
// The same bits as the three launches (kernels_gemv.hip, attn_decode_body.h, kernels_gemv_fused.hip MergePro): lanes take the same columns in the same order, units
// the same pages, and their sums are joined first within what was a block of four, then over the splits.  A 36-layer stack with a bf16 residual stream moves its logits
// by 3 % of their spread for another order of sums.
#include "attn_common.h"
#include "gemv_body.h"
#include "kernels.h"
#include "stack_exchange.h"

namespace aha {

namespace {
using namespace stack;

constexpr int H = 4096, NH = 32, KVH = 8, D = 128, GR = NH / KVH, XCDS = 8, GROUP = DECODE_STACK_BLOCKS / XCDS;
constexpr int QKV = (GR + 2) * D, QR = QKV / GROUP / 4, OR = H / DECODE_STACK_BLOCKS / 4;   // a kv head's rows; rows of q k v and of o_proj per wave
constexpr int MAX_SPLITS = 4, NW = 4, MAX_UNITS = MAX_SPLITS * NW, PG = 2, DIRECT_SPLITS = GROUP * PG / NW;                  // units of a split; pages of a unit
constexpr int VALUES = GR * D / (GROUP - MAX_UNITS);                                        // joined sums of a block without pages
static_assert(QR == 6 && OR == 4 && VALUES == 32, "rows of a wave");

// places of the exchange, bytes: all the joined sums; per XCD q k v, then the units' sums
constexpr int P_HEAD = 16 + D * 8, P_UNIT = GR * P_HEAD;   // max and sum, then the 128 sums, each with its tag
constexpr int AT_A = 0, AT_Q = AT_A + H * 4, AT_P = AT_Q + XCDS * QKV * 4, EXCHANGE = AT_P + XCDS * DIRECT_SPLITS * NW * P_UNIT;
static_assert(AT_P % 128 == 0 && P_UNIT % 64 == 0, "a tag's place never holds a value, whichever number of units is in use");
static_assert(EXCHANGE <= DECODE_STACK_EXCHANGE, "exchange buffer");

struct Lds {
  float xs[H];   // behind the norm, then the joined sums (gemv_body.h xs_index)
  bf16_t q[GR * D], k[D], v[D];
  float sc[PG][GR * 64];
  float red[4];
  float4 part[4][64];
};
// naps of 64 clocks (27 ns): before the first weights are asked for (x comes first: 8 naps 70.9 us a layer, 12: 70.1,
// 16: 70.3, 22: 70.4), before the units' sums, before all the joined sums
constexpr int NAP_W = 12, NAP_P = 20, NAP_A = 40;

// h of eight columns and eight weights, in the order of gemv_body.h
__device__ __forceinline__ float add_group(const Lds& lds, int u, int lane, u32x4_t wt, float y) {
  const float4 lo = *reinterpret_cast<const float4*>(lds.xs + (u << 9) + (lane << 2)), hi = *reinterpret_cast<const float4*>(lds.xs + (u << 9) + 256 + (lane << 2));
  y = fmaf(lo.x, lo_bf(wt[0]), y); y = fmaf(lo.y, hi_bf(wt[0]), y);
  y = fmaf(lo.z, lo_bf(wt[1]), y); y = fmaf(lo.w, hi_bf(wt[1]), y);
  y = fmaf(hi.x, lo_bf(wt[2]), y); y = fmaf(hi.y, hi_bf(wt[2]), y);
  y = fmaf(hi.z, lo_bf(wt[3]), y); y = fmaf(hi.w, hi_bf(wt[3]), y);
  return y;
}

// ---- the waves that hold weights -------------------------------------------------------------------------------------------------------------
// What a CU loads comes back in the order it was asked for, whoever asked, so a poll waits for every weight in front of it.  o_proj's are therefore asked for two
// rows x 512 columns a wave at a time, 16 KB a block in flight: at 24 the hand-offs, at 8 the weights are what the block waits for.  us a layer at 300 and 1400 positions: all
// asked for as registers become free, by the four waves that wait as well 71.3 / 72.3; four rows at a time 69.9 / 70.3; two 69.8 / 70.3 (each with a later start, as NAP_W has it now).
template <bool DIRECT>
__device__ __forceinline__ void weight_waves(const DecodeAttnArgs& a, Lds& lds, const int b, const int w, const bool has_page, const bool has_second) {
  const int lane = threadIdx.x & 63, G = lane >> 4, c = lane & 15, x = b % XCDS, s = b / XCDS;
  const uint32_t t16 = a.epoch & 0xffffu, l16 = (uint32_t)lane * 16;
  const auto ex = rsrc(a.exchange, EXCHANGE);
  nap(NAP_W);
  const int r24 = s * 24 + w * QR, row_o = b * 16 + w * OR;   // of the kv head's rows; of o_proj's
  u32x4_t wq[8][QR], wo[8][OR];
  {
    const auto rs = rsrc(a.wqkv, (NH + 2 * KVH) * D * H * 2);
    uint32_t at[QR];
#pragma unroll
    for (int i = 0; i < QR; ++i) {
      const int j = r24 + i;
      at[i] = (uint32_t)(j < GR * D ? x * GR * D + j : j < GR * D + D ? NH * D + x * D + (j - GR * D) : (NH + KVH) * D + x * D + (j - GR * D - D)) * (H * 2) + l16;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
#pragma unroll
      for (int i = 0; i < QR; ++i) wq[u][i] = __builtin_amdgcn_raw_buffer_load_b128(rs, at[i], u * 1024, AUX_NT);
      IN_ORDER;
    }
  }
  const uint32_t at_o = (uint32_t)row_o * (H * 2) + l16;
  auto get_o = [&](int u, int from, int to) {
    const auto rs = rsrc(a.wo, H * H * 2);
#pragma unroll
    for (int i = from; i < to; ++i) wo[u][i] = __builtin_amdgcn_raw_buffer_load_b128(rs, at_o + i * (H * 2), u * 1024, AUX_NT);
  };
  auto next_o = [&](int u) {
    IN_ORDER;
#pragma unroll
    for (int i = 0; i < OR; i += 2) {
      asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
      IN_ORDER;
      get_o(u, i, i + 2);
      IN_ORDER;
    }
  };
  meet();
  meet();
  // ---- q, k, v ----
  {
    float y[QR] = {};
#pragma unroll
    for (int u = 0; u < 8; ++u) {
#pragma unroll
      for (int i = 0; i < QR; ++i) y[i] = add_group(lds, u, lane, wq[u][i], y[i]);
      IN_ORDER;
      if (u == 3) get_o(0, 0, OR);
      IN_ORDER;
    }
    const float ya = four_sums(y[0], y[1], y[2], y[3]), yb = four_sums(y[4], y[5], y[4], y[5]);   // (the order of wave_sum)
    const int j = r24 + (c == 0 ? G : 4 + G);
    __builtin_amdgcn_raw_buffer_store_b32(((uint32_t)f2bf(c == 0 ? ya : yb) << 16) | t16, ex, c == 0 || (c == 1 && G < 2) ? AT_Q + x * QKV * 4 + j * 4 : NOWHERE, 0, 0);
  }
  next_o(1);
  meet();
  next_o(2);
  if (has_page) meet();
  if (has_second) meet();
  if constexpr (DIRECT) meet();
  next_o(3);
  next_o(4);
  next_o(5);
  next_o(6);
  next_o(7);
  const bf16_t res = ((const bf16_t*)a.x)[row_o + G];   // (of this block's rows, which nobody else writes)
  // ---- o_proj, residual ----
  // (half of the weights as f32 before the sums are there: what follows them is a chain of 512 instructions a SIMD)
  float wf[4][OR][8];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int i = 0; i < OR; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        wf[u][i][2 * e] = lo_bf(wo[u][i][e]);
        wf[u][i][2 * e + 1] = hi_bf(wo[u][i][e]);
        asm volatile("" : "+v"(wf[u][i][2 * e]), "+v"(wf[u][i][2 * e + 1]));
      }
  meet();
  float y[OR] = {};
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float4 lo = *reinterpret_cast<const float4*>(lds.xs + (u << 9) + (lane << 2)), hi = *reinterpret_cast<const float4*>(lds.xs + (u << 9) + 256 + (lane << 2));
#pragma unroll
    for (int i = 0; i < OR; ++i) {
      y[i] = fmaf(lo.x, wf[u][i][0], y[i]); y[i] = fmaf(lo.y, wf[u][i][1], y[i]); y[i] = fmaf(lo.z, wf[u][i][2], y[i]); y[i] = fmaf(lo.w, wf[u][i][3], y[i]);
      y[i] = fmaf(hi.x, wf[u][i][4], y[i]); y[i] = fmaf(hi.y, wf[u][i][5], y[i]); y[i] = fmaf(hi.z, wf[u][i][6], y[i]); y[i] = fmaf(hi.w, wf[u][i][7], y[i]);
    }
  }
#pragma unroll
  for (int u = 4; u < 8; ++u)
#pragma unroll
    for (int i = 0; i < OR; ++i) y[i] = add_group(lds, u, lane, wo[u][i], y[i]);
  const float r = four_sums(y[0], y[1], y[2], y[3]);
  if (c == 0) ((bf16_t*)a.x)[row_o + G] = f2bf(bf2f(res) + rbf(r));
}

// ---- the waves that wait, and attend ---------------------------------------------------------------------------------------------------------
template <bool DIRECT>
__device__ __forceinline__ void gather_waves(const DecodeAttnArgs& a, Lds& lds, const int b, const int w, const int npages, const bool has_page, const bool has_second) {
  const int lane = threadIdx.x & 63, tid = w * 64 + lane, G = lane >> 4, c = lane & 15, x = b % XCDS, s = b / XCDS;
  const uint32_t tag = a.epoch, t16 = tag & 0xffffu, q_at = AT_Q + x * QKV * 4, p_at = AT_P + x * (DIRECT ? DIRECT_SPLITS * NW : MAX_UNITS) * P_UNIT, l16 = (uint32_t)lane * 16;
  const int L_old = a.kv_len - 1, step = DIRECT ? GROUP : a.nsplit * NW, new_pg = L_old / KV_PAGE_TOKENS;   // step: from a block's first page to its second

  // ---- requests ----
  const uint64_t my_page = a.page_ptrs[lane < PG ? min(s + lane * step, new_pg) : new_pg];   // lanes 0, 1: the unit's pages, 2: the new token's
  u32x4_t xv[2], nv[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    xv[j] = ld16((const bf16_t*)a.x + (tid + j * 256) * 8);
    nv[j] = ld16((const bf16_t*)a.in_norm + (tid + j * 256) * 8);
  }
  const unsigned fail = *global_at<unsigned>(a.fail_dev);
  const float cs = a.rope[lane], sn = a.rope[64 + lane];
  const bf16_t q0 = ((const bf16_t*)a.q_norm)[lane], q1 = ((const bf16_t*)a.q_norm)[lane + 64], k0 = ((const bf16_t*)a.k_norm)[lane], k1 = ((const bf16_t*)a.k_norm)[lane + 64];
  IN_ORDER;
  // ---- h = RMSNorm(x) ----
  {
    float ss = 0.f;
    float f[2][8];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int e = 0; e < 4; ++e) { f[j][2 * e] = lo_bf(xv[j][e]); f[j][2 * e + 1] = hi_bf(xv[j][e]); }
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += f[j][e] * f[j][e];
    }
    ss = wave_sum(ss);
    if (lane == 0) lds.red[w] = ss;
    meet();
    const float tot = lds.red[0] + lds.red[1] + lds.red[2] + lds.red[3];
    const float rinv = 1.0f / sqrtf(tot / (float)H + a.eps);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int base = xs_index((tid + j * 256) * 8);
      float h[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) { h[2 * e] = rbf(f[j][2 * e] * rinv * lo_bf(nv[j][e])); h[2 * e + 1] = rbf(f[j][2 * e + 1] * rinv * hi_bf(nv[j][e])); }
      *reinterpret_cast<float4*>(lds.xs + base) = make_float4(h[0], h[1], h[2], h[3]);
      *reinterpret_cast<float4*>(lds.xs + base + 256) = make_float4(h[4], h[5], h[6], h[7]);
    }
    meet();
  }
  auto page_at = [&](int i) {
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)my_page, i), hi = __builtin_amdgcn_readlane((uint32_t)(my_page >> 32), i);
    return (((uint64_t)hi << 32) | lo) + a.layer_off;
  };
  // keys of the wave's 16 tokens, values of its 32 dims
  u32x4_t kf[PG][4], vf[PG][4];
#pragma unroll
  for (int i = 0; i < PG; ++i) {
    const auto rs = rsrc(reinterpret_cast<const void*>(page_at(i)), (i == 0 ? has_page : has_second) ? KVH * KV_PAGE_TOKENS * 512 : 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) kf[i][j] = __builtin_amdgcn_raw_buffer_load_b128(rs, l16 + j * 1024, x * KV_PAGE_TOKENS * 256 + w * 4096, AUX_NT);
#pragma unroll
    for (int j = 0; j < 4; ++j) vf[i][j] = __builtin_amdgcn_raw_buffer_load_b128(rs, l16 + j * 1024, (KVH + x) * KV_PAGE_TOKENS * 256 + w * 4096, AUX_NT);
  }
  const uint64_t new_page = page_at(PG);
  IN_ORDER;
  const bool failed = __builtin_amdgcn_readfirstlane(fail) != 0;   // an earlier launch: this step is thrown away
  Poller poll{rsrc(a.exchange, EXCHANGE), failed ? 0 : a.polls};

  // ---- a query head per wave, k by wave 0, v by wave 1 ----
  bf16_t y0, y1;
  {
    const uint32_t at0 = q_at + (w * D + lane) * 4, at1 = q_at + ((GR + (w & 1)) * D + lane) * 4;
    uint32_t v[4];
    poll.until(false, [&] {
      v[0] = __builtin_amdgcn_raw_buffer_load_b32(poll.ex, at0, 0, AUX_SC1);
      v[1] = __builtin_amdgcn_raw_buffer_load_b32(poll.ex, at0 + 256, 0, AUX_SC1);
      v[2] = __builtin_amdgcn_raw_buffer_load_b32(poll.ex, at1, 0, AUX_SC1);
      v[3] = __builtin_amdgcn_raw_buffer_load_b32(poll.ex, at1 + 256, 0, AUX_SC1);
      return (((v[0] ^ t16) | (v[1] ^ t16) | (v[2] ^ t16) | (v[3] ^ t16)) & 0xffffu) == 0;
    }, [&] { v[0] = v[1] = v[2] = v[3] = 0; });
    auto norm_rope = [&](uint32_t d0, uint32_t d1, bf16_t w0, bf16_t w1, bf16_t& y0, bf16_t& y1) {
      float x0 = bf2f((bf16_t)(d0 >> 16)), x1 = bf2f((bf16_t)(d1 >> 16));
      const float ss = wave_sum(fmaf(x0, x0, x1 * x1));
      const float rinv = 1.0f / sqrtf(ss / 128.0f + a.eps);
      x0 = rbf(x0 * rinv * bf2f(w0));
      x1 = rbf(x1 * rinv * bf2f(w1));
      y0 = f2bf(rbf(x0 * cs) + rbf(-x1 * sn));
      y1 = f2bf(rbf(x1 * cs) + rbf(x0 * sn));
    };
    norm_rope(v[0], v[1], q0, q1, y0, y1);
    lds.q[w * D + lane] = y0;
    lds.q[w * D + lane + 64] = y1;
    if (w < 2) {
      if (w == 0) norm_rope(v[2], v[3], k0, k1, y0, y1);
      if (w == 1) y0 = (bf16_t)(v[2] >> 16), y1 = (bf16_t)(v[3] >> 16);
      bf16_t* dst = w == 0 ? lds.k : lds.v;
      dst[lane] = y0;
      dst[lane + 64] = y1;
    }
  }
  meet();

  // ---- the unit's pages ----
  if (has_page) {
    bf16x8_t qf[4];
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4) {
      u32x4_t v = *reinterpret_cast<const u32x4_t*>(lds.q + min(c, GR - 1) * D + k4 * 32 + G * 8);
      if (c >= GR) v = u32x4_t{0u, 0u, 0u, 0u};
      qf[k4] = as_frag(v);
    }
    float m = -INFINITY, z = 0.f;
    f32x4_t o[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
    auto do_page = [&](int page, float* sc, const u32x4_t (&kf)[4], const u32x4_t (&vf)[4]) {
      f32x4_t st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k4 = 0; k4 < 4; ++k4) st = mfma16(as_frag(kf[k4]), qf[k4], st);
      if (c < GR) *reinterpret_cast<f32x4_t*>(sc + c * 64 + w * 16 + G * 4) = st;
      meet();
      f32x4_t sg[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) sg[i] = *reinterpret_cast<const f32x4_t*>(sc + min(c, GR - 1) * 64 + i * 16 + G * 4);
      float alpha;
      bf16x8_t pf[2];
      const int t0 = page * KV_PAGE_TOKENS;
      softmax_tile(sg, a.scale, [&](int t) { return t0 + t < L_old; }, G, m, z, alpha, pf);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        o[i] *= alpha;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) o[i] = mfma16(as_frag(vf[i * 2 + kk]), pf[kk], o[i]);
      }
    };
    auto publish = [&](int unit) {
      z = group_sum(z);
      const uint32_t at = p_at + unit * P_UNIT + c * P_HEAD;
      if (w == 0) {
        const u32x4_t v = {__float_as_uint(m), tag, __float_as_uint(z), tag};
        __builtin_amdgcn_raw_buffer_store_b128(v, poll.ex, lane < GR ? at : NOWHERE, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const u32x4_t v = {__float_as_uint(o[i][2 * j]), tag, __float_as_uint(o[i][2 * j + 1]), tag};
          __builtin_amdgcn_raw_buffer_store_b128(v, poll.ex, c < GR ? at + 16 + (w * 32 + i * 16 + G * 4 + j * 2) * 8 : NOWHERE, 0, 0);
        }
    };
    do_page(s, lds.sc[0], kf[0], vf[0]);
    if (has_second) {
      if (DIRECT) {   // (a unit of its own)
        publish(s);
        m = -INFINITY, z = 0.f;
        o[0] = o[1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
      do_page(s + step, lds.sc[1], kf[1], vf[1]);
    }
    publish(DIRECT && has_second ? s + step : s);
    IN_ORDER;
  }

  if (s == 0 && w < 2) {   // append (here: a wait for other stores would be one for these)
    typedef __attribute__((address_space(1))) bf16_t* gbf_t;
    const int t = L_old % KV_PAGE_TOKENS;
    const gbf_t at = reinterpret_cast<gbf_t>(new_page) + (w == 0 ? x : KVH + x) * KV_PAGE_TOKENS * D;
    at[w == 0 ? kpage_elem(t, lane, 4) : vpage_elem(t, lane)] = y0;
    at[w == 0 ? kpage_elem(t, lane + 64, 4) : vpage_elem(t, lane + 64)] = y1;
  }

  // ---- sums joined: lane (split, value) what was a block's four waves, then the splits ----
  // up to four splits: 32 values by each of the XCD's blocks without pages, two waves of (4 splits, 16 values); more: 16 by every block, four such waves for 16 splits
  const int first = DIRECT ? s * 16 : (s - MAX_UNITS) * VALUES + w * 16, q = first / D, dim = first % D + c;
  if (DIRECT || (s >= MAX_UNITS && w < 2)) {
    const int split = DIRECT ? w * 4 + G : G;
    const bool part = split < a.nsplit, own = split == a.nsplit - 1;
    // the new token's scores (lane: head c, 32 dims)
    float d4[4] = {0.f, 0.f, 0.f, 0.f};
    const u32x4_t* qr = reinterpret_cast<const u32x4_t*>(lds.q + min(c, GR - 1) * D + G * 32);
    const u32x4_t* kr = reinterpret_cast<const u32x4_t*>(lds.k + G * 32);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u32x4_t qv = qr[j], kv = kr[j];
#pragma unroll
      for (int e = 0; e < 4; ++e) d4[e] = fmaf(hi_bf(qv[e]), hi_bf(kv[e]), fmaf(lo_bf(qv[e]), lo_bf(kv[e]), d4[e]));
    }
    const float sc = rbf(rbf(group_sum((d4[0] + d4[1]) + (d4[2] + d4[3]))) * a.scale);
    const float s_new = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(sc), q));
    nap(NAP_P);
    u32x4_t ml[NW];
    u32x2_t p[NW];
    auto unit_of = [&](int i) { return DIRECT ? split * NW + i : i * a.nsplit + split; };   // of the block's wave i
    poll.until(!part, [&] {
      uint32_t bad = 0;
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        const int unit = unit_of(i);
        const uint32_t at = unit < npages ? p_at + unit * P_UNIT + q * P_HEAD : NOWHERE;   // (past the range: zeros)
        ml[i] = __builtin_amdgcn_raw_buffer_load_b128(poll.ex, at, 0, AUX_SC1);
        p[i] = __builtin_amdgcn_raw_buffer_load_b64(poll.ex, unit < npages ? at + 16 + dim * 8 : NOWHERE, 0, AUX_SC1);
      }
#pragma unroll
      for (int i = 0; i < NW; ++i)
        if (unit_of(i) < npages) bad |= (ml[i][1] ^ tag) | (ml[i][3] ^ tag) | (p[i][1] ^ tag);
      return bad == 0;
    }, [&] {
#pragma unroll
      for (int i = 0; i < NW; ++i) ml[i] = NO_SPLIT, p[i] = u32x2_t{0u, 0u};
    });
    float mw[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) mw[i] = part && unit_of(i) < npages ? __uint_as_float(ml[i][0]) : -INFINITY;
    float M = own ? s_new : -INFINITY, acc = 0.f, z = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) M = fmaxf(M, mw[i]);
    if (own) {
      z = __expf(s_new - M);
      acc = z * bf2f(lds.v[dim]);
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const float wt = mw[i] == -INFINITY ? 0.f : __expf(mw[i] - M);
      acc = fmaf(wt, mw[i] == -INFINITY ? 0.f : __uint_as_float(p[i][0]), acc);
      z = fmaf(wt, mw[i] == -INFINITY ? 0.f : __uint_as_float(ml[i][2]), z);
    }
    lds.part[w][lane] = make_float4(M, z, acc, 0.f);   // (a split that is not there: nothing, by weight 0)
  }
  auto share = [&](float v) {
    __builtin_amdgcn_raw_buffer_store_b32(((uint32_t)f2bf(v) << 16) | t16, poll.ex, lane < 16 ? AT_A + (x * GR * D + first + c) * 4 : NOWHERE, 0, AUX_SC1);
  };
  if (DIRECT) {
    meet();
    if (w == 0) {
      const float4* const part = &lds.part[0][0];
      const float4 mine4 = part[c * 16];   // lane c: split c's maximum and sum
      const float MM = row_max(mine4.x), wt = mine4.x == -INFINITY ? 0.f : __expf(mine4.x - MM);
      float wz = wt * mine4.y;
      asm volatile("" : "+v"(wz));   // (rounded, not fused into the sum)
      const float inv = 1.0f / row_sum(wz);
      float t[DIRECT_SPLITS], h = 0.f;
#pragma unroll
      for (int i = 0; i < DIRECT_SPLITS; ++i) t[i] = part[i * 16 + c].z;
#pragma unroll
      for (int i = 0; i < DIRECT_SPLITS; ++i) h = fmaf(__uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(wt), i)), t[i], h);
      share(h * inv);
    }
  } else if (s >= MAX_UNITS && w < 2) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (of this wave, read by it alone)
    float4 t[MAX_SPLITS];
#pragma unroll
    for (int i = 0; i < MAX_SPLITS; ++i) t[i] = lds.part[w][i * 16 + c];
    const float MM = fmaxf(fmaxf(t[0].x, t[1].x), fmaxf(t[2].x, t[3].x));
    float h = 0.f, zz = 0.f;
#pragma unroll
    for (int i = 0; i < MAX_SPLITS; ++i) {
      const float wt = t[i].x != -INFINITY ? __expf(t[i].x - MM) : 0.f;
      zz = fmaf(wt, t[i].y, zz);
      h = fmaf(wt, t[i].z, h);
    }
    share(h * (1.0f / zz));
  }
  nap(NAP_A);

  // ---- all joined sums ----
  {
    u32x4_t v[4];
    poll.until(false, [&] {
      uint32_t bad = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = __builtin_amdgcn_raw_buffer_load_b128(poll.ex, AT_A + tid * 16, j * 4096, AUX_SC1);
#pragma unroll
      for (int j = 0; j < 4; ++j) bad |= (v[j][0] ^ t16) | (v[j][1] ^ t16) | (v[j][2] ^ t16) | (v[j][3] ^ t16);
      return (bad & 0xffffu) == 0;
    }, [&] { v[0] = v[1] = v[2] = v[3] = u32x4_t{0u, 0u, 0u, 0u}; });
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<float4*>(lds.xs + xs_index(tid * 4 + j * 1024)) = make_float4(hi_bf(v[j][0]), hi_bf(v[j][1]), hi_bf(v[j][2]), hi_bf(v[j][3]));
    meet();
  }
  poll.report(failed, a.fail_dev, a.fail_host, a.epoch);
}

template <bool DIRECT>
__global__ __launch_bounds__(512, 2) void decode_attn_kernel(const DecodeAttnArgs a) {
  __shared__ __attribute__((aligned(16))) Lds lds;
  const int b = blockIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), s = b / XCDS;
  const int npages = (a.kv_len - 1 + KV_PAGE_TOKENS - 1) / KV_PAGE_TOKENS, units = DIRECT ? GROUP : a.nsplit * NW;   // (direct: as many blocks as there are)
  const bool has_page = s < units && s < npages, has_second = s < units && s + units < npages;
  if (wave < 4) weight_waves<DIRECT>(a, lds, b, wave, has_page, has_second);
  else gather_waves<DIRECT>(a, lds, b, wave - 4, npages, has_page, has_second);
}

}  // namespace

bool decode_attn_sizes_ok(int width, int heads, int kv_heads, int head_dim) { return width == H && heads == NH && kv_heads == KVH && head_dim == D; }
bool decode_attn_splits_ok(int nsplit, int npages, bool direct) {
  return direct ? nsplit <= DIRECT_SPLITS && npages <= NW * nsplit : nsplit >= 1 && nsplit <= MAX_SPLITS && npages <= PG * NW * nsplit;
}
void launch_decode_attn(const DecodeAttnArgs& a, hipStream_t st) { hipLaunchKernelGGL(a.direct ? decode_attn_kernel<true> : decode_attn_kernel<false>, dim3(DECODE_STACK_BLOCKS), dim3(512), 0, st, a); }

}  // namespace aha
