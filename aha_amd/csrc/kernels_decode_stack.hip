// All decoder layers of one decode step in ONE launch (1024 columns, 16 query and 8 kv heads of 128 dims, 3072 features).
//
// What bounds a step of this size is the chain of its launches: five a layer, each of which waits ~2 us for the one before it, ~1 us for the vector that
// launch wrote and ~1 us for its first weights, for 5 us of weight traffic a layer.  Here a block per CU stays for the whole step.  It owns the same part of
// every projection in every layer (120 KB of weights), which four of its waves keep in flight a whole layer ahead, in registers: as soon as a stage has used its
// rows it requests the next layer's.  What the blocks exchange are the vectors between the stages; the other four waves wait for those, and no weight request
// stands in front of their loads.
//
// Who does what.  Blocks are dealt to the eight XCDs in turn, so block b is on XCD x = b % 8, number s = b / 8 of 32 there, and an XCD takes what needs no other:
// kv head x with its two query heads (q, k, v: 16 rows a block; pages s, s + 32, ..; 8 of the joined sums), o_proj over that head's 256 columns (32 rows a
// block), 384 features of gate and up (12 a block), down over these (32 rows a block).  Only o_proj's and down's f32 sums cross: block s of every XCD adds up
// the eight parts of rows 32 s .. and shares the new residual with its XCD.
//
// Exchange.  A value travels with its tag in one dword (bf16 and the low half of the tag) or two (f32 and the tag) and is polled past the L1: whoever sees the tag
// has the value, so nothing is acknowledged, counted or fenced.  Inside an XCD stores stop at its L2 (0.46 us from store to use on an idle chip); what crosses is
// stored through to memory (1.0 us), in 64 bytes that one wave writes -- with four waves' dwords side by side a line is written piece by piece, and the hand-off
// of 1024 values to everyone took 3.5 us.  Every place is written once a layer, by the same block, and its next value needs something that every reader of this
// one sends later: one buffer per stage.  And every launch writes every place that is told by the low half of a tag, which comes again after 65536 layers.
//
// What it gives, us a token of 28 layers with the head's 50: 19 positions 524 (separate launches) -> 326, 400: 580 -> 348, 2048: 607 -> 370, 7000: 682 -> 475, 32000:
// 1210 -> 980.  A layer is 10 us: 31 MB of weights (5.4 at the rate HBM reaches, most of it under what follows), 2.7 of arithmetic, four hand-offs inside an XCD, two across.
//
// Waits are bounded: the blocks have to be on the GPU together (and where they are thought to be), which nothing promises.  A wave that has polled in vain for long
// enough waits no more in this launch and goes on with zeros; the launch then ends by itself, with numbers that mean nothing, and says so in `fail`, and the host runs the
// step as separate launches (model.hip).
#include "attn_common.h"
#include "kernels.h"
#include "stack_exchange.h"

namespace aha {

namespace {
using namespace stack;

constexpr int H = 1024, NH = 16, KVH = 8, D = 128, FF = 3072, NQ = NH * D;
constexpr int BLOCKS = DECODE_STACK_BLOCKS, XCDS = 8, GROUP = BLOCKS / XCDS;   // blocks of an XCD
constexpr int OC = NQ / XCDS, DC = FF / XCDS, RB = H / GROUP;                  // columns of o_proj and down per XCD; rows of the residual per block

// places of the exchange, bytes: per XCD the residual (twice a layer), q k v, attention output, features, attention splits; then what crosses
constexpr int AT_X = 0, AT_X2 = AT_X + H * 4, AT_Q = AT_X2 + H * 4, AT_A = AT_Q + 512 * 4, AT_M = AT_A + OC * 4, AT_P = AT_M + DC * 4;
constexpr int P_HEAD = 16 + D * 8, P_SPLIT = 2 * P_HEAD;                       // a split's share of two heads: max and sum, then the 128 sums, each with its tag
constexpr int PER_XCD = (AT_P + GROUP * P_SPLIT + 127) / 128 * 128;
constexpr int AT_O = XCDS * PER_XCD, AT_D = AT_O + BLOCKS * RB * 8;            // (x, row) f32 with its tag
constexpr int EXCHANGE = AT_D + BLOCKS * RB * 8;
static_assert(EXCHANGE <= DECODE_STACK_EXCHANGE, "exchange buffer");
typedef const __attribute__((address_space(4))) DecodeStackLayer* layer_ptr_t;

struct Lds {
  bf16_t x[H], x2[H], a[OC], m[DC];   // x, x2: behind the norm
  bf16_t q[2 * D], k[D], v[D];
  float sc[2][2 * 64];
  float ss[4];
};

// ---- the waves that compute ------------------------------------------------------------------------------------------------------------------

// PG: pages that are requested a layer ahead (1: no block has a second one)
template <int PG>
__device__ __forceinline__ void compute_waves(const DecodeStackArgs& a, Lds& lds, const int b, const int w) {
  const int lane = threadIdx.x & 63, G = lane >> 4, c = lane & 15, x = b % XCDS, s = b / XCDS;
  const layer_ptr_t layers = (layer_ptr_t)(uintptr_t)a.layers;
  const auto ex = rsrc(a.exchange, EXCHANGE);
  const uint32_t mine = x * PER_XCD, l16 = (uint32_t)lane * 16;
  const int npages = (a.kv_len - 1 + KV_PAGE_TOKENS - 1) / KV_PAGE_TOKENS;

  // q, k, v: rows 16 s .. of the kv head's 512 (two heads of q, k, v)
  const int r16 = s * 16, qkv0 = r16 < 256 ? x * 256 + r16 : r16 < 384 ? NQ + x * 128 + (r16 - 256) : NQ + KVH * 128 + x * 128 + (r16 - 384);
  const int row8 = s * RB + w * 8, f0 = x * DC + s * 12 + w * 3;

  u32x4_t wq[8], wo[4], wg[12], wd[6], kf[PG][4], vf[PG][4];
  // (rows as lane offsets: a layer's descriptors are its pointers)
  const uint32_t at_q = (qkv0 + w * 4) * (H * 2) + l16, at_o = row8 * (NQ * 2) + x * (OC * 2) + (lane >> 5) * (NQ * 2) + (lane & 31) * 16;
  const uint32_t at_d = row8 * (FF * 2) + x * (DC * 2) + G * (FF * 2) + c * 16;
  uint32_t at_g[3];   // 16-row blocks alternating gate / up
#pragma unroll
  for (int j = 0; j < 3; ++j) at_g[j] = (((f0 + j) >> 4) * 32 + ((f0 + j) & 15)) * (H * 2) + l16;
  auto get_qkv = [&](const void* p, bool have) {
    const auto rs = rsrc(p, have ? (NQ + 2 * KVH * D) * H * 2 : 0);
#pragma unroll
    for (int i = 0; i < 8; ++i) wq[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, at_q + i % 4 * 1024, i / 4 * 4096, AUX_NT);
  };
  auto get_o = [&](const void* p, bool have) {   // two rows a load
    const auto rs = rsrc(p, have ? H * NQ * 2 : 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) wo[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, at_o, i * (2 * NQ * 2), AUX_NT);
  };
  auto get_gu = [&](const void* p, bool have, int from, int to) {   // features [from, to) of the wave's three
    const auto rs = rsrc(p, have ? 2 * FF * H * 2 : 0);
#pragma unroll
    for (int j = from; j < to; ++j)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        wg[j * 4 + u] = __builtin_amdgcn_raw_buffer_load_b128(rs, at_g[j] + u * 1024, 0, AUX_NT);
        wg[j * 4 + 2 + u] = __builtin_amdgcn_raw_buffer_load_b128(rs, at_g[j] + u * 1024, 16 * H * 2, AUX_NT);
      }
  };
  auto get_d = [&](const void* p) {   // four rows x 128 columns a load
    const auto rs = rsrc(p, H * FF * 2);
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int j = 0; j < 3; ++j) wd[q * 3 + j] = __builtin_amdgcn_raw_buffer_load_b128(rs, at_d + j * 256, q * (4 * FF * 2), AUX_NT);
  };
  // lane i: where page s + 32 i of layer 0 lies
  uint64_t my_pages = 0;
  if (s + lane * GROUP < npages) my_pages = a.page_ptrs[s + lane * GROUP];
  auto page_at = [&](int i, int layer) {
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)my_pages, i & 63), hi = __builtin_amdgcn_readlane((uint32_t)(my_pages >> 32), i & 63);
    return (((uint64_t)hi << 32) | lo) + (uint64_t)layer * a.layer_stride;
  };
  // keys of the wave's 16 tokens, values of its 32 dims
  auto get_k = [&](uint64_t base, bool have, u32x4_t (&kf)[4]) {
    const auto rs = rsrc(reinterpret_cast<const void*>(base), have ? KVH * KV_PAGE_TOKENS * 512 : 0);
    const int at_k = x * KV_PAGE_TOKENS * 256 + w * 4096;
#pragma unroll
    for (int i = 0; i < 4; ++i) kf[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, l16 + i * 1024, at_k, AUX_NT);
  };
  auto get_v = [&](uint64_t base, bool have, u32x4_t (&vf)[4]) {
    const auto rs = rsrc(reinterpret_cast<const void*>(base), have ? KVH * KV_PAGE_TOKENS * 512 : 0);
    const int at_v = (KVH + x) * KV_PAGE_TOKENS * 256 + w * 4096;
#pragma unroll
    for (int i = 0; i < 4; ++i) vf[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, l16 + i * 1024, at_v, AUX_NT);
  };

  DecodeStackLayer L;
  auto layer = [&](int l) {
    const auto p = layers + l;
    L.wqkv = p->wqkv; L.wo = p->wo; L.wgu = p->wgu; L.wdown = p->wdown;
  };
  layer(0);
  // When a layer's weights are requested.  What a CU loads comes back in the order it was asked for, whoever asked: a poll that was sent behind 16 KB from HBM
  // returns behind them, 1.0 us later, behind 56 KB 1.6; and where more is asked for than the CU keeps in flight, a stage's own results wait to be sent.  So
  // requests are spread over the layer: small ones where a stage begins to compute (HBM's latency passes under it), 32 KB behind what q, k, v of the next layer and
  // gate and up left, where the others' parts need a microsecond to cross anyway.  us a token at 400 / 2048 positions: everything requested behind its stage
  // 424 / 469; all in front of the stages 362 / 413; in two bursts in front of what crosses 394 / 448, behind it 362 / 413; so 346 / 368.
  auto get_pages = [&](int l, bool have) {
#pragma unroll
    for (int i = 0; i < PG; ++i) {
      get_k(page_at(i, l), have && s + i * GROUP < npages, kf[i]);
      get_v(page_at(i, l), have && s + i * GROUP < npages, vf[i]);
    }
  };
  // (in the order of the loop: the counted waits of its first round are those of the others)
  get_pages(0, true);
  IN_ORDER;
  get_qkv(L.wqkv, true);
  IN_ORDER;
  get_o(L.wo, true);
  IN_ORDER;
  get_gu(L.wgu, true, 0, 2);
  IN_ORDER;

  for (int l = 0; l < a.n_layers; ++l) {
    const uint32_t tag = a.epoch * (uint32_t)a.n_layers + (uint32_t)l, t16 = tag & 0xffffu;
    const bool more = l + 1 < a.n_layers;

    // ---- q, k, v ----
    meet();
    meet();
    {
      IN_ORDER;
      get_gu(L.wgu, true, 2, 3);
      IN_ORDER;
      u32x4_t h[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) h[u] = *reinterpret_cast<const u32x4_t*>(lds.x + u * 512 + lane * 8);
      float y[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = dot8_bf(h[1], wq[r * 2 + 1], dot8_bf(h[0], wq[r * 2], 0.f));
      const float v = four_sums(y[0], y[1], y[2], y[3]);
      __builtin_amdgcn_raw_buffer_store_b32(((uint32_t)f2bf(v) << 16) | t16, ex, c == 0 ? mine + AT_Q + (r16 + w * 4 + G) * 4 : NOWHERE, 0, 0);
      IN_ORDER;
    }

    // ---- attention over the pages s, s + 32, ..: a wave the scores of 16 tokens, then 32 dims of the sums ----
    meet();
    IN_ORDER;
    get_d(L.wdown);
    IN_ORDER;
    if (s < npages) {
      bf16x8_t qf[4];
#pragma unroll
      for (int k4 = 0; k4 < 4; ++k4) {
        u32x4_t v = *reinterpret_cast<const u32x4_t*>(lds.q + min(c, 1) * D + k4 * 32 + G * 8);
        if (c >= 2) v = u32x4_t{0u, 0u, 0u, 0u};
        qf[k4] = as_frag(v);
      }
      float m = -INFINITY, z = 0.f;
      f32x4_t o[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
      auto do_page = [&](int page, int it, const u32x4_t (&kf)[4], const u32x4_t (&vf)[4]) {
        f32x4_t st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4) st = mfma16(as_frag(kf[k4]), qf[k4], st);
        const int t0 = page * KV_PAGE_TOKENS + w * 16 + G * 4;
        f32x4_t sv;
#pragma unroll
        for (int r = 0; r < 4; ++r) sv[r] = t0 + r < a.kv_len - 1 ? st[r] * a.scale : -INFINITY;
        float* sc = lds.sc[it & 1];
        if (c < 2) *reinterpret_cast<f32x4_t*>(sc + c * 64 + w * 16 + G * 4) = sv;
        meet();
        f32x4_t sg[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) sg[i] = *reinterpret_cast<const f32x4_t*>(sc + min(c, 1) * 64 + i * 16 + G * 4);
        float alpha;
        bf16x8_t pf[2];
        softmax_tile(sg, 1.0f, [](int) { return true; }, G, m, z, alpha, pf);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          o[i] *= alpha;
#pragma unroll
          for (int kk = 0; kk < 2; ++kk) o[i] = mfma16(as_frag(vf[i * 2 + kk]), pf[kk], o[i]);
        }
        IN_ORDER;
      };
      // (two pages are there; the loop is for more: its waits are good for requests made inside it)
      do_page(s, 0, kf[0], vf[0]);
      if constexpr (PG > 1) {
        if (s + GROUP < npages) do_page(s + GROUP, 1, kf[1], vf[1]);
        for (int page = s + 2 * GROUP, it = 2; page < npages; page += GROUP, ++it) {
          get_k(page_at(it, l), true, kf[0]);
          get_v(page_at(it, l), true, vf[0]);
          IN_ORDER;
          do_page(page, it, kf[0], vf[0]);
        }
      }
      z = rows_sum(z);
      const uint32_t at = mine + AT_P + s * P_SPLIT + c * P_HEAD;
      if (w == 0) {
        const u32x4_t v = {__float_as_uint(m), tag, __float_as_uint(z), tag};
        __builtin_amdgcn_raw_buffer_store_b128(v, ex, lane < 2 ? at : NOWHERE, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const u32x4_t v = {__float_as_uint(o[i][2 * j]), tag, __float_as_uint(o[i][2 * j + 1]), tag};
          __builtin_amdgcn_raw_buffer_store_b128(v, ex, c < 2 ? at + 16 + (w * 32 + i * 16 + G * 4 + j * 2) * 8 : NOWHERE, 0, 0);
        }
      IN_ORDER;
    }

    IN_ORDER;
    get_pages(l + 1, more);
    layer(more ? l + 1 : l);

    // ---- o_proj over the kv head's columns ----
    meet();
    {
      const u32x4_t h = *reinterpret_cast<const u32x4_t*>(lds.a + (lane & 31) * 8);
      float y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = dot8_bf(h, wo[i], 0.f);
      const float y01 = row_sum(quarters(y[0], y[1])), y23 = row_sum(quarters(y[2], y[3]));   // load 2 c + (G & 1), row G >> 1 of its two
      const u32x2_t p = {__float_as_uint(c == 0 ? y01 : y23), tag};
      __builtin_amdgcn_raw_buffer_store_b64(p, ex, c < 2 ? AT_O + (x * H + row8 + c * 4 + (G & 1) * 2 + (G >> 1)) * 8 : NOWHERE, 0, AUX_SC1);
      IN_ORDER;
      get_qkv(L.wqkv, more);
      IN_ORDER;
    }

    // ---- gate and up ----
    meet();
    meet();
    {
      IN_ORDER;
      get_o(L.wo, more);
      IN_ORDER;
      u32x4_t h[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) h[u] = *reinterpret_cast<const u32x4_t*>(lds.x2 + u * 512 + lane * 8);
      float y[6];
#pragma unroll
      for (int r = 0; r < 6; ++r) y[r] = dot8_bf(h[1], wg[r * 2 + 1], dot8_bf(h[0], wg[r * 2], 0.f));
      const float gt = four_sums(y[0], y[2], y[4], y[4]), up = four_sums(y[1], y[3], y[5], y[5]);   // feature G
      const bf16_t v = f2bf(rbf(silu_of(rbf(gt))) * rbf(up));
      __builtin_amdgcn_raw_buffer_store_b32(((uint32_t)v << 16) | t16, ex, c == 0 && G < 3 ? mine + AT_M + (s * 12 + w * 3 + G) * 4 : NOWHERE, 0, 0);
      IN_ORDER;
    }

    // ---- down over the XCD's features ----
    meet();
    {
      float y[2] = {0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const u32x4_t h = *reinterpret_cast<const u32x4_t*>(lds.m + j * 128 + c * 8);
#pragma unroll
        for (int q = 0; q < 2; ++q) y[q] = dot8_bf(h, wd[q * 3 + j], y[q]);
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) y[q] = row_sum(y[q]);
      const u32x2_t p = {__float_as_uint(c == 0 ? y[0] : y[1]), tag};
      __builtin_amdgcn_raw_buffer_store_b64(p, ex, c < 2 ? AT_D + (x * H + row8 + c * 4 + G) * 8 : NOWHERE, 0, AUX_SC1);
      IN_ORDER;
      get_gu(L.wgu, more, 0, 2);
      IN_ORDER;
    }
  }
}

// ---- the waves that wait ---------------------------------------------------------------------------------------------------------------------
// How long a stage's results are not asked for, in naps of 64 clocks (27 ns): a poll sent earlier finds nothing, and the next one waits for it.  Without any: 360 / 367 /
// 397 us a token at 19 / 400 / 2048 positions; 338 / 346 / 368 with (each tried from 0 to 58: flat by 4 either way).
// Splits that every block joins for itself: one hand-off less for twice (one split: eight times) the values.  us a token: 1 page 337 -> 326, 7 pages 346 -> 350, so up to two.
constexpr int DIRECT = 2;
constexpr int NAP_Q = 24, NAP_P = 8, NAP_A = 28, NAP_O = 44, NAP_X = 20, NAP_M = 24, NAP_D = 50;
__device__ __forceinline__ void put4(bf16_t* dst, u32x4_t v) { *reinterpret_cast<uint2*>(dst) = pack4(v); }

__device__ __forceinline__ void gather_waves(const DecodeStackArgs& a, Lds& lds, const int b, const int w) {
  const int lane = threadIdx.x & 63, t = w * 64 + lane, x = b % XCDS, s = b / XCDS;
  const layer_ptr_t layers = (layer_ptr_t)(uintptr_t)a.layers;
  const bool failed = __builtin_amdgcn_readfirstlane(*(volatile const unsigned*)a.fail_dev) != 0;   // an earlier step: this one is thrown away
  Poller poll{rsrc(a.exchange, EXCHANGE), failed ? 0 : a.polls};
  const uint32_t mine = x * PER_XCD;
  const int L_old = a.kv_len - 1, npages = (L_old + KV_PAGE_TOKENS - 1) / KV_PAGE_TOKENS, nsplit = min(npages, GROUP);
  const int my_np = s < npages ? (npages - s + GROUP - 1) / GROUP : 0;
  const float cs = a.rope[lane], sn = a.rope[64 + lane];
  const uint64_t new_page = a.page_ptrs[L_old / KV_PAGE_TOKENS];
  const int new_t = L_old % KV_PAGE_TOKENS;
  const int hd = s / 16, d0 = s % 16 * 8 + (lane >> 5) * 4;   // of wave 0's merge: head, dims of this lane's half
  const int row = s * RB + (lane & 31);                       // of wave 0's sums

  bf16_t res = 0;   // wave 0: the residual at `row`
  if (w == 0) res = ((const bf16_t*)a.x_in)[row];
  // res + the sum of the parts (o_proj, down), shared with the XCD
  auto add_parts = [&](uint32_t at, uint32_t tag, uint32_t to, uint32_t t16) {
    res = f2bf(bf2f(res) + rbf(poll.sum_parts<H>(at, row, tag)));
    __builtin_amdgcn_raw_buffer_store_b32(((uint32_t)res << 16) | t16, poll.ex, lane < 32 ? mine + to + row * 4 : NOWHERE, 0, 0);
  };

  // four columns of the residual behind the norm, to LDS: the waves' sums of squares meet in between
  auto norm4 = [&](uint2 v, uint2 nw, bf16_t* dst) {
    const float x0 = lo_bf(v.x), x1 = hi_bf(v.x), x2 = lo_bf(v.y), x3 = hi_bf(v.y);
    const float ss = wave_sum(fmaf(x0, x0, x1 * x1) + fmaf(x2, x2, x3 * x3));
    if (lane == 0) lds.ss[w] = ss;
    meet();
    const float4 q = *reinterpret_cast<const float4*>(lds.ss);
    const float rinv = 1.0f / sqrtf(((q.x + q.y) + (q.z + q.w)) / (float)H + a.eps);
    *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf(x0 * rinv * lo_bf(nw.x), x1 * rinv * hi_bf(nw.x)), pack_bf(x2 * rinv * lo_bf(nw.y), x3 * rinv * hi_bf(nw.y)));
  };
  auto norm_w = [&](const void* p) {
    const u32x2_t v = global_at<u32x2_t>(p)[t];
    return make_uint2(v[0], v[1]);
  };
  auto head_w = [&](int l) { return global_at<bf16_t>(w == 2 ? layers[l].k_norm : layers[l].q_norm); };

  uint2 in_w = norm_w(layers[0].in_norm), post_w;
  bf16_t w0 = head_w(0)[lane], w1 = head_w(0)[lane + 64];
  uint2 xv = *reinterpret_cast<const uint2*>((const bf16_t*)a.x_in + t * 4);
  for (int l = 0; l < a.n_layers; ++l) {
    const uint32_t tag = a.epoch * (uint32_t)a.n_layers + (uint32_t)l, t16 = tag & 0xffffu;
    const int next = min(l + 1, a.n_layers - 1);
    if (l > 0) {
      if (w == 0) add_parts(AT_D, tag - 1, AT_X, t16);
      if (w) nap(NAP_X);
      xv = pack4(poll.values(true, mine + AT_X + t * 16, t16));
    }
    norm4(xv, in_w, lds.x + t * 4);
    meet();
    post_w = norm_w(layers[l].post_norm);
    nap(NAP_Q);

    // ---- this wave's head: q, q, k with norm and rotation, v as it is ----
    {
      const uint32_t at = mine + AT_Q + (w * 128 + lane) * 4;
      uint32_t v0 = 0, v1 = 0;
      poll.until(false, [&] {
        v0 = __builtin_amdgcn_raw_buffer_load_b32(poll.ex, at, 0, AUX_SC1);
        v1 = __builtin_amdgcn_raw_buffer_load_b32(poll.ex, at + 256, 0, AUX_SC1);
        return (((v0 ^ t16) | (v1 ^ t16)) & 0xffffu) == 0;
      }, [&] { v0 = v1 = 0; });
      bf16_t y0 = (bf16_t)(v0 >> 16), y1 = (bf16_t)(v1 >> 16);
      if (w < 3) {
        float x0 = bf2f(y0), x1 = bf2f(y1);
        const float ss = wave_sum(fmaf(x0, x0, x1 * x1));
        const float rinv = 1.0f / sqrtf(ss / 128.0f + a.eps);
        x0 = rbf(x0 * rinv * bf2f(w0));
        x1 = rbf(x1 * rinv * bf2f(w1));
        y0 = f2bf(rbf(x0 * cs) + rbf(-x1 * sn));
        y1 = f2bf(rbf(x1 * cs) + rbf(x0 * sn));
      }
      bf16_t* dst = w < 2 ? lds.q + w * D : w == 2 ? lds.k : lds.v;
      dst[lane] = y0;
      dst[lane + 64] = y1;
      if (s == 0 && w >= 2) {   // append
        typedef __attribute__((address_space(1))) bf16_t* gbf_t;
        const uint64_t base = new_page + (uint64_t)l * a.layer_stride;
        if (w == 2) {
          gbf_t kd = reinterpret_cast<gbf_t>(base) + x * KV_PAGE_TOKENS * 128;
          kd[kpage_elem(new_t, lane, 4)] = y0;
          kd[kpage_elem(new_t, lane + 64, 4)] = y1;
        } else {
          gbf_t vd = reinterpret_cast<gbf_t>(base) + (KVH + x) * KV_PAGE_TOKENS * 128;
          vd[vpage_elem(new_t, lane)] = y0;
          vd[vpage_elem(new_t, lane + 64)] = y1;
        }
      }
    }
    meet();
    for (int i = 0; i < my_np; ++i) meet();

    // ---- the splits and the new token joined.  Few splits: all 256 sums by every block for itself, a value a thread; more: 8 per block, shared ----
    if (nsplit <= DIRECT) {
      constexpr int N = DIRECT;   // (splits past the last: the last again, without weight)
      const int hh = w >> 1, dim = t & (D - 1);
      const float s_new = wave_sum(fmaf(bf2f(lds.q[hh * D + lane]), bf2f(lds.k[lane]), bf2f(lds.q[hh * D + lane + 64]) * bf2f(lds.k[lane + 64]))) * a.scale;
      nap(NAP_P);
      u32x4_t ml[N];
      u32x2_t p[N];
      poll.until(nsplit == 0, [&] {
        uint32_t bad = 0;
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const uint32_t at = mine + AT_P + min(i, nsplit - 1) * P_SPLIT + hh * P_HEAD;
          ml[i] = __builtin_amdgcn_raw_buffer_load_b128(poll.ex, at, 0, AUX_SC1);
          p[i] = __builtin_amdgcn_raw_buffer_load_b64(poll.ex, at + 16 + dim * 8, 0, AUX_SC1);
        }
#pragma unroll
        for (int i = 0; i < N; ++i) bad |= (ml[i][1] ^ tag) | (ml[i][3] ^ tag) | (p[i][1] ^ tag);
        return bad == 0;
      }, [&] {
#pragma unroll
        for (int i = 0; i < N; ++i) ml[i] = NO_SPLIT, p[i] = u32x2_t{0u, 0u};
      });
      float M = s_new;
#pragma unroll
      for (int i = 0; i < N; ++i) M = fmaxf(M, i < nsplit ? __uint_as_float(ml[i][0]) : -INFINITY);
      float z = __expf(s_new - M), o = z * bf2f(lds.v[dim]);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const float wt = i < nsplit ? __expf(__uint_as_float(ml[i][0]) - M) : 0.f;
        z = fmaf(wt, i < nsplit ? __uint_as_float(ml[i][2]) : 0.f, z);
        o = fmaf(wt, i < nsplit ? __uint_as_float(p[i][0]) : 0.f, o);
      }
      lds.a[t] = f2bf(o * (1.0f / z));
      // the places of the shared sums, which this launch has no use for: a value that thousands of launches leave there has the 16 bits of a tag to come
      if (l + 1 == a.n_layers && w == 0) __builtin_amdgcn_raw_buffer_store_b32(t16, poll.ex, lane < 8 ? mine + AT_A + (s * 8 + lane) * 4 : NOWHERE, 0, 0);
    } else if (w == 0) {
      nap(NAP_P);
      const float dot = wave_sum(fmaf(bf2f(lds.q[hd * D + lane]), bf2f(lds.k[lane]), bf2f(lds.q[hd * D + lane + 64]) * bf2f(lds.k[lane + 64])));
      const float s_new = dot * a.scale;
      const int split = lane & 31;
      const uint32_t at = mine + AT_P + split * P_SPLIT + hd * P_HEAD;
      u32x4_t ml = NO_SPLIT, p0 = {0u, 0u, 0u, 0u}, p1 = {0u, 0u, 0u, 0u};
      poll.until(split >= nsplit, [&] {
        ml = __builtin_amdgcn_raw_buffer_load_b128(poll.ex, at, 0, AUX_SC1);
        p0 = __builtin_amdgcn_raw_buffer_load_b128(poll.ex, at + 16 + d0 * 8, 0, AUX_SC1);
        p1 = __builtin_amdgcn_raw_buffer_load_b128(poll.ex, at + 32 + d0 * 8, 0, AUX_SC1);
        return ml[1] == tag && ml[3] == tag && p0[1] == tag && p0[3] == tag && p1[1] == tag && p1[3] == tag;
      }, [&] { ml = NO_SPLIT, p0 = p1 = u32x4_t{0u, 0u, 0u, 0u}; });
      const float m = __uint_as_float(ml[0]), M = fmaxf(wave_max(m), s_new);
      const float wt = __expf(m - M), wn = __expf(s_new - M);
      const float z = half_wave_sum(wt * __uint_as_float(ml[2])) + wn;
      // rows of 16 lanes: sums 0 and 2 of the half's four in the even one, 1 and 3 in the odd one
      const float s01 = row_sum(quarters(wt * __uint_as_float(p0[0]), wt * __uint_as_float(p0[2]))), s23 = row_sum(quarters(wt * __uint_as_float(p1[0]), wt * __uint_as_float(p1[2])));
      const int e = (lane >> 4 & 1) + (lane & 15) * 2;   // (lanes 0 and 1 of a row)
      const float o = fmaf(wn, bf2f(lds.v[d0 + (e & 3)]), (lane & 15) == 0 ? s01 : s23) * (1.0f / z);
      __builtin_amdgcn_raw_buffer_store_b32(((uint32_t)f2bf(o) << 16) | t16, poll.ex, e < 4 ? mine + AT_A + (hd * D + d0 + e) * 4 : NOWHERE, 0, 0);
    }
    if (w == 1 && nsplit > DIRECT) {
      nap(NAP_A);
      put4(lds.a + lane * 4, poll.values(true, mine + AT_A + lane * 16, t16));
    }
    meet();
    w0 = head_w(next)[lane], w1 = head_w(next)[lane + 64];
    nap(NAP_O);
    if (w == 0) add_parts(AT_O, tag, AT_X2, t16);
    if (w) nap(NAP_X);
    norm4(pack4(poll.values(true, mine + AT_X2 + t * 16, t16)), post_w, lds.x2 + t * 4);
    meet();
    in_w = norm_w(layers[next].in_norm);
    nap(NAP_M);
    if (w < 2) {
      const u32x4_t v = poll.values(t < DC / 4, mine + AT_M + t * 16, t16);
      if (t < DC / 4) put4(lds.m + t * 4, v);
    }
    meet();
    nap(NAP_D);
  }
  if (w == 0) {
    const uint32_t tag = a.epoch * (uint32_t)a.n_layers + (uint32_t)a.n_layers - 1;
    res = f2bf(bf2f(res) + rbf(poll.sum_parts<H>(AT_D, row, tag)));
    if (x == 0 && lane < 32) ((bf16_t*)a.x_out)[row] = res;
  }
  poll.report(failed, a.fail_dev, a.fail_host, a.epoch);
}

template <int PG>
__global__ __launch_bounds__(512, 2) void decode_stack_kernel(const DecodeStackArgs a) {
  __shared__ __attribute__((aligned(16))) Lds lds;
  const int b = blockIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (wave < 4) compute_waves<PG>(a, lds, b, wave);
  else gather_waves(a, lds, b, wave - 4);
}

__global__ __launch_bounds__(64) void stack_dot_kernel(const bf16_t* __restrict__ w, const bf16_t* __restrict__ x, float* __restrict__ y, int k, bool chain) {
  float s = 0.f;
  for (int i = threadIdx.x * 8; i < k; i += 512) {
    const u32x4_t h = ld16(x + i), wt = ld16(w + (int64_t)blockIdx.x * k + i);
    if (!chain) s = dot8_bf(h, wt, s);
    else
      for (int j = 0; j < 4; ++j) s = fmaf(hi_bf(h[j]), hi_bf(wt[j]), fmaf(lo_bf(h[j]), lo_bf(wt[j]), s));
  }
  s = wave_sum(s);
  if (threadIdx.x == 0) y[blockIdx.x] = s;
}

}  // namespace

void launch_stack_dot(const void* w, const void* x, float* y, int n, int k, bool chain, hipStream_t st) {
  hipLaunchKernelGGL(stack_dot_kernel, dim3((unsigned)n), dim3(64), 0, st, (const bf16_t*)w, (const bf16_t*)x, y, k, chain);
}
bool decode_stack_sizes_ok(int width, int heads, int kv_heads, int head_dim, int ff) {
  return width == H && heads == NH && kv_heads == KVH && head_dim == D && ff == FF;
}
void launch_decode_stack(const DecodeStackArgs& a, hipStream_t st) {
  const bool one = a.kv_len - 1 <= GROUP * KV_PAGE_TOKENS;
  hipLaunchKernelGGL(one ? decode_stack_kernel<1> : decode_stack_kernel<2>, dim3(BLOCKS), dim3(512), 0, st, a);
}

}  // namespace aha
