// Runs of pre-norm sublayers of one token of one sequence in ONE launch: state-space mixers and feed-forwards, dense or routed (1024 columns; 32 state-space heads of
// 64 x 128 in 8 groups, 4 taps; 3072 features, or 32 experts of 768 of which two, and a shared one of 1536).
//
// The chain of launches bounds these steps as it does the ones of kernels_decode_stack.hip, whose scheme this is: a block per CU, four waves that compute and keep
// their part of the next sublayer's weights in flight, four that wait for what other blocks send; block b is on XCD x = b % 8, number s = b / 8 there.  A sublayer is
//   LayerNorm of the residual (f32), by every block for itself;
//   state space: the XCD has group x: heads 4 x .. 4 x + 3, their z, x, dt and the group's B and C.  A block computes 8 columns of one head (their x and z, dt again in
//     each of the head's 8 blocks) and 8 of the 256 rows of B and C, which the XCD shares behind the convolution; then its 8 x 128 states, and the 8 gated sums, which
//     the XCD shares for the norm over the group's 256 columns; out over these columns, 32 rows a block;
//   dense: 12 of the XCD's 384 features, shared; down over these;
//   routed: the router's row s, so that an XCD has all 32 logits; every block finds the two experts; 6 features of the shared expert (computed under that), 3 of
//     each chosen one; down over the XCD's 96 + 96 + 192 columns of them.  The chosen experts' rows cannot be asked for earlier than their names are known;
//   the f32 sums of out / down cross XCDs, as there.
// us a token of 28 layers (21 state-space mixers and 28 feed-forwards in 8 runs; 7 attention mixers of their own, 22 each): 655 in 113 launches, 1000 positions -> 480.  A
// sublayer takes 6: 70 KB of weights a CU (3 at the rate HBM reaches), LayerNorm 0.5, 0.6 to 1.2 of f32 arithmetic a stage, hand-offs as there; a routed one waits 2.2 for
// rows that nobody could ask for earlier.  When weights are asked for: 480; both parts in one burst 489 to 495, everything where a stage begins 485 to 500.
#include "expert_choice.h"
#include "kernels_prenorm.h"
#include "rows_common.h"
#include "stack_exchange.h"

namespace aha {

namespace {
using namespace stack;

constexpr int H = 1024, XCDS = 8, GROUP = DECODE_STACK_BLOCKS / XCDS, RB = H / GROUP;
constexpr int HEADS = 32, VD = 64, NS = 128, GROUPS = 8, TAPS = 4, INNER = HEADS * VD, CP = INNER + 2 * GROUPS * NS, C_OFF = INNER, DT_OFF = INNER + CP;
constexpr int GC = INNER / XCDS;                                  // columns of a group = of a norm part
constexpr int FF = 3072, DC = FF / XCDS, EXPERTS = 32, TOP = 2, EFF = 768, SFF = 1536, EC = EFF / XCDS, SC = SFF / XCDS;
static_assert(TOP * EC + SC == DC, "a block's twelve features");
constexpr int PAR_DT = (TAPS + 1) * CP, PAR_A = PAR_DT + HEADS, PAR_D = PAR_A + HEADS;   // places in PrenormOp::par

// places of the exchange, bytes: per XCD the residual, B and C, gated sums, logits (f32), features (bf16); then what crosses, by turns
constexpr int AT_X = 0, AT_BC = AT_X + H * 8, AT_G = AT_BC + 2 * NS * 8, AT_R = AT_G + GC * 8, AT_M = AT_R + EXPERTS * 8, PER_XCD = AT_M + DC * 4;
static_assert(PER_XCD % 128 == 0, "lines");
constexpr int AT_PART = XCDS * PER_XCD, PART = XCDS * H * 8, EXCHANGE = AT_PART + 2 * PART;
static_assert(EXCHANGE <= DECODE_STACK_EXCHANGE, "exchange buffer");

typedef const __attribute__((address_space(4))) PrenormOp* op_ptr_t;

// An op in scalar registers, asked for in front of a wait: behind it, an entry's first use would wait for memory (0.6 to 1.2 us)
struct Op {
  int kind;
  const char *w1, *w2, *router, *egu, *edown, *nw, *nb, *gnorm;
  const float* par;
  int64_t hist, state;
  __device__ __forceinline__ void read(op_ptr_t o) {
    kind = o->kind; w1 = (const char*)o->w1; w2 = (const char*)o->w2; router = (const char*)o->router; egu = (const char*)o->egu; edown = (const char*)o->edown;
    nw = (const char*)o->nw; nb = (const char*)o->nb; gnorm = (const char*)o->gnorm; par = o->par; hist = o->hist; state = o->state;
  }
};
struct Lds {
  float h[H], bc[2 * NS], g[GC];   // h, g: behind the norms
  bf16_t m[DC];
  float xs[8], zs[8], dt[2], red[4][8];
  float conv[16][8], dtp[2];   // the block's channels (x, then B or C): weights, bias, the last inputs; dt_bias and a of its head
  float ss[8];
  int sel[TOP];
  float wt[TOP];
};
__device__ __forceinline__ float softplus(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }

__device__ __forceinline__ float dot8(const float (&h)[8], u32x4_t w, float s) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    s = fmaf(h[2 * j], lo_bf(w[j]), s);
    s = fmaf(h[2 * j + 1], hi_bf(w[j]), s);
  }
  return s;
}
__device__ __forceinline__ void ld8(const float* p, float (&h)[8]) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  h[0] = a.x; h[1] = a.y; h[2] = a.z; h[3] = a.w; h[4] = b.x; h[5] = b.y; h[6] = b.z; h[7] = b.w;
}
__device__ __forceinline__ int pair_row(int f) { return (f >> 4) * 32 + (f & 15); }   // gate row of a feature (16-row blocks alternating gate / up)

// ---- the waves that compute ------------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ void compute_waves(const PrenormStackArgs& a, Lds& lds, const int b, const int w) {
  const int lane = threadIdx.x & 63, G = lane >> 4, c = lane & 15, x = b % XCDS, s = b / XCDS;
  const op_ptr_t ops = (op_ptr_t)(uintptr_t)a.ops;
  const auto ex = rsrc(a.exchange, EXCHANGE);
  const uint32_t mine = x * PER_XCD, l16 = (uint32_t)lane * 16;
  const int head = x * 4 + s / 8, vs8 = s % 8 * 8, row8 = s * RB + w * 8;
  const int k_bc = s * 8 + w * 2;   // of the 256 rows of B and C; a multiple of two, B or C both
  const int ch_bc = INNER + (k_bc < NS ? 0 : GROUPS * NS) + x * NS + k_bc % NS;   // their first channel
  // lane's channel of the convolution: c = 0: x, c = 1: B or C, rows G = 0, 1
  const uint32_t conv_at = G < 2 && c < 2 ? (uint32_t)(c == 0 ? head * VD + vs8 + w * 2 + G : ch_bc + G) * 4 : NOWHERE;
  // lane's places in the rows of w1 and w2, bytes
  uint32_t at_ssm[7], at_dense[3], at_shared[3], at_router = (uint32_t)s * (H * 2) + l16;
#pragma unroll
  for (int j = 0; j < 7; ++j)
    at_ssm[j] = (uint32_t)(j < 2 ? C_OFF + head * VD + vs8 + w * 2 + j : j < 4 ? head * VD + vs8 + w * 2 + j - 2 : j < 6 ? C_OFF + ch_bc + j - 4 : DT_OFF + head) * (H * 2) + l16;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    at_dense[j] = (uint32_t)pair_row(x * DC + s * 12 + w * 3 + j) * (H * 2) + l16;
    at_shared[j] = (uint32_t)pair_row(x * SC + s * 6 + (w & 1) * 3 + j) * (H * 2) + l16;
  }
  const uint32_t at_out = row8 * (INNER * 2) + x * (GC * 2) + (lane >> 5) * (INNER * 2) + (lane & 31) * 16, at_down = row8 * (FF * 2) + x * (DC * 2) + G * (FF * 2) + c * 16;
  u32x4_t w1[7][2], w2[6], S;
  // rows [from, to) of the seven: state space: x, x, z, z, B or C twice, dt; features: gate, up of three, and the router's
  auto get1 = [&](const Op& o, bool have, int from, int to) {
    const int kind = o.kind;
    const auto rs = rsrc(o.w1, have && (kind != PRENORM_MOE || w < 2) ? (kind == PRENORM_SSM ? DT_OFF + HEADS : kind == PRENORM_DENSE ? 2 * FF : 2 * SFF) * H * 2 : 0);
    const auto r6 = rsrc(kind == PRENORM_MOE ? o.router : o.w1, have && w == 0 && kind != PRENORM_DENSE ? (kind == PRENORM_SSM ? DT_OFF + HEADS : EXPERTS) * H * 2 : 0);
#pragma unroll
    for (int j = from; j < to; ++j) {
      const uint32_t at = kind == PRENORM_SSM ? at_ssm[j] : j == 6 ? at_router : (kind == PRENORM_DENSE ? at_dense[j / 2] : at_shared[j / 2]) + (j & 1) * (16 * H * 2);
#pragma unroll
      for (int u = 0; u < 2; ++u) w1[j][u] = __builtin_amdgcn_raw_buffer_load_b128(j == 6 ? r6 : rs, at + u * 1024, 0, AUX_NT);
    }
  };
  const uint32_t st_at = (((uint32_t)head * (VD / 16) + (s % 8) / 2) * NS + ((w * 64 + lane) >> 1)) * 64 + (s % 2) * 32 + (lane & 1) * 16;   // bytes: 16 columns of a row, this block's 8, four of them
  auto get_state = [&](const Op& o, bool have) {
    S = __builtin_amdgcn_raw_buffer_load_b128(rsrc(a.state_in + o.state, have && o.kind == PRENORM_SSM && a.pos0 > 0 ? HEADS * VD * NS * 4 : 0), st_at, 0, 0);
  };
  auto get2 = [&](const Op& o) {   // state space: two rows a load, four loads; dense: four rows x 128 columns; routed: nothing yet
    const bool ssm = o.kind == PRENORM_SSM;
    const auto rs = rsrc(o.w2, ssm ? H * INNER * 2 : o.kind == PRENORM_DENSE ? H * FF * 2 : 0);
#pragma unroll
    for (int i = 0; i < 6; ++i)
      w2[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, ssm ? i < 4 ? at_out + i * (2 * INNER * 2) : NOWHERE : at_down + i / 3 * (4 * FF * 2) + i % 3 * 256, 0, AUX_NT);
  };
  auto feature = [&](float gate, float up, float by) { return f2bf(rbf(silu_of(rbf(gate * by))) * rbf(up * by)); };
  auto features = [&](const float (&h)[2][8], const u32x4_t (*wt)[2], float by, uint32_t at, uint32_t t16) {   // three, rows gate, up
    float y[6];
#pragma unroll
    for (int r = 0; r < 6; ++r) y[r] = dot8(h[1], wt[r][1], dot8(h[0], wt[r][0], 0.f));
    const float gt = four_sums(y[0], y[2], y[4], y[4]), up = four_sums(y[1], y[3], y[5], y[5]);   // feature G
    __builtin_amdgcn_raw_buffer_store_b32(((uint32_t)feature(gt, up, by) << 16) | t16, ex, c == 0 && G < 3 ? mine + AT_M + (at + G) * 4 : NOWHERE, 0, 0);
  };
  auto down = [&](uint32_t part, uint32_t tag) {
    float y[2] = {0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const u32x4_t h = *reinterpret_cast<const u32x4_t*>(lds.m + j * 128 + c * 8);
#pragma unroll
      for (int q = 0; q < 2; ++q) y[q] = dot8_bf(h, w2[q * 3 + j], y[q]);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) y[q] = row_sum(y[q]);
    const u32x2_t p = {__float_as_uint(c == 0 ? y[0] : y[1]), tag};
    __builtin_amdgcn_raw_buffer_store_b64(p, ex, c < 2 ? part + (x * H + row8 + c * 4 + G) * 8 : NOWHERE, 0, AUX_SC1);
  };

  Op o, next;
  next.read(ops);
  get1(next, true, 4, 7);
  IN_ORDER;
  get1(next, true, 0, 4);
  get_state(next, true);
  IN_ORDER;
  for (int i = 0; i < a.n_ops; ++i) {
    const uint32_t tag = a.epoch * PRENORM_STACK_OPS + i, t16 = tag & 0xffffu, part = AT_PART + (i & 1) * PART;
    const bool more = i + 1 < a.n_ops;
    o = next;
    next.read(ops + (more ? i + 1 : i));
    asm volatile("" ::"s"(next.kind), "s"(next.w1), "s"(next.w2), "s"(next.router), "s"(next.state));   // (in front of the wait)
    const int kind = o.kind;
    meet();
    meet();
    float h[2][8];
#pragma unroll
    for (int u = 0; u < 2; ++u) ld8(lds.h + u * 512 + lane * 8, h[u]);

    if (kind == PRENORM_SSM) {
      // ---- z, x, B, C, dt; convolution ----
      const int64_t hist = ops[i].hist, state = ops[i].state;
      float y[7];
#pragma unroll
      for (int r = 0; r < 7; ++r) y[r] = dot8(h[1], w1[r][1], dot8(h[0], w1[r][0], 0.f));
      const float ya = four_sums(y[0], y[1], y[2], y[3]), yb = four_sums(y[4], y[5], y[6], y[6]);
      const float v = c == 0 ? ya : yb;   // c = 0: x, x, z, z by G; c = 1: B or C, B or C, dt, dt
      const float4 cw = *reinterpret_cast<const float4*>(lds.conv[(c & 1) * 8 + w * 2 + (G & 1)]), ch = *reinterpret_cast<const float4*>(lds.conv[(c & 1) * 8 + w * 2 + (G & 1)] + 4);
      float acc = fmaf(cw.w, v, ch.x);
      acc = fmaf(cw.z, ch.y, acc);
      acc = fmaf(cw.y, ch.z, acc);
      acc = fmaf(cw.x, ch.w, acc);
      const float act = silu_f32(G < 2 ? acc : v);
      const u32x2_t p = {__float_as_uint(act), tag};
      __builtin_amdgcn_raw_buffer_store_b64(p, ex, c == 1 && G < 2 ? mine + AT_BC + (k_bc + G) * 8 : NOWHERE, 0, 0);
      if (c == 0) (G < 2 ? lds.xs : lds.zs)[w * 2 + (G & 1)] = act;
      if (w == 0 && lane == 33) {
        const float t = softplus(v + lds.dtp[0]);
        lds.dt[0] = t;
        lds.dt[1] = expf(lds.dtp[1] * t);
      }
      const auto rh = rsrc(a.hist_out + hist, (TAPS - 1) * CP * 4);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rh, conv_at, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ch.y), rh, conv_at, CP * 4, 0);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ch.z), rh, conv_at, 2 * CP * 4, 0);
      IN_ORDER;
      get2(o);
      IN_ORDER;
      // ---- eight columns of the head's state: thread (row n, four columns) ----
      meet();
      {
        const int n = (w * 64 + lane) >> 1, par = lane & 1;
        const float B = lds.bc[n], C = lds.bc[NS + n], dt = lds.dt[0], da = lds.dt[1];
        const float4 xv = *reinterpret_cast<const float4*>(lds.xs + par * 4);
        const float xx[4] = {xv.x, xv.y, xv.z, xv.w};
        float yv[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float st = fmaf(B, dt * xx[q], da * __uint_as_float(S[q]));
          S[q] = __float_as_uint(st);
          yv[q] = C * st;
        }
        float r = quarters(halves(yv[0], yv[1]), halves(yv[2], yv[3]));   // by G: columns 0, 2, 1, 3
        r += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(r), 0x128, 0xf, 0xf, false));
        r += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(r), 0x124, 0xf, 0xf, false));
        r += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(r), 0x122, 0xf, 0xf, false));
        if (c < 2) lds.red[w][c * 4 + (G & 1) * 2 + (G >> 1)] = r;
        __builtin_amdgcn_raw_buffer_store_b128(S, rsrc(a.state_out + state, HEADS * VD * NS * 4), st_at, 0, 0);
      }
      meet();
      meet();
      // ---- out over the group's columns ----
      meet();
      IN_ORDER;
      get1(next, more, 4, 7);
      IN_ORDER;
      float g8[8], yo[4];
      ld8(lds.g + (lane & 31) * 8, g8);
#pragma unroll
      for (int q = 0; q < 4; ++q) yo[q] = dot8(g8, w2[q], 0.f);
      const float y01 = row_sum(quarters(yo[0], yo[1])), y23 = row_sum(quarters(yo[2], yo[3]));
      const u32x2_t po = {__float_as_uint(c == 0 ? y01 : y23), tag};
      __builtin_amdgcn_raw_buffer_store_b64(po, ex, c < 2 ? part + (x * H + row8 + c * 4 + (G & 1) * 2 + (G >> 1)) * 8 : NOWHERE, 0, AUX_SC1);
    } else if (kind == PRENORM_DENSE) {
      features(h, w1, 1.f, s * 12 + w * 3, t16);
      IN_ORDER;
      get2(o);
      IN_ORDER;
      meet();
      IN_ORDER;
      get1(next, more, 4, 7);
      IN_ORDER;
      down(part, tag);
    } else {
      {
        const float z = wave_sum(dot8(h[1], w1[6][1], dot8(h[0], w1[6][0], 0.f)));
        const u32x2_t p = {__float_as_uint(z), tag};
        __builtin_amdgcn_raw_buffer_store_b64(p, ex, w == 0 && lane == 0 ? mine + AT_R + s * 8 : NOWHERE, 0, 0);
      }
      if (w < 2) features(h, w1, 1.f, TOP * EC + s * 6 + w * 3, t16);
      const char *egu = (const char*)ops[i].egu, *edown = (const char*)ops[i].edown;
      asm volatile("" ::"s"(egu), "s"(edown));
      meet();
      const int e0 = __builtin_amdgcn_readfirstlane(lds.sel[0]), e1 = __builtin_amdgcn_readfirstlane(lds.sel[1]);
      if (w >= 2) {
        const int f0 = x * EC + s * 3;
        const auto rs = rsrc(egu + (int64_t)(w == 2 ? e0 : e1) * (2 * EFF * H * 2), 2 * EFF * H * 2);
#pragma unroll
        for (int j = 0; j < 6; ++j)
#pragma unroll
          for (int u = 0; u < 2; ++u) w1[j][u] = __builtin_amdgcn_raw_buffer_load_b128(rs, (uint32_t)(pair_row(f0 + j / 2) + (j & 1) * 16) * (H * 2) + l16 + u * 1024, 0, AUX_NT);
      }
      IN_ORDER;
      {   // columns of down: the choices', then the shared expert's
        const char *ed = edown, *sd = o.w2;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const int col = j * 128 + c * 8, k = col < EC ? 0 : col < 2 * EC ? 1 : 2;
          const char* m = k == 2 ? sd + (x * SC + col - 2 * EC) * 2 : ed + (int64_t)(k == 0 ? e0 : e1) * (H * EFF * 2) + (x * EC + col - k * EC) * 2;
          const int pitch = k == 2 ? SFF * 2 : EFF * 2;
#pragma unroll
          for (int q = 0; q < 2; ++q) w2[q * 3 + j] = __builtin_nontemporal_load(global_at<u32x4_t>(m + (row8 + q * 4 + G) * pitch));
        }
      }
      IN_ORDER;
      if (w >= 2) features(h, w1, lds.wt[w - 2], (w - 2) * EC + s * 3, t16);
      meet();
      IN_ORDER;
      get1(next, more, 4, 7);
      IN_ORDER;
      down(part, tag);
    }
    IN_ORDER;
    get1(next, more, 0, 4);
    get_state(next, more);
    IN_ORDER;
  }
}

// ---- the waves that wait ---------------------------------------------------------------------------------------------------------------------
// naps of 64 clocks before asking (kernels_decode_stack.hip), for B and C, gated sums, features, what crosses, the residual, logits, features behind the choice
constexpr int N_BC = 12, N_G = 4, N_M = 40, N_PART = 24, N_X = 30, N_R = 8, N_ME = 12;
__device__ __forceinline__ void gather_waves(const PrenormStackArgs& a, Lds& lds, const int b, const int w) {
  const int lane = threadIdx.x & 63, t = w * 64 + lane, x = b % XCDS, s = b / XCDS;
  const op_ptr_t ops = (op_ptr_t)(uintptr_t)a.ops;
  const bool failed = __builtin_amdgcn_readfirstlane(*(volatile const unsigned*)a.fail_dev) != 0;   // an earlier step: this one is thrown away
  Poller poll{rsrc(a.exchange, EXCHANGE), failed ? 0 : a.polls};
  const uint32_t mine = x * PER_XCD;
  const int row = s * RB + (lane & 31), head = x * 4 + s / 8;   // of wave 0
  float res = w == 0 ? a.x_in[row] : 0.f;
  auto f32_at = [&](bool part, uint32_t at, uint32_t tag) {
    u32x2_t v = {0u, 0u};
    poll.until(!part, [&] {
      v = __builtin_amdgcn_raw_buffer_load_b64(poll.ex, at, 0, AUX_SC1);
      return v[1] == tag;
    }, [&] { v = u32x2_t{0u, 0u}; });
    return __uint_as_float(v[0]);
  };
  auto four = [&](const void* p) {
    const u32x2_t v = global_at<u32x2_t>(p)[t];
    return make_uint2(v[0], v[1]);
  };
  Op o, next;
  next.read(ops);
  uint2 nw = four(next.nw), nb = four(next.nb);
  float gw = 0.f, dd = 0.f;
  // wave 1: the 16 channels' weights, bias and last inputs, 8 floats each, two a lane
  float cv[2] = {0.f, 0.f}, dtp = 0.f;
  const int k_bc = s * 8, ch_x = head * VD + s % 8 * 8, ch_bc = INNER + (k_bc < NS ? 0 : GROUPS * NS) + x * NS + k_bc % NS;
  auto get_conv = [&](const Op& o) {
    if (w != 1 || o.kind != PRENORM_SSM) return;
    const float *par = o.par, *hist = a.hist_in + o.hist;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int i = lane + k * 64, ch = i / 8 < 8 ? ch_x + i / 8 : ch_bc + i / 8 - 8, e = i % 8;   // weights, bias, the input e - 4 tokens back (none: zero)
      cv[k] = e > TAPS && a.pos0 < e - TAPS ? 0.f : *global_at<float>(e <= TAPS ? par + e * CP + ch : hist + (e - TAPS - 1) * CP + ch);
    }
    dtp = *global_at<float>(par + (lane & 1 ? PAR_A : PAR_DT) + head);
  };
  get_conv(next);
  float4 xv = *reinterpret_cast<const float4*>(a.x_in + t * 4);
  for (int i = 0; i < a.n_ops; ++i) {
    const uint32_t tag = a.epoch * PRENORM_STACK_OPS + i, t16 = tag & 0xffffu;
    o = next;
    next.read(ops + min(i + 1, a.n_ops - 1));
    asm volatile("" ::"s"(next.kind), "s"(next.nw), "s"(next.nb), "s"(next.gnorm), "s"(next.par), "s"(next.hist));
    const int kind = o.kind;
    if (i > 0) {
      if (w == 0) {
        res += poll.sum_parts<H>(AT_PART + ((i - 1) & 1) * PART, row, tag - 1);
        const u32x2_t p = {__float_as_uint(res), tag};
        __builtin_amdgcn_raw_buffer_store_b64(p, poll.ex, lane < 32 ? mine + AT_X + row * 8 : NOWHERE, 0, 0);
      } else {
        nap(N_X);
      }
      u32x4_t v0, v1;
      poll.until(false, [&] {
        v0 = __builtin_amdgcn_raw_buffer_load_b128(poll.ex, mine + AT_X + t * 32, 0, AUX_SC1);
        v1 = __builtin_amdgcn_raw_buffer_load_b128(poll.ex, mine + AT_X + t * 32 + 16, 0, AUX_SC1);
        return v0[1] == tag && v0[3] == tag && v1[1] == tag && v1[3] == tag;
      }, [&] { v0 = v1 = u32x4_t{0u, 0u, 0u, 0u}; });
      xv = make_float4(__uint_as_float(v0[0]), __uint_as_float(v0[2]), __uint_as_float(v1[0]), __uint_as_float(v1[2]));
    }
    {   // LayerNorm: the waves' means and squares about them, joined
      const float m = wave_sum((xv.x + xv.y) + (xv.z + xv.w)) * (1.0f / 256);
      const float d0 = xv.x - m, d1 = xv.y - m, d2 = xv.z - m, d3 = xv.w - m;
      const float q = wave_sum(fmaf(d0, d0, d1 * d1) + fmaf(d2, d2, d3 * d3));
      if (lane == 0) lds.ss[w] = m, lds.ss[4 + w] = q;
      meet();
      const float4 mm = *reinterpret_cast<const float4*>(lds.ss), qq = *reinterpret_cast<const float4*>(lds.ss + 4);
      const float mean = ((mm.x + mm.y) + (mm.z + mm.w)) * 0.25f, e0 = mm.x - mean, e1 = mm.y - mean, e2 = mm.z - mean, e3 = mm.w - mean;
      const float var = (((qq.x + qq.y) + (qq.z + qq.w)) + 256.f * (fmaf(e0, e0, e1 * e1) + fmaf(e2, e2, e3 * e3))) / (float)H;
      const float rinv = 1.0f / sqrtf(var + a.eps);
      *reinterpret_cast<float4*>(lds.h + t * 4) = make_float4(fmaf((xv.x - mean) * rinv, lo_bf(nw.x), lo_bf(nb.x)), fmaf((xv.y - mean) * rinv, hi_bf(nw.x), hi_bf(nb.x)),
                                                              fmaf((xv.z - mean) * rinv, lo_bf(nw.y), lo_bf(nb.y)), fmaf((xv.w - mean) * rinv, hi_bf(nw.y), hi_bf(nb.y)));
    }
    if (w == 1 && kind == PRENORM_SSM) {
#pragma unroll
      for (int k = 0; k < 2; ++k) (&lds.conv[0][0])[lane + k * 64] = cv[k];
      if (lane < 2) lds.dtp[lane] = dtp;
    }
    meet();
    nw = four(next.nw), nb = four(next.nb);
    get_conv(next);
    if (kind == PRENORM_SSM) {
      gw = bf2f(global_at<bf16_t>(o.gnorm)[x * GC + t]);
      dd = global_at<float>(o.par)[PAR_D + head];
      nap(N_BC);
      lds.bc[t] = f32_at(true, mine + AT_BC + t * 8, tag);
      meet();
      meet();
      if (w == 0) {
        const int v = lane & 7;
        const float y = fmaf(dd, lds.xs[v], (lds.red[0][v] + lds.red[1][v]) + (lds.red[2][v] + lds.red[3][v]));
        const u32x2_t p = {__float_as_uint(y * lds.zs[v]), tag};
        __builtin_amdgcn_raw_buffer_store_b64(p, poll.ex, lane < 8 ? mine + AT_G + (s * 8 + v) * 8 : NOWHERE, 0, 0);
      } else {
        nap(N_G);
      }
      const float g = f32_at(true, mine + AT_G + t * 8, tag);
      const float ss = wave_sum(g * g);
      if (lane == 0) lds.ss[w] = ss;
      meet();
      const float4 q = *reinterpret_cast<const float4*>(lds.ss);
      lds.g[t] = g * (1.0f / sqrtf(((q.x + q.y) + (q.z + q.w)) / (float)GC + a.eps)) * gw;
      meet();
    } else {
      if (kind == PRENORM_MOE) {
        if (w == 0) {
          nap(N_R);
          float z = choice_logit(lane < EXPERTS ? f32_at(true, mine + AT_R + (lane & 31) * 8, tag) : -INFINITY);
          if (lane >= EXPERTS) z = -INFINITY;
#pragma unroll
          for (int k = 0; k < TOP; ++k) {
            const float m = wave_max(z);
            const int bi = choice_lane(m, __ballot(z == m), EXPERTS);
            if (lane == bi) z = -INFINITY;
            if (lane == 0) lds.sel[k] = bi, lds.wt[k] = choice_weight(m);
          }
        }
        meet();
      }
      if (w < 2) {
        nap(kind == PRENORM_MOE ? N_ME : N_M);
        const u32x4_t v = poll.values(t < DC / 4, mine + AT_M + t * 16, t16);
        if (t < DC / 4) *reinterpret_cast<uint2*>(lds.m + t * 4) = pack4(v);
      }
      meet();
    }
    nap(N_PART);
  }
  if (w == 0) {
    res += poll.sum_parts<H>(AT_PART + ((a.n_ops - 1) & 1) * PART, row, a.epoch * PRENORM_STACK_OPS + a.n_ops - 1);
    if (x == 0 && lane < 32) a.x_out[row] = res;
  }
  poll.report(failed, a.fail_dev, a.fail_host, a.epoch);
}

__global__ __launch_bounds__(512, 2) void prenorm_stack_kernel(const PrenormStackArgs a) {
  __shared__ __attribute__((aligned(16))) Lds lds;
  const int b = blockIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (wave < 4) compute_waves(a, lds, b, wave);
  else gather_waves(a, lds, b, wave - 4);
}

}  // namespace

bool prenorm_stack_ssm_ok(const SsmDims& d, int n_out) {
  return d.heads == HEADS && d.vdim == VD && d.vdp == VD && d.groups == GROUPS && d.state == NS && d.np == NS && d.norm_groups == GROUPS && d.taps == TAPS && n_out == INNER;
}
bool prenorm_stack_dense_ok(int ff) { return ff == FF; }
bool prenorm_stack_moe_ok(int experts, int top, int ff, int shared_ff) { return experts == EXPERTS && top == TOP && ff == EFF && shared_ff == SFF; }
bool prenorm_stack_width_ok(int64_t ld, int width) { return ld == H && width == H; }
void launch_prenorm_stack(const PrenormStackArgs& a, hipStream_t st) { hipLaunchKernelGGL(prenorm_stack_kernel, dim3(DECODE_STACK_BLOCKS), dim3(512), 0, st, a); }

}  // namespace aha
