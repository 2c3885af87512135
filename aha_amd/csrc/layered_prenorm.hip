// The pre-norm stack of layered.hip (AHA_ARCH_VAMATAR): its weights, buffers and layers.
//
//   x = embed[token] * embed_scale                       residual stream: f32
//   per layer:   x = x + mixer(LN1(x)),   x = x + ff(LN2(x))                            LN: weight and bias
//   mixer        a state-space recurrence (kernels_ssm.hip) or latent attention (kernels_latent.hip)
//   ff           gated (silu(gate) * up), or routed experts with a shared one (kernels_moe.hip)
//   logits = cap tanh(head . LN(x) / cap)
//
// Rows, decode and single forms as in layered.hip: a step is a ragged batch; GEMMs over all rows, row kernels between them.  Steps of one token
// per sequence take the recurrence's step kernel and the attention in the latent space, prompts the chunked recurrence and expanded keys and
// values; one token of one sequence goes through matvecs (prenorm_single).  compute_dtype f32: f32 activations and cache, f32 GEMMs, the
// recurrence token by token, attention in the latent space throughout.
#include "layered_model.h"

namespace aha {

namespace {

// rows [r0, r0 + n) x columns [c0, c0 + nc) of a (rows, cols) tensor into dst (pitch ld) at (row0, col0); rows row_step apart in dst, src_step in
// the tensor
int put_sub(aha_model* m, const aha_tensor_view* t, int64_t rows, int64_t cols, int64_t r0, int64_t n, int64_t src_step, int64_t c0, int64_t nc, void* dst,
            int64_t row0, int64_t row_step, int64_t col0, int64_t ld) {
  std::vector<uint16_t> tmp;
  const void* src;
  const int rc = bf16_source(t, rows * cols, tmp, &src);
  if (rc) return rc;
  if (n <= 0) return AHA_OK;
  AHA_HIP_CHECK(hipStreamSynchronize(m->stream));   // (the zero fill)
  AHA_HIP_CHECK(hipMemcpy2D((char*)dst + (size_t)(row0 * ld + col0) * 2, (size_t)(ld * row_step) * 2, (const char*)src + (size_t)(r0 * cols + c0) * 2,
                            (size_t)(cols * src_step) * 2, (size_t)nc * 2, (size_t)n, hipMemcpyDefault));
  return AHA_OK;
}
int upload_f32(aha_model* m, const std::vector<float>& v, const float** out) {
  void* p = nullptr;
  const int rc = dev_alloc(m, std::max<size_t>(v.size(), 4) * 4, &p);
  if (rc) return rc;
  AHA_HIP_CHECK(hipMemcpy(p, v.data(), v.size() * 4, hipMemcpyHostToDevice));
  *out = (const float*)p;
  return AHA_OK;
}
int upload_bf16(aha_model* m, const std::vector<uint16_t>& v, void** out) {
  const int rc = dev_alloc(m, std::max<size_t>(v.size(), 8) * 2, out);
  if (rc) return rc;
  AHA_HIP_CHECK(hipMemcpy(*out, v.data(), v.size() * 2, hipMemcpyHostToDevice));
  return AHA_OK;
}

struct Loader {
  aha_model* m;
  const aha_tensor_view* w;
  size_t nw;
  const aha_tensor_view* t = nullptr;
  int need(const std::string& name) { return need_tensor(w, nw, name, &t); }
  int vec(const std::string& name, int64_t n, int64_t np, void** out) {   // (n) -> bf16 padded with zeros
    const int rc = need(name);
    return rc ? rc : put_matrix(m, t, 1, n, 1, np, out);
  }
  int host(const std::string& name, int64_t n, std::vector<float>* out) {
    int rc = need(name);
    std::vector<uint16_t> h;
    if (rc || (rc = host_bf16(t, n, &h))) return rc;
    out->resize((size_t)n);
    for (int64_t i = 0; i < n; ++i) (*out)[i] = bf_host(h[i]);
    return AHA_OK;
  }
  int norm(const std::string& name, int64_t n, int64_t np, void** wt, void** b) {
    const int rc = vec(name, n, np, wt);
    return rc ? rc : vec(name + ".b", n, np, b);
  }
  // gate / up (ff, H) in alternating blocks of 16 rows of dst (2 ffp, ld); down (H, ff) -> dst (ld rows, ffp)
  int gated(const std::string& p, int ff, int ffp, int H, int64_t ld, void* gu, void* down) {
    for (int up = 0; up < 2; ++up) {
      int rc = need(p + (up ? "up" : "gate"));
      if (rc) return rc;
      for (int r = 0; r < 16 && r < ff; ++r)
        if ((rc = put_sub(m, t, ff, H, r, (ff - r + 15) / 16, 16, 0, H, gu, r + up * 16, 32, 0, ld))) return rc;
    }
    const int rc = need(p + "down");
    return rc ? rc : put_sub(m, t, H, ff, 0, H, 1, 0, ff, down, 0, 1, 0, ffp);
  }
};

bool same_rotation(const RopeCfg& r, const aha_layer_desc& d) { return r.base == d.rope_base && r.dims == d.rope_dims; }

int load_ssm(Loader& L, PWeights& W, const aha_layer_desc& d, const std::string& mx, int H, int64_t ld) {
  aha_model* m = L.m;
  LayeredModel& l = *m->layered;
  SsmDims& s = W.sd;
  s = SsmDims{d.heads, d.vdim, (int)round_up(d.vdim, 16), d.groups, d.state, (int)round_up(d.state, 32), d.norm_groups, d.conv_taps};
  const int inner = s.inner(), real = d.heads * d.vdim, cp = s.cp(), gn = d.groups * d.state, ch = real + 2 * gn, rows = real + ch + d.heads;
  W.c_off = inner;
  W.dt_off = inner + cp;
  W.n_in = (int)round_up(W.dt_off + d.heads, 64);
  int rc;
#define TRY(e) do { if ((rc = (e))) return rc; } while (0)
  TRY(L.need(mx + "in"));
  TRY(new_matrix(m, W.n_in, ld, &W.w_in));
  for (int h = 0; h < d.heads; ++h)
    for (int x = 0; x < 2; ++x)   // z, x
      TRY(put_sub(m, L.t, rows, H, x * real + h * d.vdim, d.vdim, 1, 0, H, W.w_in, x * inner + h * s.vdp, 1, 0, ld));
  for (int g = 0; g < d.groups; ++g)
    for (int x = 0; x < 2; ++x)   // B, C
      TRY(put_sub(m, L.t, rows, H, 2 * real + x * gn + g * d.state, d.state, 1, 0, H, W.w_in, 2 * inner + (x * d.groups + g) * s.np, 1, 0, ld));
  TRY(put_sub(m, L.t, rows, H, real + ch, d.heads, 1, 0, H, W.w_in, W.dt_off, 1, 0, ld));
  // padded channel of a checkpoint channel
  auto chan = [&](int i) {
    if (i < real) return i / d.vdim * s.vdp + i % d.vdim;
    const int j = i - real;
    return inner + j / d.state * s.np + j % d.state;
  };
  std::vector<float> cw, cb, v, pw((size_t)s.taps * cp, 0.f), pb(cp, 0.f);
  TRY(L.host(mx + "conv", (int64_t)ch * s.taps, &cw));
  TRY(L.host(mx + "conv.b", ch, &cb));
  for (int i = 0; i < ch; ++i) {
    pb[chan(i)] = cb[i];
    for (int j = 0; j < s.taps; ++j) pw[(size_t)j * cp + chan(i)] = cw[(size_t)i * s.taps + j];
  }
  TRY(upload_f32(m, pw, &W.sp.conv_w));
  TRY(upload_f32(m, pb, &W.sp.conv_b));
  TRY(L.host(mx + "dt_bias", d.heads, &v));
  TRY(upload_f32(m, v, &W.sp.dt_bias));
  TRY(L.host(mx + "A_log", d.heads, &v));
  for (float& x : v) x = (float)-exp((double)x);
  TRY(upload_f32(m, v, &W.sp.a));
  TRY(L.host(mx + "D", d.heads, &v));
  TRY(upload_f32(m, v, &W.sp.d));
  W.ko = (int)round_up(inner, 64);
  TRY(L.need(mx + "norm"));
  std::vector<uint16_t> nb, npad(W.ko, 0);
  TRY(host_bf16(L.t, real, &nb));
  for (int i = 0; i < real; ++i) npad[chan(i)] = nb[i];
  TRY(upload_bf16(m, npad, &W.gnorm));
  TRY(L.need(mx + "o"));
  TRY(new_matrix(m, ld, W.ko, &W.wo));
  for (int h = 0; h < d.heads; ++h) TRY(put_sub(m, L.t, H, real, 0, H, 1, h * d.vdim, d.vdim, W.wo, 0, 1, h * s.vdp, W.ko));
  W.hist_off = l.hist_slot;
  l.hist_slot += (int64_t)CONV_HISTORIES * (s.taps - 1) * cp;
  W.state_off = l.pool_stride;
  l.pool_stride += s.state_floats();
  l.max_proj = std::max(l.max_proj, W.n_in);
  l.max_cp = std::max(l.max_cp, cp);
  l.max_dt = std::max(l.max_dt, d.heads);
  l.max_yb = std::max(l.max_yb, W.ko);
  l.max_inner = std::max(l.max_inner, inner);
  if (!l.f32 && ssm_chunk_ok(s)) l.seg_floats = std::max(l.seg_floats, ssm_segment_floats(s));
  return AHA_OK;
}

int load_latent(Loader& L, PWeights& W, int li, const std::string& mx, int H, int64_t ld, uint64_t* kv_bytes) {
  aha_model* m = L.m;
  LayeredModel& l = *m->layered;
  const aha_layer_desc& d = m->desc.layers[li];
  LatentDims& a = W.la;
  a.heads = d.heads; a.dim = d.dim; a.rot = d.rope_dims; a.vdim = d.vdim; a.rank = d.kv_rank; a.window = d.window; a.scale = d.scale;
  a.rp = (int)round_up(d.kv_rank, 64);
  W.prefill_ok = latent_prefill_dims(d.dim, d.rope_dims, d.vdim, &a.dp, &a.tp, &a.vp) && !l.f32 && d.scale > 0.f;
  W.decode_ok = !l.f32 && latent_decode_ok(a);
  const bool own = d.kv_from < 0;
  const int nq = d.heads * a.qd(), qd = d.dim + d.rope_dims;
  W.kv_col = own ? nq : -1;
  W.n_q = (int)round_up(nq + (own ? a.rp + a.tp : 0), 64);
  int rc;
  TRY(L.need(mx + "q"));
  TRY(new_matrix(m, W.n_q, ld, &W.w_q));
  for (int h = 0; h < d.heads; ++h) {
    TRY(put_sub(m, L.t, (int64_t)d.heads * qd, H, (int64_t)h * qd, d.dim, 1, 0, H, W.w_q, (int64_t)h * a.qd(), 1, 0, ld));
    TRY(put_sub(m, L.t, (int64_t)d.heads * qd, H, (int64_t)h * qd + d.dim, d.rope_dims, 1, 0, H, W.w_q, (int64_t)h * a.qd() + a.dp, 1, 0, ld));
  }
  if (own) {
    TRY(L.need(mx + "dkv"));
    TRY(put_sub(m, L.t, d.kv_rank + d.rope_dims, H, 0, d.kv_rank, 1, 0, H, W.w_q, nq, 1, 0, ld));
    TRY(put_sub(m, L.t, d.kv_rank + d.rope_dims, H, d.kv_rank, d.rope_dims, 1, 0, H, W.w_q, nq + a.rp, 1, 0, ld));
    TRY(L.vec(mx + "dkv.norm", d.kv_rank, a.rp, &W.dkv_norm));
    W.kv_off = *kv_bytes;
    *kv_bytes += (uint64_t)round_up(KV_PAGE_TOKENS * a.ldc() * (l.f32 ? 4 : 2), 1024);
  } else {
    W.kv_off = l.P[d.kv_from].kv_off;
  }
  // W_uk: per head, transposed, for the queries of the latent space; with W_uv stacked for the expanded keys and values
  std::vector<uint16_t> uk, t((size_t)d.heads * a.rp * a.dp, 0);
  TRY(L.need(mx + "uk"));
  TRY(host_bf16(L.t, (int64_t)d.heads * d.dim * d.kv_rank, &uk));
  for (int h = 0; h < d.heads; ++h)
    for (int i = 0; i < d.dim; ++i)
      for (int j = 0; j < d.kv_rank; ++j) t[((size_t)h * a.rp + j) * a.dp + i] = uk[((size_t)h * d.dim + i) * d.kv_rank + j];
  TRY(upload_bf16(m, t, &W.w_ukt));
  W.n_ukv = (int)round_up((int64_t)d.heads * (a.dp + a.vp), 64);
  TRY(new_matrix(m, W.n_ukv, a.rp, &W.w_ukv));
  for (int h = 0; h < d.heads; ++h) TRY(put_sub(m, L.t, (int64_t)d.heads * d.dim, d.kv_rank, (int64_t)h * d.dim, d.dim, 1, 0, d.kv_rank, W.w_ukv, (int64_t)h * a.dp, 1, 0, a.rp));
  TRY(L.need(mx + "uv"));
  const int64_t v0 = (int64_t)d.heads * a.dp;
  for (int h = 0; h < d.heads; ++h) TRY(put_sub(m, L.t, (int64_t)d.heads * d.vdim, d.kv_rank, (int64_t)h * d.vdim, d.vdim, 1, 0, d.kv_rank, W.w_ukv, v0 + (int64_t)h * a.vp, 1, 0, a.rp));
  W.w_uv = (char*)W.w_ukv + (size_t)v0 * a.rp * 2;   // (heads, vp, rp)
  W.ko = (int)round_up((int64_t)d.heads * a.vp, 64);
  TRY(L.need(mx + "o"));
  TRY(new_matrix(m, ld, W.ko, &W.wo));
  for (int h = 0; h < d.heads; ++h) TRY(put_sub(m, L.t, H, (int64_t)d.heads * d.vdim, 0, H, 1, (int64_t)h * d.vdim, d.vdim, W.wo, 0, 1, (int64_t)h * a.vp, W.ko));
  for (size_t i = 0; i < l.ropes.size(); ++i)
    if (same_rotation(l.ropes[i], d)) W.rope = (int)i;
  if (W.rope < 0) {
    W.rope = (int)l.ropes.size();
    l.ropes.push_back({d.rope_base, d.rope_dims});
  }
  if (W.prefill_ok) {
    const auto it = std::find(l.windows.begin(), l.windows.end(), d.window);
    W.win = (int)(it - l.windows.begin());
    if (it == l.windows.end()) l.windows.push_back(d.window);
    l.max_ldc = std::max(l.max_ldc, a.ldc());
    l.max_ukv = std::max<int64_t>(l.max_ukv, (int64_t)d.heads * (a.dp + a.vp));
  }
  l.max_proj = std::max(l.max_proj, W.n_q);
  l.max_yb = std::max(l.max_yb, W.ko);
  l.max_qa = std::max(l.max_qa, d.heads * std::max(a.rp, a.tp));   // (also holds the rotated queries of a decode step)
  l.max_lat_heads = std::max(l.max_lat_heads, d.heads);
  l.max_rp = std::max(l.max_rp, a.rp);
  return AHA_OK;
}

int load_mlp(Loader& L, PWeights& W, const aha_layer_desc& d, const std::string& p, int H, int64_t ld) {
  aha_model* m = L.m;
  LayeredModel& l = *m->layered;
  const int ff = d.mlp == AHA_MLP_MOE ? d.shared_ff : d.ff;
  int rc;
  W.ep = d.mlp == AHA_MLP_MOE ? (int)round_up(d.experts, 64) : 0;
  W.ffp = ff > 0 ? (int)round_up(ff, 64) : 0;
  if (ff > 0) {
    TRY(new_matrix(m, 2 * W.ffp, ld, &W.wgu));
    TRY(new_matrix(m, ld, W.ffp, &W.wdown));
    TRY(L.gated(p + (d.mlp == AHA_MLP_MOE ? "shared." : ""), ff, W.ffp, H, ld, W.wgu, W.wdown));
    l.max_ffp = std::max(l.max_ffp, W.ffp);
  }
  if (d.mlp != AHA_MLP_MOE) return AHA_OK;
  W.effp = (int)round_up(d.ff, 64);
  TRY(L.need(p + "router"));
  TRY(new_matrix(m, W.ep, ld, &W.w_router));
  TRY(put_sub(m, L.t, d.experts, H, 0, d.experts, 1, 0, H, W.w_router, 0, 1, 0, ld));
  TRY(new_matrix(m, (int64_t)d.experts * 2 * W.effp, ld, &W.w_egu));
  TRY(new_matrix(m, (int64_t)d.experts * ld, W.effp, &W.w_edown));
  for (int e = 0; e < d.experts; ++e)
    TRY(L.gated(p + "e" + std::to_string(e) + ".", d.ff, W.effp, H, ld, (char*)W.w_egu + (size_t)e * 2 * W.effp * ld * 2, (char*)W.w_edown + (size_t)e * ld * W.effp * 2));
  l.max_ep = std::max(l.max_ep, W.ep);
  l.max_effp = std::max(l.max_effp, W.effp);
  l.max_slots = std::max(l.max_slots, d.top);
  return AHA_OK;
}
#undef TRY

SsmHist ssm_hist(const LayeredModel& l, const PWeights& W) { return SsmHist{l.d_hist + W.hist_off, l.hist_slot}; }
SsmState ssm_state(const LayeredModel& l, const PWeights& W) { return SsmState{l.d_pool + W.state_off, l.pool_stride}; }
LatentCache latent_cache(const LayeredModel& l, const PWeights& W) { return LatentCache{l.d_tab, (int64_t)l.tab_ld, W.kv_off}; }

// KV splits of a decode launch: at least two 32-position tiles per block, the blocks in one round over the CUs, and none without a tile (129 tiles are 43
// blocks of three, not 64).  Four tiles per block, one a wave, read their keys through too few CUs: 7.2 -> 8.0 us at 4096 positions, 5.1 -> 4.4 for the join.
int latent_splits(const LatentDims& d, const SeqEntry* e, int n) {
  int nt = 1;
  for (int i = 0; i < n; ++i) nt = std::max(nt, (e[i].pos0 >> 5) - (d.first(e[i].pos0) >> 5) + 1);
  const int round = 256 * latent_decode_blocks_per_cu(d);
  const int most = std::max(1, std::min({LATENT_MAX_SPLIT, (nt + 1) / 2, round / std::max(1, n * ((d.heads + 15) / 16))})), per = (nt + most - 1) / most;
  return (nt + per - 1) / per;
}

// mixer over the rows of a step: h -> y
void ssm_rows(aha_model* m, const PWeights& W, const SeqBatch& b) {
  LayeredModel& l = *m->layered;
  const float eps = m->desc.rms_norm_eps;
  hipStream_t st = m->stream;
  const int rows = b.rows;
  const double es = l.f32 ? 4.0 : 2.0;
  gemm(m, l.h, l.ld, W.w_in, l.proj, W.n_in, rows, W.n_in, (int)l.ld);
  const SsmIn in{l.proj, W.n_in, W.c_off, W.dt_off};
  GatedNormArgs g{};
  g.d = W.sd; g.w = W.gnorm; g.out = l.ob; g.ldo = W.ko; g.eps = eps; g.rows = rows;
  if (b.max_len == 1 && !l.f32 && ssm_chunk_ok(W.sd)) {
    SsmStepArgs s{};
    s.d = W.sd; s.in = in; s.in_f32 = 0; s.p = W.sp; s.h = ssm_hist(l, W); s.s = ssm_state(l, W); s.g = (float*)l.u; s.ssq = l.ssq;
    {
      ProfScope ps(m, "ssm", (double)rows * (W.sd.state_floats() * 8.0 + W.n_in * es), 0);
      launch_ssm_step(s, b, st);
    }
    g.y = l.u; g.ldy = W.sd.inner();
  } else {
    ShortConvArgs c{};
    c.d = W.sd; c.in = in; c.p = W.sp; c.h = ssm_hist(l, W); c.u = l.u; c.dt = l.dt; c.dt_ld = rows;
    {
      ProfScope ps(m, "elem", (double)rows * W.sd.cp() * 2 * es, 0);
      launch_short_conv(c, b, l.f32, st);
    }
    SsmScanArgs s{};
    s.d = W.sd; s.p = W.sp; s.s = ssm_state(l, W); s.u = l.u; s.dt = l.dt; s.dt_ld = rows; s.y = l.yb; s.ldy = W.ko;
    {
      ProfScope ps(m, "ssm", (double)rows * (W.sd.cp() + W.sd.inner()) * es, 4.0 * rows * W.sd.heads * W.sd.vdp * W.sd.np);
      if (!l.f32 && ssm_chunk_ok(W.sd)) launch_ssm_chunks(s, b, l.seg, l.seg_floats, st);
      else launch_ssm_scan(s, b, l.f32, st);
    }
    g.y = l.yb; g.ldy = W.ko; g.z = l.proj; g.ldz = W.n_in;
  }
  {
    ProfScope ps(m, "elem", (double)rows * W.sd.inner() * 3 * es, 0);
    launch_gated_norm(g, l.f32, st);
  }
  gemm(m, l.ob, W.ko, W.wo, l.y, l.ld, rows, (int)l.ld, W.ko);
}

LatentPostArgs latent_post(aha_model* m, const PWeights& W, void* in, bool in_f32) {
  LayeredModel& l = *m->layered;
  LatentPostArgs p{};
  p.d = W.la; p.in = in; p.ld = W.n_q; p.kv_off = W.kv_col; p.in_f32 = in_f32; p.norm_w = W.dkv_norm; p.eps = m->desc.rms_norm_eps; p.rope = l.ropetab[W.rope];
  p.q = in; p.ldq = W.n_q; p.c = latent_cache(l, W);
  return p;
}

// one token per sequence: q | latent | key part -> values of the attention (l.ob)
void latent_decode(aha_model* m, const PWeights& W, const SeqBatch& b, const SeqEntry* h_ents, const LatentPostArgs& p) {
  LayeredModel& l = *m->layered;
  hipStream_t st = m->stream;
  const LatentDims& d = W.la;
  LatentQueryArgs q{};
  q.p = p; q.w_ukt = W.w_ukt; q.qa = l.qa; q.qr = l.yb;
  {
    ProfScope ps(m, "gemv", (double)d.heads * d.rp * d.dp * 2, 2.0 * b.n * d.heads * d.rp * d.dp);
    launch_latent_query(q, b, st);
  }
  LatentDecodeArgs a{};
  a.d = d; a.qa = l.qa; a.qr = l.yb; a.c = p.c; a.part_o = l.part_o; a.part_ml = l.part_ml; a.nsplit = latent_splits(d, h_ents, b.n);
  double keys = 0;
  for (int i = 0; i < b.n; ++i) keys += h_ents[i].pos0 - d.first(h_ents[i].pos0) + 1;
  {
    ProfScope ps(m, "attn_decode", keys * d.ldc() * 2, 2.0 * keys * d.heads * (d.ldc() + d.rp));
    launch_latent_decode(a, b, st);
  }
  const bool fused = b.n <= 4;   // W_uv with the join; more sequences: their joined latents first, so that W_uv is read once
  LatentMergeArgs g{};
  g.d = d; g.part_o = l.part_o; g.part_ml = l.part_ml; g.nsplit = a.nsplit; g.n = b.n; g.ldo = W.ko;
  g.wuv = fused ? W.w_uv : nullptr;
  g.o = fused ? l.ob : l.yb;
  const double wb = (double)d.heads * d.rp * d.vp;
  {
    ProfScope ps(m, "gemv", fused ? wb * 2 : 0, fused ? 2.0 * b.n * wb : 0);
    launch_latent_merge(g, st);
  }
  if (fused) return;
  HeadsGemmArgs u{};
  u.A = l.yb; u.lda = (int64_t)d.heads * d.rp; u.sa = d.rp; u.W = W.w_uv; u.C = l.ob; u.ldc = W.ko; u.sc = d.vp; u.rows = b.n; u.heads = d.heads; u.n = d.vp; u.k = d.rp;
  ProfScope ps(m, "gemm", wb * 2, 2.0 * b.n * wb);
  launch_heads_gemm(u, false, st);
}

void latent_rows(aha_model* m, const PWeights& W, const SeqBatch& b, const SeqEntry* h_ents) {
  LayeredModel& l = *m->layered;
  hipStream_t st = m->stream;
  const LatentDims& d = W.la;
  const int rows = b.rows;
  const double es = l.f32 ? 4.0 : 2.0;
  gemm(m, l.h, l.ld, W.w_q, l.proj, W.n_q, rows, W.n_q, (int)l.ld);
  LatentPostArgs p = latent_post(m, W, l.proj, l.f32);
  if (b.max_len == 1 && W.decode_ok) {
    latent_decode(m, W, b, h_ents, p);
    gemm(m, l.ob, W.ko, W.wo, l.y, l.ld, rows, (int)l.ld, W.ko);
    return;
  }
  {
    ProfScope ps(m, "elem", (double)rows * (d.heads * d.tp + d.ldc()) * 2 * es, 0);
    launch_latent_post(p, b, l.f32, st);
  }
  if (b.max_len > 1 && W.prefill_ok) {
    const int32_t* ext0 = l.ext_dev + (size_t)W.win * b.n;
    const int total = l.ext_total[W.win];
    {
      ProfScope ps(m, "elem", (double)total * d.ldc() * 2 * es, 0);
      launch_latent_gather(d, p.c, ext0, l.lat, b, l.ext_max[W.win], false, st);
    }
    gemm(m, l.lat, d.ldc(), W.w_ukv, l.ukv, (int64_t)d.heads * (d.dp + d.vp), total, d.heads * (d.dp + d.vp), d.rp);
    LatentPrefillArgs a{};
    a.d = d; a.q = l.proj; a.ldq = W.n_q; a.kv = l.ukv; a.lat = l.lat; a.ext0 = ext0; a.o = l.ob; a.ldo = W.ko;
    double pairs = 0;
    for (int i = 0; i < b.n; ++i) {
      const double s = h_ents[i].len, w = d.window > 0 ? d.window : 1e18, first = std::max(0.0, std::min(s, w - h_ents[i].pos0));   // rows that see everything in front of them
      pairs += first * (h_ents[i].pos0 + 0.5 * first) + (s - first) * w;
    }
    ProfScope ps(m, "attn_prefill", (double)rows * d.heads * (d.qd() + d.vp) * es, 2.0 * pairs * d.heads * (d.dim + d.rot + d.vdim));
    launch_latent_prefill(a, b, st);
  } else {
    HeadsGemmArgs g{};
    g.A = l.proj; g.lda = W.n_q; g.sa = d.qd(); g.W = W.w_ukt; g.C = l.qa; g.ldc = (int64_t)d.heads * d.rp; g.sc = d.rp; g.rows = rows; g.heads = d.heads; g.n = d.rp; g.k = d.dp;
    {
      ProfScope ps(m, "gemm", (double)d.heads * d.rp * d.dp * 2, 2.0 * rows * d.heads * d.rp * d.dp);
      launch_heads_gemm(g, l.f32, st);
    }
    LatentRowsArgs a{};
    a.d = d; a.qa = l.qa; a.q = l.proj; a.ldq = W.n_q; a.o = l.yb; a.c = p.c;
    {
      ProfScope ps(m, "attn_prefill", 0, 0);
      launch_latent_rows(a, b, l.f32, st);
    }
    g.A = l.yb; g.lda = (int64_t)d.heads * d.rp; g.sa = d.rp; g.W = W.w_uv; g.C = l.ob; g.ldc = W.ko; g.sc = d.vp; g.n = d.vp; g.k = d.rp;
    ProfScope ps(m, "gemm", (double)d.heads * d.rp * d.vp * 2, 2.0 * rows * d.heads * d.rp * d.vp);
    launch_heads_gemm(g, l.f32, st);
  }
  gemm(m, l.ob, W.ko, W.wo, l.y, l.ld, rows, (int)l.ld, W.ko);
}

void gated_rows(aha_model* m, const PWeights& W, int rows) {
  LayeredModel& l = *m->layered;
  if (l.f32) {
    gemm(m, l.h, l.ld, W.wgu, l.gu, 2 * W.ffp, rows, 2 * W.ffp, (int)l.ld);
    launch_silu_pairs(l.gu, 2 * W.ffp, (float*)l.act, W.ffp, rows, W.ffp, nullptr, m->stream);
  } else {
    gemm(m, l.h, l.ld, W.wgu, l.act, W.ffp, rows, 2 * W.ffp, (int)l.ld, ACT_SILU_MUL_PAIRS);
  }
  gemm(m, l.act, W.ffp, W.wdown, l.y, l.ld, rows, (int)l.ld, W.ffp);
}

PendingAdd moe_rows(aha_model* m, const PWeights& W, const aha_layer_desc& d, int rows) {
  LayeredModel& l = *m->layered;
  hipStream_t st = m->stream;
  const int slots = rows * d.top, bm = moe_tile_rows(slots, d.experts, l.f32);
  gemm(m, l.h, l.ld, W.w_router, l.zr, W.ep, rows, W.ep, (int)l.ld, ACT_PARTIAL_F32);
  {
    ProfScope ps(m, "elem", (double)rows * W.ep * 4, 0);
    launch_moe_route(l.zr, W.ep, rows, d.experts, d.top, bm, l.route, st);
  }
  const double es = l.f32 ? 4.0 : 2.0, used = std::min(d.experts, slots);
  MoeGemmArgs g{};
  g.A = l.h; g.lda = l.ld; g.W = W.w_egu; g.n = 2 * W.effp; g.k = (int)l.ld; g.slots = slots; g.experts = d.experts; g.gather = 1; g.pairs = 1;
  g.C = l.f32 ? (void*)l.egu : l.eact; g.ldc = l.f32 ? 2 * W.effp : W.effp;
  {
    ProfScope ps(m, "moe", used * g.n * g.k * 2.0 + slots * (g.k + W.effp) * es, 2.0 * slots * g.n * g.k);
    launch_moe_gemm(g, l.route, bm, l.f32, st);
  }
  if (l.f32) launch_silu_pairs(l.egu, 2 * W.effp, (float*)l.eact, W.effp, slots, W.effp, l.route.slot_w, st);
  g.A = l.eact; g.lda = W.effp; g.W = W.w_edown; g.C = l.ey; g.ldc = l.ld; g.n = (int)l.ld; g.k = W.effp; g.gather = 0; g.pairs = 0;
  {
    ProfScope ps(m, "moe", used * g.n * g.k * 2.0 + slots * (g.k + g.n) * es, 2.0 * slots * g.n * g.k);
    launch_moe_gemm(g, l.route, bm, l.f32, st);
  }
  PendingAdd p;
  p.slots = l.ey; p.slot_of = l.route.slot_of; p.top = d.top; p.ld_slots = l.ld;
  if (W.ffp > 0) {
    gated_rows(m, W, rows);
    p.y = l.y; p.ldy = l.ld;
  }
  return p;
}

}  // namespace

int prenorm_check(const aha_model_desc& c) {
  if (c.hidden_size <= 0 || c.vocab_size <= 0 || c.num_hidden_layers <= 0 || c.num_hidden_layers > AHA_MAX_LAYERS || c.n_stop_tokens < 0 || c.n_stop_tokens > 8 ||
      c.logit_softcap < 0.f)
    return err(AHA_ERR_INVALID, "model_create: sizes must be positive (at most 256 layers, 8 stop tokens)");
  if (c.hidden_size > 8192) return err(AHA_ERR_UNSUPPORTED, "hidden_size above 8192");
  if (c.tp_size > 1) return err(AHA_ERR_UNSUPPORTED, "this architecture runs on one GPU (tp_size 1)");
  for (int i = 0; i < c.num_hidden_layers; ++i) {
    const aha_layer_desc& l = c.layers[i];
    const std::string at = "layer " + std::to_string(i) + ": ";
    if (l.mixer == AHA_MIXER_MAMBA2) {
      if (l.heads <= 0 || l.vdim <= 0 || l.state <= 0 || l.groups <= 0 || l.heads % l.groups || l.norm_groups <= 0 || l.conv_taps < 1 || (int64_t)l.heads * l.vdim % l.norm_groups)
        return err(AHA_ERR_INVALID, at + "inconsistent sizes");
      if (round_up(l.state, 32) > 2048 || (round_up(l.vdim, 16) * l.heads + l.norm_groups) * 4 > 160 * 1024) return err(AHA_ERR_UNSUPPORTED, at + "state or inner width exceeds the kernels' LDS");
    } else if (l.mixer == AHA_MIXER_LATENT) {
      if (l.heads <= 0 || l.dim <= 0 || l.vdim <= 0 || l.kv_rank <= 0 || l.rope_dims <= 0 || l.rope_dims % 2 || l.window < 0 || !(l.rope_base > 0.0) || l.kv_from >= i)
        return err(AHA_ERR_INVALID, at + "inconsistent sizes");
      if (l.kv_rank > 1024) return err(AHA_ERR_UNSUPPORTED, at + "kv_rank above 1024");
      if (l.kv_from >= 0) {
        const aha_layer_desc& s = c.layers[l.kv_from];
        if (s.mixer != AHA_MIXER_LATENT || s.kv_from >= 0 || s.kv_rank != l.kv_rank || s.rope_dims != l.rope_dims || s.rope_base != l.rope_base)
          return err(AHA_ERR_INVALID, at + "kv_from must name an earlier latent attention layer with a cache of its own and the same kv_rank and rotation");
      }
    } else {
      return err(AHA_ERR_UNSUPPORTED, at + "unknown mixer");
    }
    if (l.mlp != AHA_MLP_NONE && l.mlp != AHA_MLP_GATED && l.mlp != AHA_MLP_MOE) return err(AHA_ERR_UNSUPPORTED, at + "unknown feed-forward");
    if ((l.mlp != AHA_MLP_NONE && l.ff <= 0) || (l.mlp == AHA_MLP_MOE && (l.experts <= 0 || l.top <= 0 || l.top > l.experts || l.shared_ff < 0)))
      return err(AHA_ERR_INVALID, at + "inconsistent feed-forward sizes");
    if (l.mlp == AHA_MLP_MOE && l.experts > 1024) return err(AHA_ERR_UNSUPPORTED, at + "more than 1024 experts");
  }
  return AHA_OK;
}

int prenorm_create(aha_model* m, const aha_tensor_view* w, size_t nw, uint64_t* kv_bytes) {
  LayeredModel& l = *m->layered;
  const aha_model_desc& c = m->desc;
  Loader L{m, w, nw};
  l.P.resize(c.num_hidden_layers);
  for (int li = 0; li < c.num_hidden_layers; ++li) {
    PWeights& W = l.P[li];
    const aha_layer_desc& d = c.layers[li];
    const std::string p = "l" + std::to_string(li) + ".";
    int rc = L.norm(p + "norm1", c.hidden_size, l.ld, &W.n1w, &W.n1b);
    if (!rc) rc = d.mixer == AHA_MIXER_MAMBA2 ? load_ssm(L, W, d, p + "mix.", c.hidden_size, l.ld) : load_latent(L, W, li, p + "mix.", c.hidden_size, l.ld, kv_bytes);
    if (!rc && d.mlp != AHA_MLP_NONE) {
      rc = L.norm(p + "norm2", c.hidden_size, l.ld, &W.n2w, &W.n2b);
      if (!rc) rc = load_mlp(L, W, d, p + "mlp.", c.hidden_size, l.ld);
    }
    if (rc) return rc;
  }
  return l.seg_floats ? dev_alloc(m, l.seg_floats * 4, (void**)&l.seg) : AHA_OK;
}

int prenorm_ensure_rows(aha_model* m, size_t cap) {
  LayeredModel& l = *m->layered;
  const size_t es = l.f32 ? 4 : 2;
  int rc;
  auto al = [&](size_t bytes, void** out) { return grow(m, l.row_bufs, bytes, out); };
  const size_t yb = std::max<size_t>(l.max_yb, l.max_qa);
  if ((rc = al(cap * l.ld * 4, (void**)&l.xa)) || (rc = al(cap * l.ld * 4, (void**)&l.xb)) || (rc = al(cap * l.ld * es, &l.h)) || (rc = al(cap * l.max_proj * es, &l.proj)) ||
      (rc = al(cap * std::max<size_t>(l.max_cp * es, (size_t)l.max_inner * 4), &l.u)) || (rc = al(cap * std::max(l.max_dt, 1) * 4, (void**)&l.dt)) ||
      (rc = al(cap * std::max(l.max_inner / 16, 1) * 4, (void**)&l.ssq)) || (rc = al(cap * yb * es, &l.yb)) || (rc = al(cap * l.max_yb * es, &l.ob)) ||
      (rc = al(cap * std::max(l.max_qa, 1) * es, &l.qa)) || (rc = al(cap * std::max(l.max_ffp, 64) * es, &l.act)) || (rc = al(cap * l.ld * es, &l.y)) ||
      (rc = al(cap * std::max(l.max_ep, 1) * 4, (void**)&l.zr)))
    return rc;
  const size_t slots = cap * std::max(l.max_slots, 0);
  if ((rc = al(slots * l.max_effp * es, &l.eact)) || (rc = al(slots * l.ld * es, &l.ey))) return rc;
  if (l.f32 && ((rc = al(cap * 2 * std::max(l.max_ffp, 1) * 4, (void**)&l.gu)) || (rc = al(slots * 2 * l.max_effp * 4, (void**)&l.egu)))) return rc;
  if (l.max_slots > 0) {
    const size_t tiles = slots / 16 + 1 + std::min<size_t>(l.max_ep, slots);
    int32_t* p = nullptr;
    if ((rc = al((2 * (size_t)l.max_ep + 5 * slots + 3 * tiles + 64) * 4, (void**)&p))) return rc;
    MoeRouting& r = l.route;
    r.counts = p; r.cursor = p + l.max_ep; p += 2 * l.max_ep;
    r.sel = p; r.slot_of = p + slots; r.slot_row = p + 2 * slots; r.sel_w = (float*)(p + 3 * slots); r.slot_w = (float*)(p + 4 * slots);
    r.tiles = p + 5 * slots; r.n_tiles = r.tiles + 3 * tiles;
  }
  return AHA_OK;
}

int prenorm_ensure_entries(aha_model* m, size_t cap) {
  LayeredModel& l = *m->layered;
  if (l.max_lat_heads == 0) return AHA_OK;
  const size_t parts = std::max<size_t>(cap, 512) * (size_t)l.max_lat_heads;   // splits x sequences x head groups <= max(512, sequences x head groups)
  int rc = grow(m, l.ent_bufs, parts * l.max_rp * 4, (void**)&l.part_o);
  return rc ? rc : grow(m, l.ent_bufs, parts * 2 * 4, (void**)&l.part_ml);
}

// where the gathered cache rows of every entry start, per distinct window
int prenorm_prepare_ext(aha_model* m, const SeqEntry* e, size_t n, int32_t* host_out) {
  LayeredModel& l = *m->layered;
  l.ext_total.assign(l.windows.size(), 0);
  l.ext_max.assign(l.windows.size(), 0);
  size_t most = 0;
  for (size_t w = 0; w < l.windows.size(); ++w) {
    LatentDims d{};
    d.window = l.windows[w];
    int64_t at = 0;
    for (size_t i = 0; i < n; ++i) {
      const int len = e[i].pos0 + e[i].len - (d.first(e[i].pos0) & ~(KV_PAGE_TOKENS - 1));
      host_out[w * n + i] = (int32_t)at;
      at += len;
      l.ext_max[w] = std::max(l.ext_max[w], len);
    }
    if (at > (1 << 24)) return err(AHA_ERR_INVALID, "forward_batch: too many cached rows in one step");
    l.ext_total[w] = (int)at;
    most = std::max(most, (size_t)at);
  }
  if (most <= l.ext_cap) return AHA_OK;
  int rc = free_list(m, l.ext_bufs);
  if (rc) return rc;
  l.ext_cap = 0;
  const size_t cap = (size_t)round_up((int64_t)most, 256);
  if ((rc = grow(m, l.ext_bufs, cap * l.max_ldc * 2, &l.lat)) || (rc = grow(m, l.ext_bufs, cap * l.max_ukv * 2, &l.ukv))) return rc;
  l.ext_cap = cap;
  return AHA_OK;
}

// can every layer take the matvec form (one token of one sequence, bf16)?
bool prenorm_single_ok(const aha_model* m) {
  const LayeredModel& l = *m->layered;
  constexpr int KMAX = 15872;   // 64 KB of LDS for the input vector
  if (l.f32 || l.ld > 8192) return false;
  for (int i = 0; i < m->desc.num_hidden_layers; ++i) {
    const PWeights& W = l.P[i];
    const aha_layer_desc& d = m->desc.layers[i];
    if (W.ko > KMAX || W.ffp > KMAX) return false;
    if (d.mixer == AHA_MIXER_MAMBA2 && (!ssm_chunk_ok(W.sd) || d.heads % d.norm_groups || d.norm_groups > 400)) return false;
    if (d.mixer == AHA_MIXER_LATENT && !W.decode_ok) return false;
    if (d.mlp == AHA_MLP_MOE && (d.top >= 64 || (int64_t)d.top * W.effp + W.ffp > KMAX)) return false;
  }
  return true;
}
static int prenorm_schedule(aha_model* m);
int prenorm_alloc_single(aha_model* m) {
  LayeredModel& l = *m->layered;
  int rc = dev_alloc(m, (size_t)std::max(l.max_proj, 1) * 4, (void**)&l.qkv1, true);
  if (!rc) rc = dev_alloc(m, (size_t)std::max(l.max_ep, 64) * 4, (void**)&l.z1, true);
  if (!rc) rc = dev_alloc(m, (size_t)(l.max_slots * l.max_effp + l.max_ffp + 64) * 2, &l.act1, true);
  if (!rc && l.single_ok) rc = prenorm_schedule(m);
  return rc;
}

// Halves of layers that follow each other and that the kernel takes run as one launch; a half alone is no faster there (its weights are cold).
static int prenorm_schedule(aha_model* m) {
  LayeredModel& l = *m->layered;
  std::vector<PrenormOp> ops;
  l.schedule.clear();
  auto add = [&](int li, int half, const PrenormOp* op, double weights = 0, double states = 0) {
    if (op && !l.schedule.empty() && l.schedule.back().first >= 0 && l.schedule.back().n < PRENORM_STACK_OPS) ++l.schedule.back().n;
    else l.schedule.push_back({li, half, op ? (int)ops.size() : -1, op ? 1 : 0, 0, 0});
    l.schedule.back().weights += weights;
    l.schedule.back().states += states;
    if (op) ops.push_back(*op);
  };
  bool have = false;
  if (prenorm_stack_width_ok(l.ld, m->desc.hidden_size))
    if (int rc = model_stack_alloc(m, &have)) return rc;
  for (int li = 0; li < m->desc.num_hidden_layers; ++li) {
    const PWeights& W = l.P[li];
    const aha_layer_desc& d = m->desc.layers[li];
    PrenormOp op{};
    op.nw = W.n1w; op.nb = W.n1b;
    if (have && d.mixer == AHA_MIXER_MAMBA2 && prenorm_stack_ssm_ok(W.sd, W.ko)) {
      l.stack_hist = (int64_t)(W.sd.taps - 1) * W.sd.cp();   // (one geometry)
      op.kind = PRENORM_SSM; op.w1 = W.w_in; op.w2 = W.wo; op.gnorm = W.gnorm; op.hist = W.hist_off; op.state = W.state_off;
      const size_t cp = W.sd.cp(), taps = W.sd.taps, heads = W.sd.heads;
      void* p = nullptr;
      if (int rc = dev_alloc(m, ((taps + 1) * cp + 3 * heads) * 4, &p)) return rc;
      float* at = (float*)p;
      op.par = at;
      auto put = [&](const float* src, size_t n) {
        const hipError_t e = hipMemcpy(at, src, n * 4, hipMemcpyDeviceToDevice);
        at += n;
        return e == hipSuccess;
      };
      if (!put(W.sp.conv_w, taps * cp) || !put(W.sp.conv_b, cp) || !put(W.sp.dt_bias, heads) || !put(W.sp.a, heads) || !put(W.sp.d, heads))
        return err(AHA_ERR_HIP, "model_create: copying the mixers' parameters failed");
      add(li, 0, &op, (double)l.ld * (W.n_in + W.ko), W.sd.state_floats());
    } else {
      add(li, 0, nullptr);
    }
    if (d.mlp == AHA_MLP_NONE) continue;
    op = PrenormOp{};
    op.nw = W.n2w; op.nb = W.n2b; op.w1 = W.wgu; op.w2 = W.wdown;
    if (have && d.mlp == AHA_MLP_GATED && prenorm_stack_dense_ok(W.ffp)) {
      op.kind = PRENORM_DENSE;
      add(li, 1, &op, 3.0 * l.ld * W.ffp);
    } else if (have && d.mlp == AHA_MLP_MOE && prenorm_stack_moe_ok(d.experts, d.top, W.effp, W.ffp)) {
      op.kind = PRENORM_MOE; op.router = W.w_router; op.egu = W.w_egu; op.edown = W.w_edown;
      add(li, 1, &op, (double)l.ld * (d.experts + 3.0 * d.top * W.effp + 3.0 * W.ffp));
    } else {
      add(li, 1, nullptr);
    }
  }
  if (ops.empty()) return AHA_OK;
  void* p = nullptr;
  if (int rc = dev_alloc(m, ops.size() * sizeof(PrenormOp), &p)) return rc;
  l.d_ops = (PrenormOp*)p;
  AHA_HIP_CHECK(hipMemcpy(p, ops.data(), ops.size() * sizeof(PrenormOp), hipMemcpyHostToDevice));
  return AHA_OK;
}

// one token of one sequence: matvecs whose prologue is the norm in front of the projection.  Per layer three launches (state space) or five
// (attention), then two (dense) or three (experts)
static Tail prenorm_single(aha_model* m, const SeqBatch& b, const uint32_t* ids) {
  LayeredModel& l = *m->layered;
  const aha_model_desc& c = m->desc;
  hipStream_t st = m->stream;
  const float eps = c.rms_norm_eps;
  for (size_t i = 0; i < l.ropes.size(); ++i) launch_rope_pairs(b, l.ropes[i].base, l.ropes[i].dims, l.ropetab[i], st);
  {
    PreNormArgs a{};
    a.embed = l.embed; a.ids = ids; a.embed_scale = c.embed_scale; a.x_out = l.xa; a.width = c.hidden_size; a.rows = 1; a.ld = l.ld;
    launch_prenorm_rows(a, false, st);
  }
  auto bytes = [](double n, double k) { return n * k * 2 + k * 4 + n * 4; };
  auto ln = [&](const void* w, const void* bias) { return GemvLayerNorm{l.xa, w, bias, eps, c.hidden_size}; };
  auto args = [&](const void* W, int n, int k, float* y) {
    GemvArgs g{};
    g.W = W; g.N = n; g.K = k; g.y_f32 = y; g.eps = eps; g.res_f32 = l.xa; g.res_scale = 1.f;
    return g;
  };
  auto mixer = [&](int li) {
    const PWeights& W = l.P[li];
    const aha_layer_desc& d = c.layers[li];
    if (d.mixer == AHA_MIXER_MAMBA2) {
      GemvArgs g = args(W.w_in, W.n_in, (int)l.ld, l.qkv1);
      {
        ProfScope ps(m, "gemv", bytes(g.N, g.K), 2.0 * g.N * g.K);
        launch_gemv_layernorm(g, ln(W.n1w, W.n1b), GEMV_PARTIAL_F32, st);
      }
      SsmStepArgs s{};
      s.d = W.sd; s.in = SsmIn{l.qkv1, W.n_in, W.c_off, W.dt_off}; s.in_f32 = 1; s.p = W.sp; s.h = ssm_hist(l, W); s.s = ssm_state(l, W); s.g = (float*)l.u; s.ssq = l.ssq;
      {
        ProfScope ps(m, "ssm", W.sd.state_floats() * 8.0 + W.n_in * 4.0, 0);
        launch_ssm_step(s, b, st);
      }
      g = args(W.wo, (int)l.ld, W.ko, l.xa);
      ProfScope ps(m, "gemv", bytes(g.N, g.K), 2.0 * g.N * g.K);
      launch_gemv_partsnorm(g, GemvPartsNorm{(const float*)l.u, l.ssq, W.gnorm, eps, W.sd.inner(), d.norm_groups, d.heads * d.vdim / d.norm_groups}, st);
    } else {
      GemvArgs g = args(W.w_q, W.n_q, (int)l.ld, l.qkv1);
      {
        ProfScope ps(m, "gemv", bytes(g.N, g.K), 2.0 * g.N * g.K);
        launch_gemv_layernorm(g, ln(W.n1w, W.n1b), GEMV_PARTIAL_F32, st);
      }
      latent_decode(m, W, b, &b.one, latent_post(m, W, l.qkv1, true));
      g = args(W.wo, (int)l.ld, W.ko, l.xa);
      g.x = l.ob;
      ProfScope ps(m, "gemv", bytes(g.N, g.K), 2.0 * g.N * g.K);
      launch_gemv(g, GEMV_AXPY_F32, st);
    }
  };
  auto feed_forward = [&](int li) {
    const PWeights& W = l.P[li];
    const aha_layer_desc& d = c.layers[li];
    if (d.mlp == AHA_MLP_GATED) {
      GemvArgs g = args(W.wgu, W.ffp, (int)l.ld, nullptr);
      g.y = l.act;
      {
        ProfScope ps(m, "gemv", bytes(2.0 * g.N, g.K), 4.0 * g.N * g.K);
        launch_gemv_layernorm(g, ln(W.n2w, W.n2b), GEMV_SILU_MUL, st);
      }
      g = args(W.wdown, (int)l.ld, W.ffp, l.xa);
      g.x = l.act;
      ProfScope ps(m, "gemv", bytes(g.N, g.K), 2.0 * g.N * g.K);
      launch_gemv(g, GEMV_AXPY_F32, st);
    } else if (d.mlp == AHA_MLP_MOE) {
      GemvArgs g = args(W.w_router, W.ep, (int)l.ld, l.z1);
      {
        ProfScope ps(m, "gemv", bytes(g.N, g.K), 2.0 * g.N * g.K);
        launch_gemv_layernorm(g, ln(W.n2w, W.n2b), GEMV_PARTIAL_F32, st);
      }
      const GemvExperts e{l.z1, W.w_egu, W.wgu, d.experts, d.top, W.effp, l.route.sel};
      const int k = d.top * W.effp + W.ffp;
      g = args(nullptr, k, (int)l.ld, nullptr);
      g.y = l.act1;
      {
        ProfScope ps(m, "moe", bytes(2.0 * g.N, g.K), 4.0 * g.N * g.K);
        launch_gemv_experts_up(g, ln(W.n2w, W.n2b), e, st);
      }
      g = args(nullptr, (int)l.ld, k, l.xa);
      g.x = l.act1;
      ProfScope ps(m, "moe", bytes(g.N, g.K), 2.0 * g.N * g.K);
      launch_gemv_experts_down(g, GemvExpertsDown{W.w_edown, W.wdown, e.sel, d.top, W.effp, W.ffp, (int)l.ld}, st);
    }
  };
  // (the recurrence of a run that gave up is run again: its states must not have been written over)
  StackTurn turn;
  const bool stacked = l.d_ops && !l.keep && b.one.state_in != b.one.state_out && turn.take(m, false);
  if (!stacked) {
    for (int li = 0; li < c.num_hidden_layers; ++li) {
      mixer(li);
      feed_forward(li);
      keep_rows(m, l.xa, 1, li);
    }
    return Tail{l.xa, nullptr, nullptr, 1.f, {}};
  }
  for (const LayeredModel::StackItem& it : l.schedule) {
    if (it.n < 2) {
      if (it.half == 0) mixer(it.layer);
      else feed_forward(it.layer);
      continue;
    }
    PrenormStackArgs p{};
    p.ops = l.d_ops + it.first; p.n_ops = it.n; p.x_in = p.x_out = l.xa; p.pos0 = b.one.pos0; p.eps = eps; p.exchange = m->d_stack_exchange;
    p.fail_dev = m->d_stack_fail; p.fail_host = m->h_stack_fail_dev; p.epoch = model_stack_epoch(m); p.polls = m->stack_polls;
    float* const hist = l.d_hist + l.hist_slot * b.one.slot;
    p.hist_in = hist + b.one.hist_in * l.stack_hist; p.hist_out = hist + b.one.hist_out * l.stack_hist;
    p.state_in = l.d_pool + b.one.state_in * l.pool_stride; p.state_out = l.d_pool + b.one.state_out * l.pool_stride;
    ProfScope ps(m, "decode_run", it.weights * 2 + it.states * 8, 2.0 * it.weights);
    launch_prenorm_stack(p, st);
  }
  return Tail{l.xa, nullptr, nullptr, 1.f, {}};
}

Tail prenorm_rows(aha_model* m, const SeqBatch& b, const SeqEntry* h_ents, const uint32_t* ids) {
  if (b.n == 1 && b.rows == 1 && b.has_one && m->layered->single_ok) return prenorm_single(m, b, ids);
  LayeredModel& l = *m->layered;
  const aha_model_desc& c = m->desc;
  hipStream_t st = m->stream;
  const int rows = b.rows;
  const double es = l.f32 ? 4.0 : 2.0;
  GemmWorkspaceScope ws_scope(l.ws, l.ws_bytes);
  for (size_t i = 0; i < l.ropes.size(); ++i) launch_rope_pairs(b, l.ropes[i].base, l.ropes[i].dims, l.ropetab[i], st);
  PendingAdd add;
  bool first = true;
  auto enter = [&](const void* w, const void* bias, const PWeights* moe) {   // x <- x + pending (or the embedding), h <- LN(x)
    PreNormArgs a{};
    a.x_in = l.xa; a.add = add;
    if (first) { a.embed = l.embed; a.ids = ids; a.embed_scale = c.embed_scale; }
    a.w = w; a.b = bias; a.eps = c.rms_norm_eps; a.x_out = l.xa; a.h_out = w ? l.h : nullptr; a.width = c.hidden_size; a.rows = rows; a.ld = l.ld;
    if (moe && moe->w_router) { a.zero = l.route.counts; a.n_zero = 2 * l.max_ep; }
    ProfScope ps(m, "elem", (double)rows * l.ld * (8.0 + (2 + add.top) * es), 0);
    launch_prenorm_rows(a, l.f32, st);
    add = PendingAdd{};
    first = false;
  };
  for (int li = 0; li < c.num_hidden_layers; ++li) {
    const PWeights& W = l.P[li];
    const aha_layer_desc& d = c.layers[li];
    enter(W.n1w, W.n1b, nullptr);
    if (li > 0) keep_rows(m, l.xa, rows, li - 1);
    if (d.mixer == AHA_MIXER_MAMBA2) ssm_rows(m, W, b);
    else latent_rows(m, W, b, h_ents);
    add.y = l.y; add.ldy = l.ld;
    if (d.mlp == AHA_MLP_NONE) continue;
    enter(W.n2w, W.n2b, &W);
    if (d.mlp == AHA_MLP_MOE) {
      add = moe_rows(m, W, d, rows);
    } else {
      gated_rows(m, W, rows);
      add.y = l.y; add.ldy = l.ld;
    }
  }
  if (l.keep) {   // the last layer's rows (the product path completes only the wanted ones)
    enter(nullptr, nullptr, nullptr);
    keep_rows(m, l.xa, rows, c.num_hidden_layers - 1);
  }
  return Tail{l.xa, nullptr, nullptr, 1.f, add};
}

// x + pending, model norm of the wanted rows -> l.fin
void prenorm_final(aha_model* m, const Tail& t, const int32_t* rows, int n) {
  LayeredModel& l = *m->layered;
  PreNormArgs a{};
  a.x_in = t.x; a.add = t.add; a.w = l.final_norm; a.b = l.final_norm_b; a.eps = m->desc.rms_norm_eps; a.h_out = l.fin; a.row_list = rows;
  a.width = m->desc.hidden_size; a.rows = n; a.ld = l.ld;
  launch_prenorm_rows(a, l.f32, m->stream);
}

}  // namespace aha
