// Decoders whose config lists their layers one by one: sequences, pages, per-sequence state and the step for all of them, and the layers of
// the post-norm stack (AHA_ARCH_DOSOVIK; the pre-norm one: layered_prenorm.hip).
//
//   x = embed[token] * embed_scale                                                    residual stream: f32
//   per layer, for the mixer and then the feed-forward (if any):
//     h = x + conv(x)                     causal per-channel convolution over the last conv_taps inputs of this sublayer
//     x = norm(alpha x + sublayer(h))     zero-centred RMS norm
//   logits = head . norm(x)
//
// A step is a ragged batch: row r of every buffer is one token, SeqEntry says which rows are whose and at which positions.  Three ways through
// the layers, the same equations in each:
//   rows    any mix of prompts: GEMMs over all rows, row kernels between them (kernels_layered.hip), chunked attention (kernels_attn_chunk.hip)
//   decode  one token per sequence: the same, with q/k norm + rotation + KV append + attention in one launch
//   single  one token of one sequence, bf16: five launches per layer -- matvecs whose prologue does the norm + convolution / the PolyNorm
//           (kernels_gemv_fused.hip) and the fused decode attention
// compute_dtype f32 runs the rows / decode forms with f32 activations, token-major f32 pages and the f32 GEMM.
//
// A sequence owns pages of the model's pool (model.hip alloc_slab) and one slot of convolution history.  Pages that lie in front of every
// layer's current chunk can never be read again and go back to the pool after the step that passed them.
#include "layered_model.h"

namespace aha {

namespace {

// floats of one row of the row kernel's LDS ring
int64_t conv_row_floats(int64_t width) {
  int64_t n = 1024;
  while (n < width) n *= 2;
  return n;
}

int check_desc(const aha_model_desc& c) {
  if (c.hidden_size <= 0 || c.vocab_size <= 0 || c.num_hidden_layers <= 0 || c.num_hidden_layers > AHA_MAX_LAYERS || c.n_stop_tokens < 0 || c.n_stop_tokens > 8 ||
      c.conv_taps < 1)
    return err(AHA_ERR_INVALID, "model_create: sizes must be positive (at most 256 layers, 8 stop tokens)");
  if (c.hidden_size > 8192) return err(AHA_ERR_UNSUPPORTED, "hidden_size above 8192");
  if ((int64_t)(c.conv_taps - 1) * conv_row_floats(c.hidden_size) * 4 > 60 * 1024) return err(AHA_ERR_UNSUPPORTED, "conv_taps x hidden_size exceeds the row kernel's LDS");
  if (c.tp_size > 1) return err(AHA_ERR_UNSUPPORTED, "this architecture runs on one GPU (tp_size 1)");
  for (int i = 0; i < c.num_hidden_layers; ++i) {
    const aha_layer_desc& l = c.layers[i];
    const std::string at = "layer " + std::to_string(i) + ": ";
    if (l.mixer != AHA_MIXER_ATTENTION || (l.mlp != AHA_MLP_NONE && l.mlp != AHA_MLP_POLYNORM)) return err(AHA_ERR_UNSUPPORTED, at + "unknown mixer or feed-forward");
    if (l.heads <= 0 || l.kv_heads <= 0 || l.dim <= 0 || l.vdim <= 0 || l.heads % l.kv_heads || l.chunk < 0 || l.rope_dims < 0 || l.rope_dims % 2 || l.rope_dims > l.dim ||
        (l.mlp != AHA_MLP_NONE && l.ff <= 0) || (l.rope_dims > 0 && !(l.rope_base > 0.0)))
      return err(AHA_ERR_INVALID, at + "inconsistent sizes");
    if (l.vdim > 1024 || ((int64_t)(l.heads + l.kv_heads) * l.dim + (int64_t)l.kv_heads * l.vdim) * 4 > 60 * 1024)
      return err(AHA_ERR_UNSUPPORTED, at + "q / k / v rows exceed the row kernel's LDS");
  }
  return AHA_OK;
}

int ensure_rows(aha_model* m, size_t rows) {
  LayeredModel& l = *m->layered;
  if (rows <= l.cap_rows) return AHA_OK;
  int rc = free_list(m, l.row_bufs);
  if (rc) return rc;
  l.cap_rows = 0;
  const size_t cap = (size_t)round_up((int64_t)rows, rows > 64 ? 256 : 16), es = l.f32 ? 4 : 2;
  auto al = [&](size_t bytes, void** out) { return grow(m, l.row_bufs, bytes, out); };
  if (l.prenorm) {
    if ((rc = prenorm_ensure_rows(m, cap))) return rc;
  } else if ((rc = al(cap * l.ld * 4, (void**)&l.xa)) || (rc = al(cap * l.ld * 4, (void**)&l.xb)) || (rc = al(cap * l.max_nv * 4, (void**)&l.vfirst)) ||
      (rc = al(cap * l.ld * es, &l.h)) || (rc = al(cap * l.max_nqkv * es, &l.qkv)) || (rc = al(cap * l.max_q * es, &l.q)) || (rc = al((cap * l.max_o + 64) * es, &l.o)) ||
      (rc = al(cap * std::max(l.max_ffp, 64) * es, &l.z)) || (rc = al(cap * l.ld * es, &l.y)))
    return rc;
  l.ropetab.assign(l.ropes.size(), nullptr);
  for (size_t i = 0; i < l.ropes.size(); ++i)
    if ((rc = al(cap * l.ropes[i].dims * 4, (void**)&l.ropetab[i]))) return rc;
  if (!l.f32) {
    l.ws_bytes = std::min((size_t)12 * cap * l.ld * 4, (size_t)1 << 30);   // split-K slabs
    if ((rc = al(l.ws_bytes, &l.ws))) return rc;
  }
  l.cap_rows = cap;
  return AHA_OK;
}
int ensure_entries(aha_model* m, size_t n) {
  LayeredModel& l = *m->layered;
  if (n <= l.cap_ents) return AHA_OK;
  int rc = free_list(m, l.ent_bufs);
  if (rc) return rc;
  l.cap_ents = 0;
  const size_t cap = (size_t)round_up((int64_t)n, 8);
  if (l.prenorm) {
    if ((rc = prenorm_ensure_entries(m, cap))) return rc;
  } else if ((rc = grow(m, l.ent_bufs, cap * CHUNK_DECODE_MAX_SPLIT * l.max_part * 4, (void**)&l.part_o)) ||
      (rc = grow(m, l.ent_bufs, cap * CHUNK_DECODE_MAX_SPLIT * l.max_part * 4, (void**)&l.part_ml)) ||
      (rc = grow(m, l.ent_bufs, cap * l.max_kvh * 32 * 4, (void**)&l.ctr)))
    return rc;
  l.cap_ents = cap;
  return AHA_OK;
}
int ensure_want(aha_model* m, size_t n) {
  LayeredModel& l = *m->layered;
  if (n <= l.cap_want) return AHA_OK;
  int rc = free_list(m, l.want_bufs);
  if (rc) return rc;
  l.cap_want = 0;
  const size_t cap = (size_t)round_up((int64_t)n, 16);
  if ((rc = grow(m, l.want_bufs, cap * l.ld * (l.f32 ? 4 : 2), &l.fin)) || (rc = grow(m, l.want_bufs, cap * l.Vp * 4, (void**)&l.logits)) ||
      (rc = grow(m, l.want_bufs, cap * argmax_f32_blocks(m->desc.vocab_size) * 4, (void**)&l.am_max)) ||
      (rc = grow(m, l.want_bufs, cap * argmax_f32_blocks(m->desc.vocab_size) * 4, (void**)&l.am_idx)))
    return rc;
  l.cap_want = cap;
  return AHA_OK;
}
int ensure_meta(aha_model* m, size_t bytes) {
  LayeredModel& l = *m->layered;
  if (bytes <= l.meta_bytes) return AHA_OK;
  AHA_HIP_CHECK(hipStreamSynchronize(m->stream));
  if (l.d_meta) hipFree(l.d_meta);
  if (l.h_meta) hipHostFree(l.h_meta);
  l.d_meta = l.h_meta = nullptr;
  l.meta_bytes = 0;
  const size_t cap = (size_t)round_up((int64_t)bytes * 2, 4096);
  AHA_HIP_CHECK(hipMalloc((void**)&l.d_meta, cap));
  AHA_HIP_CHECK(hipHostMalloc((void**)&l.h_meta, cap));
  l.meta_bytes = cap;
  return AHA_OK;
}
int ensure_slots(aha_model* m, size_t slots) {
  LayeredModel& l = *m->layered;
  if (slots <= l.slots) return AHA_OK;
  size_t cap = std::max<size_t>(l.slots, 4);
  while (cap < slots) cap *= 2;
  float* nh = nullptr;
  AHA_HIP_CHECK(hipMalloc((void**)&nh, std::max<size_t>(cap * (size_t)l.hist_slot * 4, 16)));
  AHA_HIP_CHECK(hipStreamSynchronize(m->stream));
  if (l.pool_stride > 0) {
    float* np = nullptr;
    AHA_HIP_CHECK(hipMalloc((void**)&np, (CONV_HISTORIES - 1 + cap) * (size_t)l.pool_stride * 4));
    if (l.d_pool) {
      AHA_HIP_CHECK(hipMemcpy(np, l.d_pool, (CONV_HISTORIES - 1 + l.slots) * (size_t)l.pool_stride * 4, hipMemcpyDeviceToDevice));
      hipFree(l.d_pool);
    }
    l.d_pool = np;
  }
  if (l.d_hist) {
    if (l.hist_slot) AHA_HIP_CHECK(hipMemcpy(nh, l.d_hist, l.slots * (size_t)l.hist_slot * 4, hipMemcpyDeviceToDevice));
    hipFree(l.d_hist);
  }
  l.d_hist = nh;
  uint64_t* nt = nullptr;
  if (l.tab_ld == 0) l.tab_ld = 64;
  AHA_HIP_CHECK(hipMalloc((void**)&nt, cap * l.tab_ld * 8));
  if (l.d_tab) {
    AHA_HIP_CHECK(hipMemcpy(nt, l.d_tab, l.slots * l.tab_ld * 8, hipMemcpyDeviceToDevice));
    hipFree(l.d_tab);
  }
  l.d_tab = nt;
  l.slots = cap;
  return AHA_OK;
}
// pages for `tokens` tokens of a sequence, mapped on the device
int ensure_seq_pages(aha_model* m, int32_t si, size_t tokens) {
  LayeredModel& l = *m->layered;
  Seq& s = l.seqs[si];
  const size_t need_p = (tokens + KV_PAGE_TOKENS - 1) / KV_PAGE_TOKENS, first_new = s.pages.size();
  if (need_p <= first_new) return AHA_OK;
  if (need_p > l.tab_ld) {
    size_t ld = l.tab_ld;
    while (ld < need_p) ld *= 2;
    uint64_t* nt = nullptr;
    AHA_HIP_CHECK(hipMalloc((void**)&nt, l.slots * ld * 8));
    AHA_HIP_CHECK(hipStreamSynchronize(m->stream));
    AHA_HIP_CHECK(hipMemcpy2D(nt, ld * 8, l.d_tab, l.tab_ld * 8, l.tab_ld * 8, l.slots, hipMemcpyDeviceToDevice));
    hipFree(l.d_tab);
    l.d_tab = nt;
    l.tab_ld = ld;
  }
  while (s.pages.size() < need_p) {
    if (m->free_pages.empty()) {
      const int rc = alloc_slab(m);
      if (rc) return rc;
    }
    s.pages.push_back(m->free_pages.back());
    m->free_pages.pop_back();
  }
  AHA_HIP_CHECK(hipMemcpyAsync(l.d_tab + (size_t)si * l.tab_ld + first_new, s.pages.data() + first_new, (s.pages.size() - first_new) * 8, hipMemcpyHostToDevice, m->stream));
  return AHA_OK;   // (pageable source: staged before the call returns)
}
// pages in front of every layer's chunk or window of the next position go back to the pool (later work on the same stream may reuse them)
void release_passed(aha_model* m, Seq& s) {
  size_t lo = s.len;
  for (int i = 0; i < m->desc.num_hidden_layers; ++i) {
    const aha_layer_desc& d = m->desc.layers[i];
    if (d.mixer == AHA_MIXER_ATTENTION) lo = std::min(lo, d.chunk > 0 ? s.len / (size_t)d.chunk * d.chunk : 0);
    if (d.mixer == AHA_MIXER_LATENT) lo = std::min(lo, d.window > 0 && s.len >= (size_t)d.window ? s.len - (size_t)d.window + 1 : 0);
  }
  for (; s.first_live < lo / KV_PAGE_TOKENS && s.first_live < s.pages.size(); ++s.first_live) {
    m->free_pages.push_back(s.pages[s.first_live]);
    s.pages[s.first_live] = 0;
  }
}
void reset_seq(aha_model* m, Seq& s) {
  for (size_t i = s.pages.size(); i > s.first_live; --i) m->free_pages.push_back(s.pages[i - 1]);
  s.pages.clear();
  s.first_live = 0;
  s.len = 0;
  s.hist = 0;
}
void advance_seq(aha_model* m, Seq& s, size_t n) {
  s.len += n;
  s.hist = (s.hist + 1) % CONV_HISTORIES;
  release_passed(m, s);
}
// which histories a step at history index `hist` of the slot reads and writes
void set_histories(SeqEntry& e, int slot, int hist) {
  e.hist_in = hist;
  e.hist_out = (hist + 1) % CONV_HISTORIES;
  e.state_in = slot == 0 ? e.hist_in : CONV_HISTORIES - 1 + slot;
  e.state_out = slot == 0 ? e.hist_out : CONV_HISTORIES - 1 + slot;
}
SeqEntry make_entry(const Seq& s, int slot, int row0, int len) {
  SeqEntry e{};
  e.row0 = row0;
  e.len = len;
  e.pos0 = (int32_t)s.len;
  e.slot = slot;
  set_histories(e, slot, s.hist);
  return e;
}

ConvIn conv_in(const LayeredModel& l, const aha_model_desc& c, int layer, int sub) {
  ConvIn v;
  v.w = sub ? l.L[layer].conv2 : l.L[layer].conv1;
  v.hist = l.d_hist + (int64_t)(layer * 2 + sub) * CONV_HISTORIES * c.conv_taps * l.ld;
  v.slot_stride = l.hist_slot;
  v.taps = c.conv_taps;
  v.ldw = l.ld;
  return v;
}
SeqKv seq_kv(const LayeredModel& l, const aha_model_desc& c, int layer) {
  SeqKv kv;
  kv.tab = l.d_tab;
  kv.ld = (int64_t)l.tab_ld;
  kv.layer_off = l.L[layer].kv_off;
  kv.kvh = c.layers[layer].kv_heads;
  kv.dq = l.L[layer].dq;
  kv.dv = l.L[layer].dv;
  kv.frag = l.L[layer].frag;
  return kv;
}
QkvPostArgs qkv_post(const LayeredModel& l, const aha_model_desc& c, int li) {
  const LWeights& W = l.L[li];
  const aha_layer_desc& d = c.layers[li];
  QkvPostArgs a{};
  a.qkv = l.qkv; a.ld = W.nqkv; a.k_off = W.k_off; a.v_off = W.v_off;
  a.q_norm = W.qn; a.k_norm = W.kn;
  a.rope_dims = W.rope >= 0 ? d.rope_dims : 0;
  a.rope = W.rope >= 0 ? l.ropetab[W.rope] : nullptr;
  a.heads = d.heads; a.kvh = d.kv_heads; a.dim = d.dim; a.vdim = d.vdim;
  a.eps = c.rms_norm_eps;
  a.lambda = W.lambda; a.v_store = W.v_store; a.v_use = W.v_use;
  a.v_first = l.vfirst;
  a.q_out = l.q;
  a.kv = seq_kv(l, c, li);
  return a;
}
// KV splits of a decode launch: about four pages per block, by the longest chunk among the step's sequences; no more blocks than the chip holds
// at once (two per CU) when a batch fills it anyway
int decode_splits(const aha_layer_desc& d, const SeqEntry* e, int n) {
  int np = 1;
  for (int i = 0; i < n; ++i) {
    const int lo = d.chunk > 0 ? e[i].pos0 / d.chunk * d.chunk : 0;
    if (e[i].pos0 > lo) np = std::max(np, (e[i].pos0 - 1) / KV_PAGE_TOKENS - lo / KV_PAGE_TOKENS + 1);
  }
  return std::max(1, std::min({CHUNK_DECODE_MAX_SPLIT, (np + 3) / 4, 512 / std::max(1, n * d.kv_heads)}));
}

int prepare_keep(aha_model* m, size_t rows) {
  LayeredModel& l = *m->layered;
  if (!l.keep) return AHA_OK;
  const size_t need_f = rows * m->desc.hidden_size * m->desc.num_hidden_layers;
  if (need_f > l.resid_cap) {
    AHA_HIP_CHECK(hipStreamSynchronize(m->stream));
    if (l.resid) hipFree(l.resid);
    l.resid = nullptr;
    l.resid_cap = 0;
    AHA_HIP_CHECK(hipMalloc((void**)&l.resid, need_f * 4));
    l.resid_cap = need_f;
  }
  l.resid_rows = rows;
  return AHA_OK;
}

// rows / decode form.  h_ents: host copy of the entries (launch shapes)
Tail run_rows(aha_model* m, const SeqBatch& b, const SeqEntry* h_ents, const uint32_t* ids) {
  LayeredModel& l = *m->layered;
  const aha_model_desc& c = m->desc;
  hipStream_t st = m->stream;
  const int rows = b.rows;
  const bool decode = b.max_len == 1;
  const double es = l.f32 ? 4.0 : 2.0;
  GemmWorkspaceScope ws_scope(l.ws, l.ws_bytes);
  for (size_t i = 0; i < l.ropes.size(); ++i) launch_rope_pairs(b, l.ropes[i].base, l.ropes[i].dims, l.ropetab[i], st);
  float *x = l.xa, *xn = l.xb;
  const void* norm = nullptr;   // norm of the sublayer whose output is in l.y; null: x comes from the embedding
  auto enter = [&](int li, int sub) {   // x <- norm(alpha x + y) (or the embedding), h <- x + conv(x)
    PostNormArgs a{};
    a.x_in = x; a.y = l.y; a.norm_w = norm; a.alpha = c.post_norm_alpha; a.eps = c.rms_norm_eps;
    if (!norm) { a.embed = l.embed; a.ids = ids; a.embed_scale = c.embed_scale; }
    a.x_out = xn; a.h_out = l.h; a.conv = conv_in(l, c, li, sub);
    a.width = c.hidden_size; a.ld = l.ld; a.ldy = l.ld;
    ProfScope ps(m, "elem", (double)rows * l.ld * (8.0 + 2 * es), 0);
    launch_postnorm_conv(a, b, l.f32, st);
    std::swap(x, xn);
    if (norm && sub == 0) keep_rows(m, x, rows, li - 1);
  };
  for (int li = 0; li < c.num_hidden_layers; ++li) {
    const LWeights& W = l.L[li];
    const aha_layer_desc& d = c.layers[li];
    enter(li, 0);
    gemm(m, l.h, l.ld, W.wqkv, l.qkv, W.nqkv, rows, W.nqkv, (int)l.ld);
    QkvPostArgs qp = qkv_post(l, c, li);
    qp.bias = W.bqkv_f32;   // (the GEMM's faster tilings have no bias epilogue)
    if (decode && W.fused_decode && !l.f32) {
      ChunkDecodeArgs a{};
      a.p = qp; a.qkv_f32 = 0; a.o = l.o; a.chunk = d.chunk; a.sink = 1; a.scale = d.scale;
      a.part_o = l.part_o; a.part_ml = l.part_ml; a.ctr = l.ctr;
      a.nsplit = decode_splits(d, h_ents, b.n);
      ProfScope ps(m, "attn_decode", (double)rows * W.nqkv * 2, 0);
      launch_chunk_attn_decode(a, b, st);
    } else {
      ChunkAttnArgs a{};
      a.q = l.q; a.o = l.o; a.kv = qp.kv; a.heads = d.heads; a.dvo = W.dvo; a.ldo = W.o_ld; a.vdim = d.vdim; a.dim = d.dim; a.chunk = d.chunk; a.sink = 1; a.scale = d.scale;
      const bool one_launch = l.f32 && chunk_attn_f32_decode_ok(qp, a, b);
      if (!one_launch) {
        ProfScope ps(m, "elem", (double)rows * (W.nqkv + W.nk + W.nv + d.heads * W.dq) * es, 0);
        launch_qkv_post(qp, b, l.f32, st);
      }
      double flops = 0;
      for (int i = 0; i < b.n; ++i) {
        const double keys = d.chunk > 0 ? std::min<double>(d.chunk, h_ents[i].pos0 + h_ents[i].len) : h_ents[i].pos0 + h_ents[i].len;
        flops += 2.0 * h_ents[i].len * keys * 0.5 * d.heads * (d.dim + d.vdim);
      }
      ProfScope ps(m, "attn_prefill", (double)rows * (one_launch ? W.nqkv + W.nk + W.nv + d.heads * W.dvo : d.heads * (W.dq + W.dvo)) * es, flops);
      if (one_launch) launch_chunk_attn_f32_decode(qp, a, b, st);
      else if (W.frag) launch_chunk_attn_prefill(a, b, st);
      else launch_chunk_attn_rows(a, b, l.f32, st);
    }
    gemm(m, l.o, W.o_ld, W.wo, l.y, l.ld, rows, (int)l.ld, W.ldo);
    norm = W.norm1;
    if (d.mlp == AHA_MLP_NONE) continue;
    enter(li, 1);
    const GemmArgs up = gemm_args(l.h, l.ld, W.wup, l.z, W.ffp, rows, W.ffp, (int)l.ld), down = gemm_args(l.z, W.ffp, W.wdown, l.y, l.ld, rows, (int)l.ld, W.ffp);
    if (!l.f32 && gemm_takes_poly(up, down)) {
      SkinnyPoly p{};
      p.stats = l.zstats; p.eps = c.rms_norm_eps; p.inv_ff = 1.0f / (float)d.ff;
      memcpy(p.coef, W.act, sizeof(p.coef));
      ProfScope ps(m, "gemm", (double)rows * (2.0 * l.ld + 2.0 * W.ffp) * 2 + (double)l.ld * W.ffp * 4, 4.0 * rows * W.ffp * l.ld);
      launch_gemm_skinny_poly(up, down, p, st);
      norm = W.norm2;
      continue;
    }
    gemm(m, l.h, l.ld, W.wup, l.z, W.ffp, rows, W.ffp, (int)l.ld);
    {
      PolyNormArgs a{};
      a.z = l.z; a.out = l.z; a.eps = c.rms_norm_eps; a.ff = d.ff; a.ld = W.ffp; a.rows = rows;
      memcpy(a.coef, W.act, sizeof(a.coef));
      ProfScope ps(m, "elem", (double)rows * W.ffp * 2 * es, 0);
      launch_polynorm_rows(a, l.f32, st);
    }
    gemm(m, l.z, W.ffp, W.wdown, l.y, l.ld, rows, (int)l.ld, W.ffp);
    norm = W.norm2;
  }
  if (l.keep) {   // the last layer's norm of every row (the product path norms only the wanted ones)
    PostNormArgs a{};
    a.x_in = x; a.y = l.y; a.norm_w = norm; a.alpha = c.post_norm_alpha; a.eps = c.rms_norm_eps;
    a.x_out = xn; a.conv = conv_in(l, c, 0, 0); a.width = c.hidden_size; a.ld = l.ld; a.ldy = l.ld;
    a.conv.taps = 1;   // (no input convolution behind the last layer)
    launch_postnorm_conv(a, b, l.f32, st);
    keep_rows(m, xn, rows, c.num_hidden_layers - 1);
  }
  return Tail{x, l.y, norm, c.post_norm_alpha, {}};
}

// single form: one token of one sequence, five launches per layer
Tail run_single(aha_model* m, const SeqBatch& b, const uint32_t* id) {
  LayeredModel& l = *m->layered;
  const aha_model_desc& c = m->desc;
  hipStream_t st = m->stream;
  const SeqEntry& e = b.one;
  for (size_t i = 0; i < l.ropes.size(); ++i) launch_rope_pairs(b, l.ropes[i].base, l.ropes[i].dims, l.ropetab[i], st);
  const void* norm = nullptr;
  auto matvec_bytes = [](double n, double k) { return n * k * 2 + k * 4 + n * 4; };
  auto post = [&](int li, int sub) {
    GemvPostNorm p{};
    p.s = l.s1; p.norm_w = norm; p.x_out = l.x1; p.conv = conv_in(l, c, li, sub); p.entry = e; p.width = c.hidden_size;
    return p;
  };
  for (int li = 0; li < c.num_hidden_layers; ++li) {
    const LWeights& W = l.L[li];
    const aha_layer_desc& d = c.layers[li];
    GemvArgs g{};
    g.W = W.wqkv; g.N = W.nqkv; g.K = (int)l.ld; g.y_f32 = l.qkv1; g.res_f32 = W.bqkv_f32; g.res_scale = 1.f; g.eps = c.rms_norm_eps;
    if (!norm) {
      PostNormArgs a{};
      a.embed = l.embed; a.ids = id; a.embed_scale = c.embed_scale; a.x_out = l.x1; a.h_out = l.h; a.conv = conv_in(l, c, li, 0);
      a.width = c.hidden_size; a.ld = l.ld; a.ldy = l.ld;
      launch_postnorm_conv(a, b, false, st);
      g.x = l.h;
    }
    {
      ProfScope ps(m, "gemv", matvec_bytes(g.N, g.K), 2.0 * g.N * g.K);
      if (norm) launch_gemv_postnorm(g, post(li, 0), GEMV_AXPY_F32, st);
      else launch_gemv(g, GEMV_AXPY_F32, st);
    }
    if (norm) keep_rows(m, l.x1, 1, li - 1);
    {
      ChunkDecodeArgs a{};
      a.p = qkv_post(l, c, li);
      a.p.qkv = l.qkv1;
      a.qkv_f32 = 1; a.o = l.o; a.chunk = d.chunk; a.sink = 1; a.scale = d.scale;
      a.part_o = l.part_o; a.part_ml = l.part_ml; a.ctr = l.ctr;
      a.nsplit = decode_splits(d, &e, 1);
      const double keys = e.pos0 + 1 - (d.chunk > 0 ? e.pos0 / d.chunk * d.chunk : 0);
      ProfScope ps(m, "attn_decode", keys * (W.nk + W.nv) * 2 + W.nqkv * 4.0, 2.0 * keys * d.heads * (d.dim + d.vdim));
      launch_chunk_attn_decode(a, b, st);
    }
    g = GemvArgs{};
    g.W = W.wo; g.x = l.o; g.N = (int)l.ld; g.K = W.ldo; g.y_f32 = l.s1; g.res_f32 = l.x1; g.res_scale = c.post_norm_alpha;
    {
      ProfScope ps(m, "gemv", matvec_bytes(g.N, g.K), 2.0 * g.N * g.K);
      launch_gemv(g, GEMV_AXPY_F32, st);
    }
    norm = W.norm1;
    if (d.mlp == AHA_MLP_NONE) continue;
    g = GemvArgs{};
    g.W = W.wup; g.N = W.ffp; g.K = (int)l.ld; g.y_f32 = l.z1; g.eps = c.rms_norm_eps;
    {
      ProfScope ps(m, "gemv", matvec_bytes(g.N, g.K), 2.0 * g.N * g.K);
      launch_gemv_postnorm(g, post(li, 1), GEMV_PARTIAL_F32, st);
    }
    PolyNormArgs pa{};
    pa.z = l.z1; pa.eps = c.rms_norm_eps; pa.ff = d.ff;
    memcpy(pa.coef, W.act, sizeof(pa.coef));
    g = GemvArgs{};
    g.W = W.wdown; g.N = (int)l.ld; g.K = W.ffp; g.y_f32 = l.s1; g.res_f32 = l.x1; g.res_scale = c.post_norm_alpha;
    {
      ProfScope ps(m, "gemv", matvec_bytes(g.N, g.K), 2.0 * g.N * g.K);
      launch_gemv_polynorm(g, pa, GEMV_AXPY_F32, st);
    }
    norm = W.norm2;
  }
  if (l.keep) {
    PostNormArgs a{};
    a.x_in = l.s1; a.norm_w = norm; a.alpha = 1.f; a.eps = c.rms_norm_eps; a.x_out = l.xb; a.conv = conv_in(l, c, 0, 0); a.width = c.hidden_size; a.ld = l.ld; a.ldy = l.ld;
    a.conv.taps = 1;
    launch_postnorm_conv(a, b, false, st);
    keep_rows(m, l.xb, 1, c.num_hidden_layers - 1);
  }
  return Tail{l.s1, nullptr, norm, 1.f, {}};
}

Tail run_step(aha_model* m, const SeqBatch& b, const SeqEntry* h_ents, const uint32_t* ids) {
  if (m->layered->prenorm) return prenorm_rows(m, b, h_ents, ids);
  return b.n == 1 && b.rows == 1 && m->layered->single_ok ? run_single(m, b, ids) : run_rows(m, b, h_ents, ids);
}

// final norm + head of n wanted rows (device row list, null = row 0 .. n - 1) into `logits` (n, Vp) f32
void run_head(aha_model* m, const Tail& t, const int32_t* rows, int n, float* logits) {
  LayeredModel& l = *m->layered;
  const aha_model_desc& c = m->desc;
  GemmWorkspaceScope ws_scope(l.ws, l.ws_bytes);
  if (l.prenorm) {
    prenorm_final(m, t, rows, n);
  } else {
    FinalRowsArgs f{};
    f.x = t.x; f.y = t.y; f.norm_w = t.norm; f.final_w = l.final_norm; f.rows = rows; f.out = l.fin; f.alpha = t.alpha; f.eps = c.rms_norm_eps;
    f.width = c.hidden_size; f.n = n; f.ld = l.ld; f.ldy = l.ld;
    launch_final_rows(f, l.f32, m->stream);
  }
  if (n == 1 && !l.f32) {   // matvec with the arg-max partials of the greedy loop
    GemvArgs g{};
    g.W = l.head; g.x = l.fin; g.N = c.vocab_size; g.K = (int)l.ld; g.y_f32 = logits; g.blk_max = m->d_blk_max; g.blk_idx = m->d_blk_idx; g.f32_logits = 1; g.softcap = c.logit_softcap;
    ProfScope ps(m, "gemv", (double)g.N * g.K * 2, 2.0 * g.N * g.K);
    launch_gemv(g, GEMV_LOGITS, m->stream);
    return;
  }
  gemm(m, l.fin, l.ld, l.head, logits, l.Vp, n, l.Vp, (int)l.ld, ACT_PARTIAL_F32);   // (f32 outputs)
  if (c.logit_softcap > 0.f) launch_softcap(logits, (int64_t)n * l.Vp, c.logit_softcap, m->stream);
}
// arg-max of the row run_head(n == 1) left in m->d_logits -> d_state->next_token
void argmax_single(aha_model* m) {
  LayeredModel& l = *m->layered;
  if (!l.f32) launch_argmax_partials(m->d_blk_max, m->d_blk_idx, gemv_num_tiles(m->desc.vocab_size, (int)l.ld), &m->d_state->next_token, m->stream);
  else launch_argmax_f32(m->d_logits, m->desc.vocab_size, m->d_blk_max, m->d_blk_idx, &m->d_state->next_token, m->stream);
}

bool seq_ok(const aha_model* m, int32_t seq) {
  return m->layered && seq >= 0 && (size_t)seq < m->layered->seqs.size() && m->layered->seqs[seq].open;
}

}  // namespace

// ---------------------------------------------------------------------------------------------------------------
int layered_create(aha_model* m, const aha_tensor_view* w, size_t nw) {
  const aha_model_desc& c = m->desc;
  const bool pre = c.arch == AHA_ARCH_VAMATAR;
  int rc = pre ? prenorm_check(c) : check_desc(c);
  if (rc) return rc;
  m->layered = new LayeredModel();
  LayeredModel& l = *m->layered;
  l.f32 = c.compute_dtype == AHA_F32;
  l.prenorm = pre;
  const int H = c.hidden_size, V = c.vocab_size, taps = c.conv_taps;
  l.ld = round_up(H, 256);   // (one wave's columns in the row kernel)
  l.Vp = (int)round_up(V, 64);
  m->lm_rows = V;
  const aha_tensor_view* t = nullptr;
  auto vec = [&](const std::string& name, int64_t n, void** out) -> int {   // (n) -> bf16 padded to 256
    int r = need_tensor(w, nw, name, &t);
    return r ? r : put_matrix(m, t, 1, n, 1, round_up(n, 256), out);
  };
  auto mat = [&](const std::string& name, int64_t rows, int64_t cols, int64_t rows_p, int64_t ld, void** out) -> int {
    int r = need_tensor(w, nw, name, &t);
    return r ? r : put_matrix(m, t, rows, cols, rows_p, ld, out);
  };
  auto conv = [&](const std::string& name, void** out) -> int {   // (H, taps) -> (taps, ld)
    int r = need_tensor(w, nw, name, &t);
    if (r) return r;
    std::vector<uint16_t> a, b((size_t)taps * l.ld, 0);
    if ((r = host_bf16(t, (int64_t)H * taps, &a))) return r;
    for (int i = 0; i < H; ++i)
      for (int j = 0; j < taps; ++j) b[(size_t)j * l.ld + i] = a[(size_t)i * taps + j];
    if ((r = dev_alloc(m, b.size() * 2, out))) return r;
    AHA_HIP_CHECK(hipMemcpy(*out, b.data(), b.size() * 2, hipMemcpyHostToDevice));
    return AHA_OK;
  };
#define TRY(e) do { if ((rc = (e))) return rc; } while (0)
  TRY(mat("embed", V, H, V, l.ld, &l.embed));
  TRY(mat("head", V, H, l.Vp, l.ld, &l.head));
  TRY(vec("final.norm", H, &l.final_norm));
  if (pre) TRY(vec("final.norm.b", H, &l.final_norm_b));
  uint64_t kv_off = 0;
  if (pre) TRY(prenorm_create(m, w, nw, &kv_off));
  else l.L.resize(c.num_hidden_layers);
  int first_mix = -1, mix_nv = 0;
  l.single_ok = pre ? prenorm_single_ok(m) : !l.f32;
  for (int li = 0; li < (int)l.L.size(); ++li) {
    LWeights& W = l.L[li];
    const aha_layer_desc& d = c.layers[li];
    const std::string p = "l" + std::to_string(li) + ".", mx = p + "mix.";
    W.nq = d.heads * d.dim; W.nk = d.kv_heads * d.dim; W.nv = d.kv_heads * d.vdim;
    W.k_off = (int)round_up(W.nq, 8); W.v_off = W.k_off + (int)round_up(W.nk, 8); W.nqkv = (int)round_up(W.v_off + W.nv, 64);
    int dq, dv;
    W.frag = chunk_attn_dims_ok(d.dim, d.vdim, &dq, &dv) && !l.f32 && d.scale > 0.f;   // (the MFMA kernels keep the maximum in raw score units)
    W.fused_decode = W.frag && d.heads / d.kv_heads <= 16;
    W.dq = W.frag ? dq : d.dim; W.dv = W.frag ? dv : d.vdim;
    W.dvo = W.frag ? dv : d.vdim;
    W.ldo = (int)round_up((int64_t)d.heads * W.dvo, 64);
    W.o_ld = W.frag ? d.heads * W.dvo : W.ldo;
    W.kv_off = kv_off;
    kv_off += (uint64_t)round_up((int64_t)d.kv_heads * KV_PAGE_TOKENS * (W.dq + W.dv) * (l.f32 ? 4 : 2), 1024);
    if (d.rope_dims > 0) {
      for (size_t i = 0; i < l.ropes.size(); ++i)
        if (l.ropes[i].base == d.rope_base && l.ropes[i].dims == d.rope_dims) W.rope = (int)i;
      if (W.rope < 0) {
        W.rope = (int)l.ropes.size();
        l.ropes.push_back({d.rope_base, d.rope_dims});
      }
    }
    if (d.v_mix) {
      if (first_mix < 0) {
        first_mix = li;
        mix_nv = W.nv;
        W.v_store = 1;
      } else {
        if (W.nv != mix_nv) return err(AHA_ERR_INVALID, "layer " + std::to_string(li) + ": mixed values must have one width");
        W.v_use = 1;
      }
    }
    // q | k | v rows of one matrix
    TRY(new_matrix(m, W.nqkv, l.ld, &W.wqkv));
    std::vector<float> bf(W.nqkv, 0.f);
    const struct { const char* n; int rows, off; } parts[3] = {{"q", W.nq, 0}, {"k", W.nk, W.k_off}, {"v", W.nv, W.v_off}};
    for (const auto& q : parts) {
      TRY(need_tensor(w, nw, mx + q.n, &t));
      TRY(put_block(m, t, q.rows, H, 0, H, W.wqkv, q.off, 0, l.ld));
      TRY(need_tensor(w, nw, mx + q.n + ".b", &t));
      std::vector<uint16_t> hb;
      TRY(host_bf16(t, q.rows, &hb));
      for (int i = 0; i < q.rows; ++i) bf[q.off + i] = bf_host(hb[i]);
    }
    TRY(dev_alloc(m, bf.size() * 4, (void**)&W.bqkv_f32));
    AHA_HIP_CHECK(hipMemcpy(W.bqkv_f32, bf.data(), bf.size() * 4, hipMemcpyHostToDevice));
    TRY(vec(mx + "q.norm", W.nq, &W.qn));
    TRY(vec(mx + "k.norm", W.nk, &W.kn));
    if (W.v_use) {
      TRY(need_tensor(w, nw, mx + "vmix", &t));
      std::vector<uint16_t> v;
      TRY(host_bf16(t, 1, &v));
      W.lambda = bf_host(v[0]);
    }
    // output projection: the columns of a head padded to the attention output's head width
    TRY(need_tensor(w, nw, mx + "o", &t));
    TRY(new_matrix(m, l.ld, W.ldo, &W.wo));
    for (int h = 0; h < d.heads; ++h) TRY(put_block(m, t, H, (int64_t)d.heads * d.vdim, (int64_t)h * d.vdim, d.vdim, W.wo, 0, (int64_t)h * W.dvo, W.ldo));
    TRY(vec(p + "norm1", H, &W.norm1));
    TRY(conv(p + "canon1", &W.conv1));
    if (d.mlp != AHA_MLP_NONE) {
      W.ffp = (int)round_up(d.ff, 64);
      TRY(mat(p + "mlp.up", d.ff, H, W.ffp, l.ld, &W.wup));
      TRY(mat(p + "mlp.down", H, d.ff, l.ld, W.ffp, &W.wdown));
      TRY(need_tensor(w, nw, p + "mlp.act", &t));
      std::vector<uint16_t> a;
      TRY(host_bf16(t, 4, &a));
      for (int i = 0; i < 4; ++i) W.act[i] = bf_host(a[i]);
      TRY(vec(p + "norm2", H, &W.norm2));
      TRY(conv(p + "canon2", &W.conv2));
    }
    l.single_ok = l.single_ok && W.fused_decode && gemv_fused_ok((int)l.ld, std::max(W.ffp, 64)) && W.ldo <= 15872;
    l.max_nqkv = std::max(l.max_nqkv, W.nqkv);
    l.max_q = std::max(l.max_q, d.heads * W.dq);
    l.max_o = std::max(l.max_o, W.ldo);
    l.max_ffp = std::max(l.max_ffp, W.ffp);
    l.max_nv = std::max(l.max_nv, W.nv);
    l.max_part = std::max(l.max_part, d.heads * std::max(W.dv, 2));
    l.max_kvh = std::max(l.max_kvh, d.kv_heads);
  }
  // page pool: a page holds all layers, layer i behind layer i - 1
  m->page_bytes = std::max<uint64_t>(kv_off, 1024);
  m->pages_per_slab = 64;
  m->slab_bytes = m->pages_per_slab * m->page_bytes;
  if (!pre) l.hist_slot = (int64_t)c.num_hidden_layers * 2 * CONV_HISTORIES * taps * l.ld;
  TRY(ensure_slots(m, 1));
  l.seqs.resize(1);
  l.seqs[0].open = true;
  for (size_t n = 0; n < (size_t)c.kv_reserve_tokens; n += m->pages_per_slab * KV_PAGE_TOKENS) TRY(alloc_slab(m));
  if (pre) {
    TRY(prenorm_alloc_single(m));
  } else {
    TRY(dev_alloc(m, (size_t)l.ld * 4, (void**)&l.s1, true));
    TRY(dev_alloc(m, (size_t)l.ld * 4, (void**)&l.x1, true));
    TRY(dev_alloc(m, (size_t)l.max_nqkv * 4, (void**)&l.qkv1, true));
    TRY(dev_alloc(m, (size_t)std::max(l.max_ffp, 64) * 4, (void**)&l.z1, true));
    if (!l.f32) TRY(dev_alloc(m, gemm_skinny_poly_floats() * 4, (void**)&l.zstats, true));
  }
  TRY(ensure_rows(m, 1));
  TRY(ensure_entries(m, 1));
  TRY(ensure_want(m, 1));
  TRY(ensure_meta(m, 4096));
#undef TRY
  return AHA_OK;
}

void layered_destroy(aha_model* m) {
  if (!m->layered) return;
  LayeredModel& l = *m->layered;
  for (auto* v : {&l.row_bufs, &l.ent_bufs, &l.want_bufs})
    for (void* p : *v) hipFree(p);
  if (l.d_tab) hipFree(l.d_tab);
  if (l.d_hist) hipFree(l.d_hist);
  if (l.d_pool) hipFree(l.d_pool);
  for (void* p : l.ext_bufs) hipFree(p);
  if (l.d_meta) hipFree(l.d_meta);
  if (l.h_meta) hipHostFree(l.h_meta);
  if (l.d_greedy) hipFree(l.d_greedy);
  if (l.resid) hipFree(l.resid);
  delete m->layered;
  m->layered = nullptr;
}

int layered_seq_open(aha_model* m, int32_t* seq) {
  LayeredModel& l = *m->layered;
  size_t i = 1;
  while (i < l.seqs.size() && l.seqs[i].open) ++i;
  if (i == l.seqs.size()) {
    const int rc = ensure_slots(m, i + 1);
    if (rc) return rc;
    l.seqs.emplace_back();
  }
  reset_seq(m, l.seqs[i]);
  l.seqs[i].open = true;
  *seq = (int32_t)i;
  return AHA_OK;
}
int layered_seq_close(aha_model* m, int32_t seq) {
  if (!seq_ok(m, seq) || seq == 0) return err(AHA_ERR_INVALID, "seq_close: not an open sequence");
  reset_seq(m, m->layered->seqs[seq]);
  m->layered->seqs[seq].open = false;
  return AHA_OK;
}
int64_t layered_seq_len(const aha_model* m, int32_t seq) { return seq_ok(m, seq) ? (int64_t)m->layered->seqs[seq].len : AHA_ERR_INVALID; }
int64_t layered_seq_pages(const aha_model* m, int32_t seq) {
  return seq_ok(m, seq) ? (int64_t)(m->layered->seqs[seq].pages.size() - m->layered->seqs[seq].first_live) : AHA_ERR_INVALID;
}
int layered_clear(aha_model* m) {
  reset_seq(m, m->layered->seqs[0]);
  m->cache_len = 0;
  return AHA_OK;
}

int layered_forward_batch(aha_model* m, const aha_batch_entry* en, size_t n_en, float* logits_out, uint32_t* argmax_out) {
  LayeredModel& l = *m->layered;
  const aha_model_desc& c = m->desc;
  if (!en || n_en == 0) return err(AHA_ERR_INVALID, "forward_batch: no entries");
  size_t rows = 0, want = 0, max_len = 0;
  std::vector<char> used(l.seqs.size(), 0);
  for (size_t i = 0; i < n_en; ++i) {
    if (!seq_ok(m, en[i].seq) || used[en[i].seq]) return err(AHA_ERR_INVALID, "forward_batch: entry " + std::to_string(i) + ": not an open sequence, or named twice");
    used[en[i].seq] = 1;
    if (!en[i].tokens || en[i].n_tokens == 0 || (en[i].n_want && !en[i].want)) return err(AHA_ERR_INVALID, "forward_batch: entry " + std::to_string(i) + ": no tokens");
    for (size_t j = 0; j < en[i].n_tokens; ++j)
      if (en[i].tokens[j] >= (uint32_t)c.vocab_size) return err(AHA_ERR_INVALID, "token id out of range");
    for (size_t j = 0; j < en[i].n_want; ++j)
      if (en[i].want[j] >= en[i].n_tokens) return err(AHA_ERR_INVALID, "forward_batch: wanted place out of range");
    rows += en[i].n_tokens;
    want += en[i].n_want;
    max_len = std::max(max_len, en[i].n_tokens);
  }
  if (rows > (1u << 24)) return err(AHA_ERR_INVALID, "forward_batch: too many rows");
  AHA_HIP_CHECK(hipSetDevice(m->ctx->device));
  const size_t o_row = round_up((int64_t)(n_en * sizeof(SeqEntry)), 64), o_ids = o_row + round_up((int64_t)rows * 4, 64), o_want = o_ids + round_up((int64_t)rows * 4, 64),
               o_ext = o_want + round_up((int64_t)want * 4, 64), o_am = o_ext + round_up((int64_t)(l.windows.size() * n_en * 4), 64), bytes = o_am + round_up((int64_t)want * 4, 64);
  // logits of many wanted rows leave in slices of a bounded buffer
  constexpr size_t SLICE = 1024;
  int rc;
  if ((rc = ensure_rows(m, rows)) || (rc = ensure_entries(m, n_en)) || (rc = ensure_want(m, std::min(std::max<size_t>(want, 1), SLICE))) || (rc = ensure_meta(m, bytes)) ||
      (rc = prepare_keep(m, rows)))
    return rc;
  for (size_t i = 0; i < n_en; ++i)
    if ((rc = ensure_seq_pages(m, en[i].seq, l.seqs[en[i].seq].len + en[i].n_tokens))) return rc;
  SeqEntry* he = (SeqEntry*)l.h_meta;
  int32_t *hr = (int32_t*)(l.h_meta + o_row), *hw = (int32_t*)(l.h_meta + o_want);
  uint32_t* hi = (uint32_t*)(l.h_meta + o_ids);
  size_t r = 0, wi = 0;
  for (size_t i = 0; i < n_en; ++i) {
    he[i] = make_entry(l.seqs[en[i].seq], en[i].seq, (int)r, (int)en[i].n_tokens);
    for (size_t j = 0; j < en[i].n_want; ++j) hw[wi++] = (int32_t)(r + en[i].want[j]);
    for (size_t j = 0; j < en[i].n_tokens; ++j, ++r) {
      hr[r] = (int32_t)i;
      hi[r] = en[i].tokens[j];
    }
  }
  if (max_len > 1 && !l.windows.empty()) {
    if ((rc = prenorm_prepare_ext(m, he, n_en, (int32_t*)(l.h_meta + o_ext)))) return rc;
    l.ext_dev = (const int32_t*)(l.d_meta + o_ext);
  }
  AHA_HIP_CHECK(hipMemcpyAsync(l.d_meta, l.h_meta, o_am, hipMemcpyHostToDevice, m->stream));
  SeqBatch b{};
  b.entries = (const SeqEntry*)l.d_meta;
  b.row_entry = (const int32_t*)(l.d_meta + o_row);
  b.n = (int)n_en; b.rows = (int)rows; b.max_len = (int)max_len;
  if (n_en == 1) {
    b.has_one = 1;
    b.one = he[0];
  }
  const uint32_t* ids = (const uint32_t*)(l.d_meta + o_ids);
  const uint32_t before = m->stack_epoch;
  Tail t = run_step(m, b, he, ids);
  for (size_t i = 0; i < n_en; ++i) advance_seq(m, l.seqs[en[i].seq], en[i].n_tokens);
  m->cache_len = l.seqs[0].len;
  m->have_logits = false;
  l.last_want = 0;
  const int32_t* dw = (const int32_t*)(l.d_meta + o_want);
  uint32_t* dam = (uint32_t*)(l.d_meta + o_am);
  const size_t V = c.vocab_size;
again:
  for (size_t w0 = 0; w0 < want; w0 += SLICE) {
    const size_t n = std::min(SLICE, want - w0);
    float* lg = want == 1 ? m->d_logits : l.logits;
    run_head(m, t, dw + w0, (int)n, lg);
    if (want == 1) {
      argmax_single(m);
      m->have_logits = true;
    } else if (argmax_out) {
      launch_argmax_f32_rows(lg, V, l.Vp, (int)n, l.am_max, l.am_idx, dam + w0, m->stream);
    }
    if (logits_out)
      AHA_HIP_CHECK(hipMemcpy2DAsync(logits_out + w0 * V, V * 4, lg, (size_t)l.Vp * 4, V * 4, n, hipMemcpyDeviceToHost, m->stream));
    if (logits_out && want > SLICE) AHA_HIP_CHECK(hipStreamSynchronize(m->stream));
  }
  if (want == 1 && argmax_out) AHA_HIP_CHECK(hipMemcpyAsync(l.h_meta + o_am, &m->d_state->next_token, 4, hipMemcpyDeviceToHost, m->stream));
  else if (argmax_out && want) AHA_HIP_CHECK(hipMemcpyAsync(l.h_meta + o_am, dam, want * 4, hipMemcpyDeviceToHost, m->stream));
  AHA_HIP_CHECK(hipGetLastError());
  AHA_HIP_CHECK(hipStreamSynchronize(m->stream));   // (the pinned step buffer is free again)
  if (model_stack_failed(m) && m->stack_epoch != before) {   // (a token of one sequence, where such launches ran: as separate ones)
    ++m->stack_hold;
    t = run_step(m, b, he, ids);
    --m->stack_hold;
    goto again;
  }
  if (argmax_out && want) memcpy(argmax_out, l.h_meta + o_am, want * 4);
  if (want <= SLICE) l.last_want = want;
  return AHA_OK;
}

int layered_select_logits(aha_model* m, size_t row) {
  LayeredModel& l = *m->layered;
  if (row >= l.last_want) return err(AHA_ERR_STATE, "select_logits: the last batch has no such row of logits (or too many rows)");
  if (l.last_want > 1) AHA_HIP_CHECK(hipMemcpyAsync(m->d_logits, l.logits + row * l.Vp, (size_t)m->desc.vocab_size * 4, hipMemcpyDeviceToDevice, m->stream));
  m->have_logits = true;
  return AHA_OK;
}

int layered_forward_one(aha_model* m, const uint32_t* ids, size_t n, size_t offset, float* logits_out, uint32_t* argmax_out) {
  if (offset != m->layered->seqs[0].len)
    return err(AHA_ERR_STATE, "seqlen_offset " + std::to_string(offset) + " is not the sequence's length " + std::to_string(m->layered->seqs[0].len));
  const uint32_t last = (uint32_t)(n - 1);
  aha_batch_entry e{};
  e.seq = 0;
  e.tokens = ids;
  e.n_tokens = n;
  e.want = &last;
  e.n_want = 1;
  uint32_t am = 0;
  const int rc = layered_forward_batch(m, &e, 1, logits_out, &am);
  if (!rc && argmax_out) *argmax_out = am;
  return rc;
}

// ---- device-resident greedy loop (model.hip model_decode_greedy): the token of a step is d_state->token, its entry is known on the host --------
int layered_begin_greedy(aha_model* m, size_t max_new, size_t offset) {
  LayeredModel& l = *m->layered;
  Seq& s = l.seqs[0];
  if (offset != s.len) return err(AHA_ERR_STATE, "seqlen_offset is not the sequence's length");
  int rc;
  if ((rc = ensure_seq_pages(m, 0, s.len + max_new)) || (rc = ensure_rows(m, 1)) || (rc = ensure_entries(m, 1)) || (rc = ensure_want(m, 1)) || (rc = prepare_keep(m, 1))) return rc;
  if (max_new > l.greedy_cap) {
    AHA_HIP_CHECK(hipStreamSynchronize(m->stream));
    if (l.d_greedy) hipFree(l.d_greedy);
    l.d_greedy = nullptr;
    l.greedy_cap = 0;
    AHA_HIP_CHECK(hipMalloc((void**)&l.d_greedy, max_new * sizeof(SeqEntry)));
    l.greedy_cap = max_new;
  }
  std::vector<SeqEntry> es(max_new);
  for (size_t i = 0; i < max_new; ++i) {
    es[i] = make_entry(s, 0, 0, 1);
    es[i].pos0 += (int32_t)i;
    set_histories(es[i], 0, (int)((s.hist + i) % CONV_HISTORIES));
  }
  AHA_HIP_CHECK(hipMemcpyAsync(l.d_greedy, es.data(), max_new * sizeof(SeqEntry), hipMemcpyHostToDevice, m->stream));
  AHA_HIP_CHECK(hipStreamSynchronize(m->stream));
  l.greedy_base = s.len;
  return AHA_OK;
}
int layered_enqueue_step(aha_model* m, size_t kv_len_after) {
  LayeredModel& l = *m->layered;
  const size_t i = kv_len_after - 1 - l.greedy_base;
  Seq s = Seq();
  s.len = l.greedy_base + i;
  s.hist = (int)((l.seqs[0].hist + i) % CONV_HISTORIES);
  SeqBatch b{};
  b.entries = l.d_greedy + i;
  b.n = b.rows = b.max_len = 1;
  b.has_one = 1;
  b.one = make_entry(s, 0, 0, 1);
  const uint32_t* id = &m->d_state->token;
  const Tail t = run_step(m, b, &b.one, id);
  run_head(m, t, nullptr, 1, m->d_logits);
  argmax_single(m);
  return AHA_OK;
}
void layered_end_greedy(aha_model* m, size_t produced) {
  Seq& s = m->layered->seqs[0];
  s.len += produced;
  s.hist = (int)((s.hist + produced) % CONV_HISTORIES);
  release_passed(m, s);
  m->layered->last_want = 0;
}

int layered_keep_residual(aha_model* m, bool on) {
  m->layered->keep = on;
  m->layered->resid_rows = 0;
  return AHA_OK;
}
int64_t layered_residual(aha_model* m, int layer, float* out, size_t n) {
  LayeredModel& l = *m->layered;
  const size_t per = l.resid_rows * (size_t)m->desc.hidden_size;
  if (!l.keep || l.resid_rows == 0 || layer < 0 || layer >= m->desc.num_hidden_layers) return err(AHA_ERR_STATE, "debug_residual: nothing kept for that layer");
  if (out) {
    if (n < per) return err(AHA_ERR_INVALID, "debug_residual: the buffer is too small");
    AHA_HIP_CHECK(hipStreamSynchronize(m->stream));
    AHA_HIP_CHECK(hipMemcpy(out, l.resid + (size_t)layer * per, per * 4, hipMemcpyDeviceToHost));
  }
  return (int64_t)l.resid_rows;
}

}  // namespace aha
