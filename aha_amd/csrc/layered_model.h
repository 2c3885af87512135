// State of a decoder whose config lists its layers, and the helpers its two stacks share: layered.hip (sequences, step, the post-norm stack) and
// layered_prenorm.hip.
#pragma once
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>

#include "common.h"
#include "kernels_prenorm.h"
#include "layered.h"

namespace aha {

inline int64_t round_up(int64_t v, int64_t m) { return (v + m - 1) / m * m; }

struct LWeights {
  void *wqkv = nullptr, *wo = nullptr, *wup = nullptr, *wdown = nullptr;   // bf16, rows and columns padded to 64
  float* bqkv_f32 = nullptr;
  void *norm1 = nullptr, *norm2 = nullptr, *qn = nullptr, *kn = nullptr, *conv1 = nullptr, *conv2 = nullptr;
  float lambda = 0.f, act[4] = {};
  // geometry
  int nq, nk, nv, k_off, v_off, nqkv;   // columns of the qkv projection (nqkv padded)
  int dq, dv, dvo, ldo;                 // page row widths, output head width, padded width of the attention output
  int o_ld;                             // elements between its rows: heads * dvo from the MFMA kernels (a GEMM's k pad then reads into the next row, times zero)
  int ffp = 0;
  bool frag = false;                    // fragment-major bf16 pages, MFMA attention
  bool fused_decode = false;            // attn_chunk_decode_kernel takes it
  uint64_t kv_off = 0;
  int rope = -1;                        // index of the (base, dims) table, -1: no rotation
  int v_store = 0, v_use = 0;
};

struct Seq {
  bool open = false;
  size_t len = 0;
  int hist = 0;                   // history that holds the state after `len` tokens
  std::vector<uint64_t> pages;    // logical page -> address, 0 once passed
  size_t first_live = 0;
};

struct RopeCfg { double base; int dims; };

// one layer of a pre-norm stack (layered_prenorm.hip)
struct PWeights {
  void *n1w = nullptr, *n1b = nullptr, *n2w = nullptr, *n2b = nullptr;
  void* wo = nullptr;
  int ko = 0;                           // padded columns of the output projection
  // state-space mixer
  SsmDims sd{};
  void* w_in = nullptr;
  int n_in = 0, c_off = 0, dt_off = 0;  // columns of the input projection (n_in padded)
  SsmParams sp{};
  void* gnorm = nullptr;
  int64_t hist_off = 0, state_off = 0;  // floats inside a slot's histories / a state pool entry
  // latent attention
  LatentDims la{};
  void *w_q = nullptr, *dkv_norm = nullptr, *w_ukv = nullptr, *w_ukt = nullptr, *w_uv = nullptr;
  int n_q = 0, kv_col = -1, n_ukv = 0;  // columns of q | latent | key part; of the expanded keys | values
  uint64_t kv_off = 0;
  int rope = -1, win = 0;               // index of the (base, dims) table, of the window
  bool prefill_ok = false, decode_ok = false;
  // feed-forward: gate and up rows in alternating blocks of 16.  wgu / wdown: the dense one, or the shared expert
  void *wgu = nullptr, *wdown = nullptr, *w_router = nullptr, *w_egu = nullptr, *w_edown = nullptr;
  int ffp = 0, effp = 0, ep = 0;        // padded widths; padded experts
};

struct LayeredModel {
  std::vector<LWeights> L;
  std::vector<PWeights> P;
  bool prenorm = false;
  void* final_norm_b = nullptr;
  void *embed = nullptr, *head = nullptr, *final_norm = nullptr;
  int64_t ld = 0;                 // padded width
  int Vp = 0;                     // padded vocabulary
  bool f32 = false;
  bool single_ok = false;         // the five-launch decode step takes every layer
  std::vector<RopeCfg> ropes;
  int max_half = 0, max_nqkv = 0, max_q = 0, max_o = 0, max_ffp = 0, max_nv = 0, max_part = 0, max_kvh = 0;
  // sequences
  std::vector<Seq> seqs;
  size_t slots = 0;
  uint64_t* d_tab = nullptr;      // (slots, tab_ld) page addresses
  size_t tab_ld = 0;
  float* d_hist = nullptr;        // (slots, layer, sublayer, CONV_HISTORIES, conv_taps, ld)
  int64_t hist_slot = 0;          // floats per slot
  // recurrent states: pool entries 0 .. CONV_HISTORIES - 1 are sequence 0's in rotation (its greedy loop runs ahead of the host), the others
  // belong to one slot each, updated in place
  float* d_pool = nullptr;
  int64_t pool_stride = 0;        // floats per entry
  float* seg = nullptr;           // states of a prompt's segments (launch_ssm_chunks)
  size_t seg_floats = 0;
  // step buffers, grown on demand
  size_t cap_rows = 0, cap_ents = 0, cap_want = 0;
  float *xa = nullptr, *xb = nullptr, *vfirst = nullptr, *logits = nullptr;
  float* am_max = nullptr;      // arg-max partials of the wanted rows
  uint32_t* am_idx = nullptr;
  void *h = nullptr, *qkv = nullptr, *q = nullptr, *o = nullptr, *z = nullptr, *y = nullptr, *fin = nullptr, *ws = nullptr;
  size_t ws_bytes = 0;
  std::vector<float*> ropetab;
  std::vector<void*> row_bufs, ent_bufs, want_bufs;
  char* d_meta = nullptr;         // entries | row_entry | ids | wanted rows | token argmaxes of the step
  char* h_meta = nullptr;         // pinned
  size_t meta_bytes = 0;
  float *part_o = nullptr, *part_ml = nullptr;
  unsigned* ctr = nullptr;
  // single-token buffers
  float *s1 = nullptr, *x1 = nullptr, *qkv1 = nullptr, *z1 = nullptr;
  float* zstats = nullptr;   // PolyNorm between two few-row products (SkinnyPoly)
  void* act1 = nullptr;
  // logits of the last batch
  size_t last_want = 0;
  // greedy loop
  size_t greedy_base = 0;
  SeqEntry* d_greedy = nullptr;
  size_t greedy_cap = 0;
  // pre-norm stacks: buffers of a step, sizes by layer maxima
  int max_proj = 0, max_cp = 0, max_dt = 0, max_yb = 0, max_qa = 0, max_slots = 0, max_effp = 0, max_ep = 0, max_lat_heads = 0, max_rp = 0, max_inner = 0;
  int64_t max_ldc = 0, max_ukv = 0;
  void *proj = nullptr, *u = nullptr, *yb = nullptr, *ob = nullptr, *qa = nullptr, *act = nullptr, *eact = nullptr, *ey = nullptr;
  float *dt = nullptr, *zr = nullptr, *gu = nullptr, *egu = nullptr, *ssq = nullptr;
  int32_t* route_ints = nullptr;
  size_t route_cap = 0;
  MoeRouting route{};
  void *lat = nullptr, *ukv = nullptr;
  size_t ext_cap = 0;
  std::vector<void*> ext_bufs;
  std::vector<int> windows;       // the layers' distinct windows
  const int32_t* ext_dev = nullptr;   // (windows, entries) first gathered row of every entry
  std::vector<int> ext_total, ext_max;
  // one token of one sequence: which layers' halves run together (kernels_prenorm_stack.hip); first < 0: this half by itself
  struct StackItem { int layer, half, first, n; double weights, states; };   // (elements of its matrices that a step reads, f32s of its states)
  std::vector<StackItem> schedule;
  PrenormOp* d_ops = nullptr;     // null: every half by itself
  int64_t stack_hist = 0;         // floats of a history of its state-space layers
  // debug
  bool keep = false;
  float* resid = nullptr;
  size_t resid_cap = 0, resid_rows = 0;
};

inline int err(int code, const std::string& msg) {
  set_error(msg);
  return code;
}

// (rows, cols) bf16 weights into a zeroed (rows_p, ld) matrix
inline int new_matrix(aha_model* m, int64_t rows_p, int64_t ld, void** out) { return dev_alloc(m, (size_t)rows_p * ld * 2, out, true); }
inline int put_block(aha_model* m, const aha_tensor_view* t, int64_t rows, int64_t cols, int64_t c0, int64_t nc, void* dst, int64_t row0, int64_t col0, int64_t ld) {
  std::vector<uint16_t> tmp;
  const void* src;
  int rc = bf16_source(t, rows * cols, tmp, &src);
  if (rc) return rc;
  AHA_HIP_CHECK(hipStreamSynchronize(m->stream));   // (the zero fill)
  AHA_HIP_CHECK(hipMemcpy2D((char*)dst + (size_t)(row0 * ld + col0) * 2, (size_t)ld * 2, (const char*)src + (size_t)c0 * 2, (size_t)cols * 2, (size_t)nc * 2,
                            (size_t)rows, hipMemcpyDefault));
  return AHA_OK;
}
inline int put_matrix(aha_model* m, const aha_tensor_view* t, int64_t rows, int64_t cols, int64_t rows_p, int64_t ld, void** out) {
  int rc = new_matrix(m, rows_p, ld, out);
  return rc ? rc : put_block(m, t, rows, cols, 0, cols, *out, 0, 0, ld);
}
// a small tensor on the host, bf16 bit patterns
inline int host_bf16(const aha_tensor_view* t, int64_t n, std::vector<uint16_t>* out) {
  std::vector<uint16_t> tmp;
  const void* src;
  int rc = bf16_source(t, n, tmp, &src);
  if (rc) return rc;
  out->resize((size_t)n);
  AHA_HIP_CHECK(hipMemcpy(out->data(), src, (size_t)n * 2, hipMemcpyDefault));
  return AHA_OK;
}
inline float bf_host(uint16_t v) {
  const uint32_t u = (uint32_t)v << 16;
  float f;
  memcpy(&f, &u, 4);
  return f;
}

inline int free_list(aha_model* m, std::vector<void*>& v) {
  AHA_HIP_CHECK(hipStreamSynchronize(m->stream));
  for (void* p : v) hipFree(p);
  v.clear();
  return AHA_OK;
}
// zero-filled: pad columns and masked value slots are multiplied by zero weights and must be finite
inline int grow(aha_model* m, std::vector<void*>& owner, size_t bytes, void** out) {
  void* p = nullptr;
  const hipError_t e = hipMalloc(&p, bytes ? bytes : 16);
  if (e != hipSuccess) return err(e == hipErrorOutOfMemory ? AHA_ERR_OOM : AHA_ERR_HIP, std::string("step buffer hipMalloc failed: ") + hipGetErrorString(e));
  owner.push_back(p);
  AHA_HIP_CHECK(hipMemsetAsync(p, 0, bytes ? bytes : 16, m->stream));
  *out = p;
  return AHA_OK;
}

inline GemmArgs gemm_args(const void* A, int64_t lda, const void* W, void* C, int64_t ldc, int M, int N, int K, int act = ACT_NONE) {
  GemmArgs g{};
  g.A = A; g.W = W; g.C = C;
  g.M = M; g.N = N; g.K = K; g.lda = lda; g.ldw = K; g.ldc = ldc; g.act = act;
  return g;
}
inline void gemm(aha_model* m, const void* A, int64_t lda, const void* W, void* C, int64_t ldc, int M, int N, int K, int act = ACT_NONE) {
  const LayeredModel& l = *m->layered;
  ProfScope ps(m, "gemm", ((double)M * K + (double)M * N) * (l.f32 ? 4 : 2) + (double)N * K * 2, 2.0 * M * N * K);
  if (l.f32) {
    launch_gemm_f32((const float*)A, lda, W, K, (float*)C, ldc, M, N, K, m->stream);
    return;
  }
  launch_gemm(gemm_args(A, lda, W, C, ldc, M, N, K, act), m->stream);
}

inline void keep_rows(aha_model* m, const float* x, int rows, int layer) {
  LayeredModel& l = *m->layered;
  if (!l.keep || layer < 0) return;
  hipMemcpy2DAsync(l.resid + (size_t)layer * rows * m->desc.hidden_size, (size_t)m->desc.hidden_size * 4, x, (size_t)l.ld * 4, (size_t)m->desc.hidden_size * 4, rows,
                   hipMemcpyDeviceToDevice, m->stream);
}
// what the last sublayer left
struct Tail {
  const float* x;      // post-norm: the residual stream before its norm; pre-norm: the stream without the pending rows
  const void* y;       // post-norm: null: x already holds alpha x + y
  const void* norm;
  float alpha;
  PendingAdd add;      // pre-norm
};

// layered_prenorm.hip
int prenorm_check(const aha_model_desc& c);
int prenorm_create(aha_model* m, const aha_tensor_view* w, size_t nw, uint64_t* kv_bytes);
bool prenorm_single_ok(const aha_model* m);
int prenorm_alloc_single(aha_model* m);
int prenorm_ensure_rows(aha_model* m, size_t cap);
int prenorm_ensure_entries(aha_model* m, size_t cap);
int prenorm_prepare_ext(aha_model* m, const SeqEntry* e, size_t n, int32_t* host_out);
Tail prenorm_rows(aha_model* m, const SeqBatch& b, const SeqEntry* h_ents, const uint32_t* ids);
void prenorm_final(aha_model* m, const Tail& t, const int32_t* rows, int n);

}  // namespace aha
