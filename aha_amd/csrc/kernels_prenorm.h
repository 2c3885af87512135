// Launchers of the pre-norm layer-list decoders' kernels (layered_prenorm.hip): LayerNorm rows, state-space mixer, latent attention, routed
// experts.  Activation type: bf16, or float with f32 = true; all other operands have the type their comment names.
#pragma once
#include "kernels.h"

namespace aha {

// ---- residual stream and norms (kernels_prenorm.hip) ---------------------------------------------------------------------------------
// What the f32 residual stream still lacks: a dense sublayer's output rows, and the rows of the experts each token used
struct PendingAdd {
  const void* y = nullptr;           // (rows, ldy)
  int64_t ldy = 0;
  const void* slots = nullptr;       // (rows * top, ld_slots): expert outputs by slot
  const int32_t* slot_of = nullptr;  // (rows, top)
  int top = 0;
  int64_t ld_slots = 0;
};
// x = x_in + pending (or embed row * scale); h = LayerNorm(x) * w + b.  Row i of the output is row (row_list ? row_list[i] : i).
struct PreNormArgs {
  const float* x_in = nullptr;       // (rows, ld)
  PendingAdd add;
  const void* embed = nullptr;       // (V, ld) bf16
  const uint32_t* ids = nullptr;
  float embed_scale = 1.f;
  const void *w = nullptr, *b = nullptr;   // (ld) bf16, zero behind width
  float eps = 0.f;
  float* x_out = nullptr;            // (rows, ld), may alias x_in; null: not written
  void* h_out = nullptr;             // (rows, ld); null: not written
  const int32_t* row_list = nullptr;
  int width = 0, rows = 0;
  int64_t ld = 0;                    // a multiple of 256, at most 8192
  int32_t* zero = nullptr;           // n_zero counters cleared on the way (for the routing kernels behind)
  int n_zero = 0;
};
void launch_prenorm_rows(const PreNormArgs& a, bool f32, hipStream_t st);
// out[r][j] = silu(w g) * (w u); gu rows hold 16-column blocks alternating gate / up; w = row_w[r], or 1
void launch_silu_pairs(const float* gu, int64_t ld_gu, float* out, int64_t ld_out, int rows, int ff, const float* row_w, hipStream_t st);
// z <- cap tanh(z / cap)
void launch_softcap(float* z, int64_t n, float cap, hipStream_t st);

// ---- state-space mixer (kernels_ssm.hip) -----------------------------------------------------------------------------------------------
// Everything is padded: a head's vdim to vdp (multiple of 16), a group's state to np (multiple of 32); pad channels carry zeros throughout.
// Channels of the short convolution: [x: heads * vdp | B: groups * np | C: groups * np] = cp columns.
// Recurrent state, f32: [head][vdp / 16][np][16] per (model layer, pool index).
struct SsmDims {
  int heads, vdim, vdp, groups, state, np, norm_groups, taps;
  __host__ __device__ int inner() const { return heads * vdp; }
  __host__ __device__ int cp() const { return heads * vdp + 2 * groups * np; }
  __host__ __device__ int64_t state_floats() const { return (int64_t)heads * vdp * np; }
};
// input projection rows: z at column 0, the convolution's channels at c_off, step sizes at dt_off
struct SsmIn {
  const void* p;
  int64_t ld;
  int c_off, dt_off;
};
// the mixer's small parameters, f32: convolution weights (taps, cp) and bias (cp), per head dt_bias, a = -exp(A_log), d
struct SsmParams {
  const float *conv_w, *conv_b, *dt_bias, *a, *d;
};
struct SsmHist {
  float* hist;                       // this layer's convolution inputs: slot * slot_stride + which * (taps - 1) * cp, row i = i + 1 tokens back
  int64_t slot_stride;
};
struct SsmState {
  float* state;                      // this layer's states: pool index * pool_stride
  int64_t pool_stride;
};
// u = silu(conv(x | B | C)) for every row, dt = softplus(dt + bias) as [head][dt_ld]; the sequences' histories move on
struct ShortConvArgs {
  SsmDims d;
  SsmIn in;
  SsmParams p;
  SsmHist h;
  void* u;                           // (rows, cp)
  float* dt;
  int64_t dt_ld;
};
void launch_short_conv(const ShortConvArgs& a, const SeqBatch& b, bool f32, hipStream_t st);
// the recurrence over every entry's rows: y = S^T C + D x
struct SsmScanArgs {
  SsmDims d;
  SsmParams p;
  SsmState s;
  const void* u;                     // (rows, cp)
  const float* dt;
  int64_t dt_ld;
  void* y;                           // (rows, ldy)
  int64_t ldy;
};
struct SsmSegments {
  float* state;                      // [entry][segment][state]
  float* cum;                        // [entry][segment][head]: sum of a dt
  int n, chunks;                     // segments per entry, chunks per segment
};
bool ssm_chunk_ok(const SsmDims& d);                                                         // sizes launch_ssm_chunks and launch_ssm_step take
size_t ssm_segment_floats(const SsmDims& d);                                                 // scratch with which no prompt runs in fewer segments than it could
// bf16 rows, 64 tokens at a time on the matrix cores; long prompts in segments beside each other, whose states are in `scratch`
void launch_ssm_chunks(const SsmScanArgs& a, const SeqBatch& b, float* scratch, size_t scratch_floats, hipStream_t st);
void launch_ssm_scan(const SsmScanArgs& a, const SeqBatch& b, bool f32, hipStream_t st);     // token by token, any sizes
// one token per sequence: convolution, step size, recurrence and gate in one launch
struct SsmStepArgs {
  SsmDims d;
  SsmIn in;
  int in_f32;                        // in.p is f32 (behind the decode matvec) / bf16 (behind a GEMM)
  SsmParams p;
  SsmHist h;
  SsmState s;
  float* g;                          // (n, heads * vdp): y * silu(z)
  float* ssq;                        // (n, heads * vdp / 16): sums of squares of 16 columns each
};
void launch_ssm_step(const SsmStepArgs& a, const SeqBatch& b, hipStream_t st);
// out = norm over norm_groups equal parts of (y * silu(z)) * w; z null: y is gated already (f32, ld = inner)
struct GatedNormArgs {
  SsmDims d;
  const void* y;
  int64_t ldy;
  const void* z;
  int64_t ldz;
  const void* w;                     // (inner) bf16
  void* out;                         // (rows, ldo)
  int64_t ldo;
  float eps;
  int rows;
};
void launch_gated_norm(const GatedNormArgs& a, bool f32, hipStream_t st);

// ---- latent attention (kernels_latent.hip) ---------------------------------------------------------------------------------------------
// Cached per token: [latent: rp | rotated key part: tp], activation type, token-major pages of 64 rows (rp a multiple of 64, tp of 32, pads zero).
// A head's query: [unrotated: dp | rotated: tp].
struct LatentDims {
  int heads, dim, dp, rot, tp, vdim, vp, rank, rp, window;
  float scale;
  __host__ __device__ int qd() const { return dp + tp; }
  __host__ __device__ int64_t ldc() const { return rp + tp; }
  __host__ __device__ int first(int pos) const { return window > 0 && pos >= window ? pos - window + 1 : 0; }   // first position `pos` sees
};
struct LatentCache {
  const uint64_t* tab;               // page p of slot s at tab[s * ld + p] + off
  int64_t ld;
  uint64_t off;
};
// q: rotation of every head's last dims; latent: norm, key part: rotation, append (kv_off < 0: the cache belongs to another layer)
struct LatentPostArgs {
  LatentDims d;
  const void* in;                    // (rows, ld): [q: heads * qd | latent | key part at kv_off]
  int64_t ld;
  int kv_off;
  int in_f32;                        // in is f32 whatever the activation type (behind the decode matvec)
  const void* norm_w;                // (rp) bf16
  float eps;
  const float* rope;                 // (rows, rot / 2, 2)
  void* q;                           // (rows, heads * qd), pitch ldq: `in` itself (only the rotated dims are written)
  int64_t ldq;
  LatentCache c;
};
void launch_latent_post(const LatentPostArgs& a, const SeqBatch& b, bool f32, hipStream_t st);
// C[r][h * sc + j] = sum_k A[r][h * sa + k] W[h][j][k] for every head; bf16, n a multiple of 64, k of 32
struct HeadsGemmArgs {
  const void* A;
  int64_t lda, sa;
  const void* W;                     // (heads, n, k) bf16
  void* C;
  int64_t ldc, sc;
  int rows, heads, n, k;
};
void launch_heads_gemm(const HeadsGemmArgs& a, bool f32, hipStream_t st);
// attention in the latent space, any sizes: o[r][h] = sum_j p_j c_j, scores qa . c + q_rot . k_rot
struct LatentRowsArgs {
  LatentDims d;
  const void* qa;                    // (rows, heads, rp)
  const void* q;                     // (rows, ldq), head h's rotated part at h * qd + dp
  int64_t ldq;
  void* o;                           // (rows, heads, rp)
  LatentCache c;
};
void launch_latent_rows(const LatentRowsArgs& a, const SeqBatch& b, bool f32, hipStream_t st);
// cached rows first(pos0) & ~63 .. pos0 + len of every entry, gathered: row ext0[entry] on
void launch_latent_gather(const LatentDims& d, const LatentCache& c, const int32_t* ext0, void* out, const SeqBatch& b, int max_rows, bool f32, hipStream_t st);
// prompts: keys and values expanded per head
struct LatentPrefillArgs {
  LatentDims d;
  const void* q;                     // (rows, ldq) bf16
  int64_t ldq;
  const void* kv;                    // (ext rows, heads * (dp + vp)): unrotated keys by head, then values by head
  const void* lat;                   // (ext rows, ldc): the gathered cache rows (key part at rp)
  const int32_t* ext0;
  void* o;                           // (rows, ldo), head h at h * vp
  int64_t ldo;
};
bool latent_prefill_dims(int dim, int rot, int vdim, int* dp, int* tp, int* vp);   // padded dims of the kernel, false: no instantiation
void launch_latent_prefill(const LatentPrefillArgs& a, const SeqBatch& b, hipStream_t st);
// one token per sequence: the queries' unrotated part taken into the latent space (W_uk_h^T q), rotation, and the token's cache row as
// launch_latent_post does it, in one launch
struct LatentQueryArgs {
  LatentPostArgs p;                  // p.q, p.ldq unused
  const void* w_ukt;                 // (heads, rp, dp) bf16
  void* qa;                          // (n, heads, rp) bf16
  void* qr;                          // (n, heads, tp) bf16
};
void launch_latent_query(const LatentQueryArgs& a, const SeqBatch& b, hipStream_t st);
// one token per sequence, in the latent space: split partials (un-normalised), then launch_latent_merge
struct LatentDecodeArgs {
  LatentDims d;
  const void* qa;                    // (n, heads, rp) bf16
  const void* qr;                    // (n, heads, tp) bf16
  LatentCache c;
  float* part_o;                     // (n, nsplit, heads, rp)
  float* part_ml;                    // (n, nsplit, heads, 2)
  int nsplit;
};
constexpr int LATENT_MAX_SPLIT = 64;
int latent_decode_blocks_per_cu(const LatentDims& d);   // 1 or 2
bool latent_decode_ok(const LatentDims& d);
void launch_latent_decode(const LatentDecodeArgs& a, const SeqBatch& b, hipStream_t st);
// o[r][h * vp + j] = sum_k merged latent[r][h][k] W_uv[h][j][k]
struct LatentMergeArgs {
  LatentDims d;
  const float* part_o;
  const float* part_ml;
  int nsplit;
  const void* wuv;                   // (heads, vp, rp) bf16
  void* o;                           // (n, ldo) bf16
  int64_t ldo;
  int n;
};
void launch_latent_merge(const LatentMergeArgs& a, hipStream_t st);

// ---- routed experts (kernels_moe.hip) --------------------------------------------------------------------------------------------------
// A step's routing, device side.  counts / cursor: (experts), zero before launch_moe_route.
struct MoeRouting {
  int32_t* counts;
  int32_t* cursor;
  int32_t* sel;                      // (rows, top) experts
  float* sel_w;                      // (rows, top) scores
  int32_t* slot_of;                  // (rows, top)
  int32_t* slot_row;                 // (rows * top) by slot; an expert's slots are consecutive
  float* slot_w;
  int32_t* tiles;                    // (max tiles, 3): expert, first slot, slots
  int32_t* n_tiles;
};
int moe_max_tiles(int rows, int top, int experts, int bm);
// sigmoid scores of the router logits (rows, ldz) f32, the `top` largest, slots grouped by expert, tiles of bm slots
void launch_moe_route(const float* z, int64_t ldz, int rows, int experts, int top, int bm, const MoeRouting& r, hipStream_t st);
struct MoeGemmArgs {
  const void* A;                     // up: (rows, lda) gathered by slot_row; down: (slots, lda)
  int64_t lda;
  const void* W;                     // (experts, n, k) bf16
  void* C;                           // (slots, ldc)
  int64_t ldc;
  int n, k;                          // multiples of 64
  int slots, experts;                // rows * top
  int gather;                        // A rows through slot_row
  int pairs;                         // bf16: silu(w g) * (w u) of the 16-column gate / up blocks, C has n / 2 columns; f32: always plain
};
int moe_tile_rows(int slots, int experts, bool f32);   // the bm to route with: 32 (few slots per expert), 64, 128 or 256 (many)
void launch_moe_gemm(const MoeGemmArgs& a, const MoeRouting& r, int bm, bool f32, hipStream_t st);
void launch_moe_gemm256(const MoeGemmArgs& a, const MoeRouting& r, int max_tiles, hipStream_t st);   // bf16, tiles of 256 slots (kernels_moe256.hip)

// ---- decode matvecs (kernels_gemv_prenorm.hip, kernels_gemv_experts.hip) --------------------------------------------------------------------------
// h = LayerNorm(x): x (K) f32, w / b (K) bf16, zero behind width.  Epilogues GEMV_PARTIAL_F32 and GEMV_SILU_MUL
struct GemvLayerNorm {
  const float* x;
  const void *w, *b;
  float eps;
  int width;
};
void launch_gemv_layernorm(const GemvArgs& a, const GemvLayerNorm& p, GemvEpi epi, hipStream_t st);
// h = g / rms(part) * w: g (n) f32 in `parts` runs of n / parts columns (each a multiple of 16), ssq (n / 16) their sums of squares, `part` real
// columns per part.  GEMV_AXPY_F32
struct GemvPartsNorm {
  const float *g, *ssq;
  const void* w;
  float eps;
  int n, parts, part;
};
void launch_gemv_partsnorm(const GemvArgs& a, const GemvPartsNorm& p, hipStream_t st);
// y (bf16) = act(w gate h) * (w up h) of the chosen experts, one after the other, and of the shared one (w = 1): a.N = top * effp + ffp
struct GemvExperts {
  const float* z;                    // router logits
  const void *w_experts, *w_shared;  // (experts, 2 effp, K), (2 ffp, K): gate and up rows in alternating blocks of 16; effp, ffp multiples of 64
  int experts, top, effp;
  int32_t* sel;                      // (top) out
};
void launch_gemv_experts_up(const GemvArgs& a, const GemvLayerNorm& p, const GemvExperts& e, hipStream_t st);
// y = res + sum over the choices of W_down x_choice + W_down_shared x_shared, x (bf16) as above: a.K = top * effp + ffp
struct GemvExpertsDown {
  const void *w_experts, *w_shared;  // (experts, n_rows, effp), (n_rows, ffp)
  const int32_t* sel;
  int top, effp, ffp, n_rows;
};
void launch_gemv_experts_down(const GemvArgs& a, const GemvExpertsDown& d, hipStream_t st);

// ---- runs of sublayers of one token of one sequence in one launch (kernels_prenorm_stack.hip) ----------------------------------------------------
enum { PRENORM_SSM, PRENORM_DENSE, PRENORM_MOE };
struct PrenormOp {                   // a sublayer; what its kind does not have is null
  int kind;
  const void *w1, *w2;               // input and output projection; gate / up and down (of the shared expert)
  const void *nw, *nb;               // the norm in front
  const float* par;                  // f32: convolution weights (taps, cp), bias (cp), per head dt_bias, a, d
  const void* gnorm;
  int64_t hist, state;               // floats in front of the layer's share of the histories and states
  const void *router, *egu, *edown;
};
constexpr int PRENORM_STACK_OPS = 16;   // of a launch, at most
struct PrenormStackArgs {
  const PrenormOp* ops;              // device memory
  const float* x_in;                 // (1024): the residual stream in front of the first sublayer and behind the last; may be the same
  float* x_out;
  const float *hist_in, *state_in;   // the sequence's histories and states, and where the step leaves them (elsewhere)
  float *hist_out, *state_out;
  unsigned* exchange;
  unsigned *fail_dev, *fail_host;    // as DecodeStackArgs
  uint32_t epoch;
  int n_ops, pos0, polls;
  float eps;
};
bool prenorm_stack_width_ok(int64_t ld, int width);
bool prenorm_stack_ssm_ok(const SsmDims& d, int n_out);
bool prenorm_stack_dense_ok(int ff);
bool prenorm_stack_moe_ok(int experts, int top, int ff, int shared_ff);
void launch_prenorm_stack(const PrenormStackArgs& a, hipStream_t st);

}  // namespace aha
