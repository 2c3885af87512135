// State-space (Mamba-2) mixer of the layer-list decoders: per head a state S (state x vdim) with
//   S_t = exp(a dt_t) S_(t-1) + dt_t B_t x_t^T,   y_t = S_t^T C_t + D x_t,   a < 0,   dt = softplus(.),   x | B | C = silu(conv(.))
//   short_conv_kernel   the convolution of a step's rows, step sizes, histories
//   ssm_chunk_kernel    prompts, bf16: 64 tokens at a time on the matrix cores
//   ssm_scan_kernel     any sizes / the 32-bit mode: token by token
//   ssm_step_kernel     one token per sequence: convolution + recurrence + gate
//   gated_norm_kernel   (y silu(z)) normed in equal parts
// Step sizes, decays, exponentials and the state are f32.
#include <math.h>

#include <algorithm>

#include <type_traits>

#include "attn_common.h"
#include "kernels_prenorm.h"
#include "rows_common.h"

namespace aha {

namespace {

__device__ __forceinline__ float softplus_f32(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }

template <typename T>
__device__ __forceinline__ void ld8(const T* p, float (&f)[8]) {
  const float4 a = Act<T>::ld4(p), b = Act<T>::ld4(p + 4);
  f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
}

// ---- short convolution -----------------------------------------------------------------------------------------------------------------
// A thread walks `tile` rows of eight channels; the taps - 1 inputs in front of a row come from its own registers, the step's rows or the
// sequence's history.  Thread items: (tile, channel group), then one per (row, head) for the step sizes.
constexpr int MAX_TAPS_REG = 4;
template <typename T, int TAPS>   // TAPS 0: any number, every input read again
__global__ __launch_bounds__(256) void short_conv_kernel(ShortConvArgs a, SeqBatch b, int tile, int64_t conv_items) {
  const int64_t item = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int cp = a.d.cp(), ng = cp >> 3, taps = TAPS ? TAPS : a.d.taps;
  if (item >= conv_items) {
    const int64_t k = item - conv_items;
    const int r = (int)(k % b.rows), h = (int)(k / b.rows);
    if (h >= a.d.heads) return;
    const float z = Act<T>::ld((const T*)a.in.p + (int64_t)r * a.in.ld + a.in.dt_off + h) + a.p.dt_bias[h];
    a.dt[(int64_t)h * a.dt_ld + r] = softplus_f32(z);
    return;
  }
  const int cg = (int)(item % ng), r0 = (int)(item / ng) * tile, r1 = min(r0 + tile, b.rows), c0 = cg * 8;
  const T* in = (const T*)a.in.p + a.in.c_off + c0;
  float bias[8], w[TAPS ? TAPS : 1][8];
#pragma unroll
  for (int j = 0; j < 8; ++j) bias[j] = a.p.conv_b[c0 + j];
  if constexpr (TAPS > 0) {
#pragma unroll
    for (int t = 0; t < TAPS; ++t) ld8<float>(a.p.conv_w + (int64_t)t * cp + c0, w[t]);
  }
  int ei = entry_of_row(b, r0);
  SeqEntry e = seq_entry_at(b, ei);
  auto hist = [&](int which) { return a.h.hist + (int64_t)e.slot * a.h.slot_stride + (int64_t)which * (taps - 1) * cp + c0; };
  // the input of row r, or of the entry's tokens in front of it
  auto input = [&](int rel, float (&f)[8]) {
    if (rel >= 0) {
      ld8<T>(in + (int64_t)(e.row0 + rel) * a.in.ld, f);
    } else if (e.pos0 + rel >= 0) {
      ld8<float>(hist(e.hist_in) + (int64_t)(-rel - 1) * cp, f);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = 0.f;
    }
  };
  float back[TAPS > 1 ? TAPS - 1 : 1][8];   // back[q] = the input q + 1 tokens in front of the current row
  auto row = [&](int r, const float (&cur)[8]) {
    const int rel = r - e.row0;
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = bias[j];
    if constexpr (TAPS > 0) {
#pragma unroll
      for (int q = TAPS - 2; q >= 0; --q)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = fmaf(w[TAPS - 2 - q][j], back[q][j], acc[j]);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] = fmaf(w[TAPS - 1][j], cur[j], acc[j]);
    } else {
      for (int t = 0; t < taps; ++t) {
        float x[8], wt[8];
        input(rel - (taps - 1 - t), x);
        ld8<float>(a.p.conv_w + (int64_t)t * cp + c0, wt);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = fmaf(wt[j], x[j], acc[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = silu_rows<T>(acc[j]);
    T* u = (T*)a.u + (int64_t)r * cp + c0;
    Act<T>::st4(u, make_float4(acc[0], acc[1], acc[2], acc[3]));
    Act<T>::st4(u + 4, make_float4(acc[4], acc[5], acc[6], acc[7]));
    if (rel == e.len - 1) {   // history for the next step
      float* ho = hist(e.hist_out);
      for (int q = 0; q < taps - 1; ++q) {
        float x[8];
        input(rel - q, x);
        *reinterpret_cast<float4*>(ho + (int64_t)q * cp) = make_float4(x[0], x[1], x[2], x[3]);
        *reinterpret_cast<float4*>(ho + (int64_t)q * cp + 4) = make_float4(x[4], x[5], x[6], x[7]);
      }
    }
    if constexpr (TAPS > 1) {
#pragma unroll
      for (int q = TAPS - 2; q > 0; --q)
#pragma unroll
        for (int j = 0; j < 8; ++j) back[q][j] = back[q - 1][j];
#pragma unroll
      for (int j = 0; j < 8; ++j) back[0][j] = cur[j];
    }
  };
  for (int r = r0; r < r1;) {   // up to four rows of one entry, requested together
    if (r > r0 && r == e.row0 + e.len) e = seq_entry_at(b, ++ei);
    if (TAPS > 1 && (r == r0 || r == e.row0)) {
#pragma unroll
      for (int q = 0; q < TAPS - 1; ++q) input(r - e.row0 - 1 - q, back[q]);
    }
    const int n = min(min(r1, e.row0 + e.len) - r, 4);
    float cur[4][8];
#pragma unroll
    for (int q = 0; q < 4; ++q) ld8<T>(in + (int64_t)(r + min(q, n - 1)) * a.in.ld, cur[q]);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q < n) row(r + q, cur[q]);
    r += n;
  }
}

// ---- token by token ----------------------------------------------------------------------------------------------------------------------
// Block (head and 16 of its columns, entry): thread (n group, column) keeps rows n = group, group + 16, ... of its column of the state in LDS.
template <typename T>
__global__ __launch_bounds__(256) void ssm_scan_kernel(SsmScanArgs a, SeqBatch b) {
  extern __shared__ __attribute__((aligned(16))) float st[];   // [np][16]
  __shared__ float red[2][4][16];
  const int tid = threadIdx.x, v = tid & 15, g = tid >> 4, nvs = a.d.vdp >> 4, h = blockIdx.x / nvs, vs = blockIdx.x - h * nvs, np = a.d.np;
  const SeqEntry e = seq_entry_at(b, blockIdx.y);
  const int cp = a.d.cp(), inner = a.d.inner(), grp = h / (a.d.heads / a.d.groups);
  const float A = a.p.a[h], D = a.p.d[h];
  const int64_t so = ((int64_t)h * nvs + vs) * np * 16;
  const float* sin = a.s.state + (int64_t)e.state_in * a.s.pool_stride + so;
  float* sout = a.s.state + (int64_t)e.state_out * a.s.pool_stride + so;
  for (int n = g; n < np; n += 16) st[n * 16 + v] = e.pos0 > 0 ? sin[n * 16 + v] : 0.f;
  for (int i = 0; i < e.len; ++i) {
    const int64_t r = e.row0 + i;
    const T* u = (const T*)a.u + r * cp;
    const float dt = a.dt[(int64_t)h * a.dt_ld + r], da = expf(A * dt), x = Act<T>::ld(u + h * a.d.vdp + vs * 16 + v), dx = dt * x;
    const T *B = u + inner + grp * np, *C = B + a.d.groups * np;
    float y = 0.f;
    for (int n = g; n < np; n += 16) {
      const float s = fmaf(Act<T>::ld(B + n), dx, da * st[n * 16 + v]);
      st[n * 16 + v] = s;
      y = fmaf(Act<T>::ld(C + n), s, y);
    }
    y += __shfl_xor(y, 16, 64);
    y += __shfl_xor(y, 32, 64);
    if ((tid & 48) == 0) red[i & 1][tid >> 6][v] = y;
    __syncthreads();
    if (tid < 16) {
      const float s = (red[i & 1][0][v] + red[i & 1][1][v]) + (red[i & 1][2][v] + red[i & 1][3][v]);
      Act<T>::st((T*)a.y + r * a.ldy + h * a.d.vdp + vs * 16 + v, fmaf(D, x, s));
    }
  }
  for (int n = g; n < np; n += 16) sout[n * 16 + v] = st[n * 16 + v];
}

// ---- prompts: 64 tokens at a time ----------------------------------------------------------------------------------------------------------
// With cum_t = sum of a dt over the chunk's tokens up to t:
//   y_t = exp(cum_t) S^T C_t + sum_(s <= t) exp(cum_t - cum_s) dt_s (B_s . C_t) x_s + D x_t
//   S  <- exp(cum_last) S + sum_s (exp(cum_last - cum_s) dt_s B_s) x_s^T
// Block (head and VT * 16 of its columns, entry), four waves, walking the entry's chunks in order with the state in f32 accumulators.  B, C and x
// are bf16; the other operand of each product (weights of the pairs, weighted B, the state) is f32 and goes to the matrix cores as the sum of two
// bf16, high and low half, so that the products keep 16 bits of it.
// Fragments: as in attention (common.h), with B in the role of K, C of Q, x of V: wave w computes the outputs of tokens w * 16 .. of the chunk,
// (B_s . C_t) transposed, so that its accumulators are the next product's operand; transposed reads of x and B by ds_read_b64_tr_b16.
// The state's rows (np / 16 tiles of 16) are dealt to the waves.  A chunk's rows are requested into registers one chunk ahead.
// Long prompts are cut into segments of whole chunks that run beside each other: STATE_ONLY finds what every segment but the last adds to the state
// from zero, ssm_segments_kernel turns these into the segments' first states, then every segment runs from its own.
typedef short __attribute__((ext_vector_type(4))) tr4_t;
typedef __attribute__((address_space(3))) tr4_t* lds_tr_t;
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* glb_ptr_t;

// eight values f -> bf16 high halves and the bf16 rest
__device__ __forceinline__ void split8(const float (&f)[8], bf16x8_t& hi, bf16x8_t& lo) {
  u32x4_t h, l;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    h[j] = pack_bf(f[2 * j], f[2 * j + 1]);
    l[j] = pack_bf(f[2 * j] - lo_bf(h[j]), f[2 * j + 1] - hi_bf(h[j]));
  }
  hi = as_frag(h);
  lo = as_frag(l);
}

__device__ __forceinline__ float wave_prefix_sum(float x) {   // inclusive
  auto add = [&](auto ctrl, auto rows) { x += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(x), decltype(ctrl)::value, decltype(rows)::value, 0xf, false)); };
  using std::integral_constant;
  add(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});   // row_shr:1, 2, 4, 8: within 16 lanes
  add(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});
  add(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});
  add(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});
  add(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});   // row_bcast:15 into the odd rows
  add(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});   // row_bcast:31 into the upper half
  return x;
}

constexpr int SSM_XV = 64 * 32 + 64;   // bytes of 16 columns of x, 64 tokens (and a pad between them)
template <int KS, int VT>
constexpr int ssm_chunk_lds(bool state_only) { return KS * 4096 + VT * SSM_XV + (state_only ? 0 : VT * KS * 2048) + 3 * 64 * 4; }

template <int KS, int VT, bool STATE_ONLY>   // KS = np / 32
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void ssm_chunk_kernel(SsmScanArgs a, SeqBatch b, SsmSegments sg) {
  constexpr int NT = KS * 2, NTW = (NT + 3) / 4;   // state row tiles, per wave
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* const cums = reinterpret_cast<float*>(smem);   // [64] cum, [64] dt, [64] exp(cum_last - cum) dt
  char* const Bs = smem + 3 * 64 * 4;              // [4 token tiles][KS] fragments of 1 KB
  char* const Xs = Bs + KS * 4096;                 // [VT] x [64 tokens][16]
  char* const Sh = Xs + VT * SSM_XV;               // [VT][KS] fragments of the state's high halves, then the low ones
  char* const Sl = Sh + VT * KS * 1024;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), G = lane >> 4, c = lane & 15;
  const int nvs = a.d.vdp / (16 * VT), np = KS * 32;
  int wk = blockIdx.x;
  if (gridDim.x % 8 == 0) wk = (wk & 7) * (int)(gridDim.x >> 3) + (wk >> 3);   // neighbouring heads (they share B and C) on one XCD
  const int h = wk / nvs, vs = wk - h * nvs;
  const int entry = blockIdx.y / sg.n, seg = blockIdx.y - entry * sg.n;
  const SeqEntry e = seq_entry_at(b, entry);
  const int nchunk = (e.len + 63) >> 6, ch0 = seg * sg.chunks, ch1 = min(ch0 + sg.chunks, nchunk);
  if (ch0 >= nchunk || (STATE_ONLY && ch1 == nchunk)) return;   // (uniform over the block)
  const int cp = a.d.cp(), inner = a.d.inner(), grp = h / (a.d.heads / a.d.groups), xc = h * a.d.vdp + vs * VT * 16;
  const float A = a.p.a[h], D = a.p.d[h];
  const bf16_t* u = (const bf16_t*)a.u;
  const int64_t so = ((int64_t)h * (a.d.vdp >> 4) + vs * VT) * np * 16;   // [VT][np][16]
  float* const seg_state = sg.n > 1 ? sg.state + (int64_t)blockIdx.y * a.d.state_floats() + so : nullptr;
  const float* first = sg.n > 1 ? seg_state : e.pos0 > 0 ? a.s.state + (int64_t)e.state_in * a.s.pool_stride + so : nullptr;
  if (STATE_ONLY) first = nullptr;
  f32x4_t S[NTW][VT];   // rows nt * 16 + G * 4 + r, column c
#pragma unroll
  for (int j = 0; j < NTW; ++j)
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) {
      S[j][vt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      const int nt = wave + j * 4;
      if (first && nt < NT) {
        const float* p = first + ((int64_t)vt * np + nt * 16 + G * 4) * 16 + c;
#pragma unroll
        for (int r = 0; r < 4; ++r) S[j][vt][r] = p[r * 16];
      }
    }
  // 4 tokens x 16 columns per lane group, transposed: lane (G, c) gets column c of tokens G * 4 .. + 4
  const int tr_row = G * 4 + (c >> 2), tr_col = (c & 3) * 4;
  auto tr_pair = [&](const char* p0, const char* p1) {
    const tr4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)p0), hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)p1);
    union { tr4_t t[2]; u32x4_t u; } x;
    x.t[0] = lo; x.t[1] = hi;
    return x.u;
  };
  auto x_frag = [&](int vt, int kk) {   // x^T: column vt * 16 + c, tokens kk * 32 + G * 4 + {0..3, 16..19}
    const char* p = Xs + vt * SSM_XV + (kk * 32 + tr_row) * 32 + tr_col * 2;
    return tr_pair(p, p + 16 * 32);
  };
  auto b_frag = [&](int nt, int kk) {   // B^T: row nt * 16 + c, the same tokens
    const int n = nt * 16 + tr_col;
    const char* p = Bs + (((kk * 2 * KS + (n >> 5)) * 64 + ((n >> 3) & 3) * 16 + tr_row) * 16) + (n & 7) * 2;
    return tr_pair(p, p + KS * 1024);
  };
  // a chunk's rows, one chunk ahead: thread (wave, lane) holds piece (G * 8 ..) of B and C of token wave * 16 + c, and its pieces of x
  constexpr int LPR = VT * 2, XP = (64 * LPR + 255) / 256;   // 16-byte pieces of an x row, of x per thread
  u32x4_t br[KS], cr[STATE_ONLY ? 1 : KS], xr[XP];
  float dtr = 0.f;
  auto request = [&](int ch) __attribute__((always_inline)) {
    const int t0 = ch * 64, last = min(e.len - t0, 64) - 1;
    const bf16_t* row = u + (int64_t)(e.row0 + t0 + min(wave * 16 + c, last)) * cp + inner + grp * np + G * 8;
#pragma unroll
    for (int k4 = 0; k4 < KS; ++k4) br[k4] = ld16(row + k4 * 32);
    if constexpr (!STATE_ONLY) {
#pragma unroll
      for (int k4 = 0; k4 < KS; ++k4) cr[k4] = ld16(row + a.d.groups * np + k4 * 32);
    }
#pragma unroll
    for (int i = 0; i < XP; ++i) {
      const int q = min(tid + i * 256, 64 * LPR - 1), t = q / LPR;
      xr[i] = ld16(u + (int64_t)(e.row0 + t0 + min(t, last)) * cp + xc + (q % LPR) * 8);
    }
    dtr = a.dt[(int64_t)h * a.dt_ld + e.row0 + t0 + min(lane, last)];   // lane = token
  };
  request(ch0);
  float cum_seg = 0.f;
  for (int ch = ch0; ch < ch1; ++ch) {
    const int t0 = ch * 64, last = min(e.len - t0, 64) - 1;
    __syncthreads();   // everyone is past the last chunk's reads
    bf16x8_t cf[STATE_ONLY ? 1 : KS];   // C of token wave * 16 + c
#pragma unroll
    for (int k4 = 0; k4 < KS; ++k4) *reinterpret_cast<u32x4_t*>(Bs + (wave * KS + k4) * 1024 + lane * 16) = br[k4];
    if constexpr (!STATE_ONLY) {
#pragma unroll
      for (int k4 = 0; k4 < KS; ++k4) cf[k4] = as_frag(cr[k4]);
    }
#pragma unroll
    for (int i = 0; i < XP; ++i) {
      const int q = tid + i * 256, col = q % LPR;
      if (64 * LPR % 256 == 0 || q < 64 * LPR) *reinterpret_cast<u32x4_t*>(Xs + (col >> 1) * SSM_XV + q / LPR * 32 + (col & 1) * 16) = xr[i];
    }
    const float dt = lane <= last ? dtr : 0.f;
    if (ch + 1 < ch1) request(ch + 1);
    __builtin_amdgcn_sched_barrier(0);
    const float cum = wave_prefix_sum(A * dt), cum_last = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(cum), 63)), tot = __expf(cum_last);
    cum_seg += cum_last;
    if (wave == 0) {
      cums[lane] = cum;
      cums[64 + lane] = dt;
      cums[128 + lane] = __expf(cum_last - cum) * dt;
    }
    if constexpr (!STATE_ONLY) {
      // the state's halves for the other waves: four consecutive rows of one column = 8 bytes of a fragment's piece
#pragma unroll
      for (int j = 0; j < NTW; ++j) {
        const int nt = wave + j * 4;
        if (nt < NT) {
#pragma unroll
          for (int vt = 0; vt < VT; ++vt) {
            const f32x4_t s = S[j][vt];
            const uint2 hi = make_uint2(pack_bf(s[0], s[1]), pack_bf(s[2], s[3]));
            const uint2 lo = make_uint2(pack_bf(s[0] - lo_bf(hi.x), s[1] - hi_bf(hi.x)), pack_bf(s[2] - lo_bf(hi.y), s[3] - hi_bf(hi.y)));
            const int at = ((vt * KS + (nt >> 1)) * 64 + ((nt & 1) * 2 + (G >> 1)) * 16 + c) * 16 + (G & 1) * 8;
            *reinterpret_cast<uint2*>(Sh + at) = hi;
            *reinterpret_cast<uint2*>(Sl + at) = lo;
          }
        }
      }
    }
    __syncthreads();
    if constexpr (!STATE_ONLY) {
      // ---- outputs of tokens wave * 16 + c
      f32x4_t y[VT];
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        y[vt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k4 = 0; k4 < KS; ++k4) {
          const int at = ((vt * KS + k4) * 64 + lane) * 16;
          y[vt] = mfma16(as_frag(*reinterpret_cast<const u32x4_t*>(Sh + at)), cf[k4], y[vt]);
          y[vt] = mfma16(as_frag(*reinterpret_cast<const u32x4_t*>(Sl + at)), cf[k4], y[vt]);
        }
      }
      const float cum_t = cums[wave * 16 + c], ect = __expf(cum_t);
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) y[vt] *= ect;
      f32x4_t g[4];   // (B_s . C_t) of the token tiles up to the wave's own
#pragma unroll
      for (int sub = 0; sub < 4; ++sub) {
        g[sub] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (sub > wave) continue;
#pragma unroll
        for (int k4 = 0; k4 < KS; ++k4) g[sub] = mfma16(as_frag(*reinterpret_cast<const u32x4_t*>(Bs + ((sub * KS + k4) * 64 + lane) * 16)), cf[k4], g[sub]);
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        if (kk > wave >> 1) break;
        float p[8];
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          const int sub = kk * 2 + half;
          const float4 cs = *reinterpret_cast<const float4*>(cums + sub * 16 + G * 4), ds = *reinterpret_cast<const float4*>(cums + 64 + sub * 16 + G * 4);
          const float cv[4] = {cs.x, cs.y, cs.z, cs.w}, dv[4] = {ds.x, ds.y, ds.z, ds.w};
#pragma unroll
          for (int r = 0; r < 4; ++r) p[half * 4 + r] = sub * 16 + G * 4 + r <= wave * 16 + c ? g[sub][r] * __expf(cum_t - cv[r]) * dv[r] : 0.f;
        }
        bf16x8_t hi, lo;
        split8(p, hi, lo);
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
          const bf16x8_t xf = as_frag(x_frag(vt, kk));
          y[vt] = mfma16(xf, hi, y[vt]);
          y[vt] = mfma16(xf, lo, y[vt]);
        }
      }
      const int t = wave * 16 + c;
      if (t <= last) {
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
          const uint2 xv = *reinterpret_cast<const uint2*>(Xs + vt * SSM_XV + t * 32 + G * 8);
          *reinterpret_cast<uint2*>((bf16_t*)a.y + (int64_t)(e.row0 + t0 + t) * a.ldy + xc + vt * 16 + G * 4) =
              make_uint2(pack_bf(fmaf(D, lo_bf(xv.x), y[vt][0]), fmaf(D, hi_bf(xv.x), y[vt][1])), pack_bf(fmaf(D, lo_bf(xv.y), y[vt][2]), fmaf(D, hi_bf(xv.y), y[vt][3])));
        }
      }
    }
    // ---- the state behind the chunk
    if (!STATE_ONLY && ch + 1 == ch1 && ch1 < nchunk) break;   // (the next segment has its own)
#pragma unroll
    for (int j = 0; j < NTW; ++j)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) S[j][vt] *= tot;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const float4 w0 = *reinterpret_cast<const float4*>(cums + 128 + kk * 32 + G * 4), w1 = *reinterpret_cast<const float4*>(cums + 128 + kk * 32 + 16 + G * 4);
      const float w[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
      bf16x8_t xf[VT];
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) xf[vt] = as_frag(x_frag(vt, kk));
#pragma unroll
      for (int j = 0; j < NTW; ++j) {
        const int nt = wave + j * 4;
        if (nt >= NT) break;
        const u32x4_t bv = b_frag(nt, kk);
        float f[8];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f[2 * q] = lo_bf(bv[q]) * w[2 * q];
          f[2 * q + 1] = hi_bf(bv[q]) * w[2 * q + 1];
        }
        bf16x8_t bh, bl;
        split8(f, bh, bl);
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
          S[j][vt] = mfma16(bh, xf[vt], S[j][vt]);
          S[j][vt] = mfma16(bl, xf[vt], S[j][vt]);
        }
      }
    }
  }
  if (!STATE_ONLY && ch1 < nchunk) return;
  float* const behind = STATE_ONLY ? seg_state : a.s.state + (int64_t)e.state_out * a.s.pool_stride + so;
  if (STATE_ONLY && vs == 0 && tid == 0) sg.cum[(int64_t)blockIdx.y * a.d.heads + h] = cum_seg;
#pragma unroll
  for (int j = 0; j < NTW; ++j)
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) {
      const int nt = wave + j * 4;
      if (nt >= NT) break;
      float* p = behind + ((int64_t)vt * np + nt * 16 + G * 4) * 16 + c;
#pragma unroll
      for (int r = 0; r < 4; ++r) p[r * 16] = S[j][vt][r];
    }
}

// what each segment adds -> the state in front of each segment (thread: four floats of the state; four segments requested at a time)
__global__ __launch_bounds__(256) void ssm_segments_kernel(SsmScanArgs a, SeqBatch b, SsmSegments sg) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4, n = a.d.state_floats();
  if (i >= n) return;
  const SeqEntry e = seq_entry_at(b, blockIdx.y);
  const int h = (int)(i / ((int64_t)a.d.np * a.d.vdp)), own = (((e.len + 63) >> 6) + sg.chunks - 1) / sg.chunks;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  if (e.pos0 > 0) s = *reinterpret_cast<const float4*>(a.s.state + (int64_t)e.state_in * a.s.pool_stride + i);
  float* p = sg.state + (int64_t)blockIdx.y * sg.n * n + i;
  const float* cum = sg.cum + (int64_t)blockIdx.y * sg.n * a.d.heads + h;
  for (int k = 0; k < own; k += 4) {
    float4 add[4];
    float t[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {   // (the last segment adds to nobody's first state)
      const int g = min(k + j, max(own - 2, 0));
      add[j] = *reinterpret_cast<const float4*>(p + g * n);
      t[j] = cum[(int64_t)g * a.d.heads];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (k + j >= own) break;
      *reinterpret_cast<float4*>(p + (k + j) * n) = s;
      const float f = expf(t[j]);
      s = make_float4(fmaf(f, s.x, add[j].x), fmaf(f, s.y, add[j].y), fmaf(f, s.z, add[j].z), fmaf(f, s.w, add[j].w));
    }
  }
}

// ---- one token per sequence ------------------------------------------------------------------------------------------------------------------
// Block (VT * 16 columns, head of the group, group and sequence): thread (n, four columns of 16), n = tid / 4, + 64, ...  The state is requested first; the
// convolution of the block's channels (its x columns, the group's B and C) runs under that.
// NT: the state past the caches (launch_ssm_step).  ONE: one sequence and 2 to 5 taps, its places in the leading arguments (SsmStepLead), which are in registers
// before the first instruction.
// Below 16 MB of states the launch is one chain of waits, not bytes: nothing that the end needs is requested behind a barrier (the gate), wave 2 computes the
// step size that all used to, no divisions, the sums over n without the LDS crossbar.  0.6B widths, one sequence: 5.0 -> 3.6 us.
__device__ __forceinline__ float sum_stride4(float v) {   // over the sixteen lanes of one lane & 3
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x124 /* row_ror:4 */, 0xf, 0xf, false));
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x128 /* row_ror:8 */, 0xf, 0xf, false));
  return rows_sum(v);
}
enum { STEP_ANY, STEP_FEW, STEP_ONE };
constexpr int SSM_CHUNK_NP = 256;   // state dims (padded) of launch_ssm_chunks and launch_ssm_step, at most (ssm_chunk_ok)
// sizes in two words; a model's heads times their padded columns fit the LDS (layered_prenorm.hip), so heads, groups and columns fit sixteen bits
struct SsmStepLead {
  static_assert(SSM_CHUNK_NP < 1024, "np has ten bits");
  int np_taps_hpg, vdp_groups;
  __host__ __device__ int np() const { return np_taps_hpg & 1023; }
  __host__ __device__ int taps() const { return np_taps_hpg >> 10 & 63; }   // (63: that many or more)
  __host__ __device__ int hpg() const { return (int)((unsigned)np_taps_hpg >> 16); }
  __host__ __device__ int vdp() const { return vdp_groups & 65535; }
  __host__ __device__ int groups() const { return (int)((unsigned)vdp_groups >> 16); }
};
template <typename TI, int NI, int VT, bool NT, int FORM>
__global__ __launch_bounds__(256) void ssm_step_kernel(const float* sin, const TI* in_c, const float* hin, const float* conv_w, const float* conv_b, int inner, int np_taps_hpg,
                                                       int vdp_groups, int pos0, SsmStepArgs a, SeqBatch b) {
  constexpr bool ONE = FORM == STEP_ONE;
  __shared__ __attribute__((aligned(16))) float bc[2 * NI * 64], xs[VT * 16], red[4][VT * 16], step[2];
  const SsmStepLead lead{np_taps_hpg, vdp_groups};
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), vdp = lead.vdp(), nvs = vdp >> 4, vs = blockIdx.x * VT, np = lead.np(), taps = lead.taps(), groups = lead.groups();
  const int seq = ONE ? 0 : (int)blockIdx.z / groups, grp = ONE ? (int)blockIdx.z : (int)blockIdx.z - seq * groups, h = grp * lead.hpg() + blockIdx.y, cp = inner + 2 * groups * np;
  SeqEntry e = b.one;
  if constexpr (!ONE) {
    e = seq_entry_at(b, seq);
    sin += (int64_t)e.state_in * a.s.pool_stride;
    in_c += (int64_t)e.row0 * a.in.ld;
    hin += (int64_t)e.slot * a.h.slot_stride + (int64_t)e.hist_in * (a.d.taps - 1) * cp;
    pos0 = e.pos0;
  }
  const int64_t so = ((int64_t)h * nvs + vs) * np * 16;
  sin += so;
  const int n0 = tid >> 2, v4 = (tid & 3) * 4;
  float4 S[VT][NI];
#pragma unroll
  for (int vt = 0; vt < VT; ++vt)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      S[vt][i] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (pos0 > 0 && n0 + i * 64 < np) {
        const float* at = sin + (vt * np + n0 + i * 64) * 16 + v4;
        if constexpr (NT) {
          const f32x4_t x = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(at));
          S[vt][i] = make_float4(x[0], x[1], x[2], x[3]);
        } else {
          S[vt][i] = *reinterpret_cast<const float4*>(at);
        }
      }
    }
  // what wave 2 (the step size) and wave 3 (the gate of the columns it ends with) need, requested behind the convolution's inputs: it is found through the
  // arguments in memory
  const int fin = tid - 192, col = h * vdp + vs * 16 + min(fin, VT * 16 - 1);
  float ex, per_head, dt_bias;
  float* hout;
  auto others = [&] {
    ex = Act<TI>::ld(in_c - a.in.c_off + (fin >= 0 ? col : a.in.dt_off + h));
    per_head = (wave == 3 ? a.p.d : a.p.a)[h];
    dt_bias = a.p.dt_bias[h];
    hout = a.h.hist + (int64_t)e.slot * a.h.slot_stride + (int64_t)e.hist_out * (a.d.taps - 1) * cp;
  };
  // The block's channels: x, B and C, NIT per thread.  Inputs, weights and history of up to HT + 1 taps are requested together and the new history is
  // stored at the end (a wait for the state, in flight since before them, would wait for these stores too): a store between two loads orders them, and tap by tap, channel by channel the chain was most of the launch (0.6B widths,
  // one sequence: 7.5 -> 5.3 us; 8B widths, 32 sequences, bound by the 268 MB of their states: 60.7 -> 59.7 us, 50.8 past the caches).
  constexpr int NIT = (2 * NI * 64 + VT * 16 + 255) / 256, HT = 4;
  const int total = 2 * np + VT * 16;
  auto channel = [&](int i) { return i >= 2 * np ? h * vdp + vs * 16 + i - 2 * np : inner + (i < np ? grp * np + i : groups * np + grp * np + i - np); };
  auto put = [&](int i, float acc) {
    acc = silu_f32(acc);
    if (i >= 2 * np) xs[i - 2 * np] = acc;
    else bc[i < np ? i : NI * 64 + i - np] = acc;
  };
  constexpr bool few_taps = FORM != STEP_ANY;
  float cur[NIT], x[NIT][HT];
  if constexpr (few_taps) {
    float wl[NIT], bias[NIT], w[NIT][HT];
#pragma unroll
    for (int k = 0; k < NIT; ++k) {
      if (wave * 64 + k * 256 >= total) continue;
      const int ch = channel(min(tid + k * 256, total - 1));
      cur[k] = Act<TI>::ld(in_c + ch);
      wl[k] = conv_w[(int64_t)(taps - 1) * cp + ch];
      bias[k] = conv_b[ch];
#pragma unroll
      for (int q = 0; q < HT; ++q) {   // (taps that are not there: the oldest one again)
        const int qq = min(q, taps - 2);
        x[k][q] = hin[(int64_t)qq * cp + ch];
        w[k][q] = conv_w[(int64_t)(taps - 2 - qq) * cp + ch];
      }
    }
    asm volatile("" ::: "memory");
    others();
#pragma unroll
    for (int k = 0; k < NIT; ++k) {
      const int i = tid + k * 256;
      if (i >= total) continue;
      float acc = fmaf(wl[k], cur[k], bias[k]);
#pragma unroll
      for (int q = 0; q < HT; ++q) {
        if (q >= taps - 1) continue;
        if (pos0 - 1 - q < 0) x[k][q] = 0.f;
        acc = fmaf(w[k][q], x[k][q], acc);
      }
      put(i, acc);
    }
  } else {
    const int taps = a.d.taps;
    others();
    for (int i = tid; i < total; i += 256) {
      const int ch = channel(i);
      const float cur = Act<TI>::ld(in_c + ch);
      float acc = fmaf(conv_w[(int64_t)(taps - 1) * cp + ch], cur, conv_b[ch]);
      const bool owner = i >= 2 * np || (blockIdx.y == 0 && vs == 0);
      float prev = cur;
      for (int q = 0; q < taps - 1; ++q) {   // the input q + 1 tokens back
        const float x = pos0 - 1 - q >= 0 ? hin[(int64_t)q * cp + ch] : 0.f;
        acc = fmaf(conv_w[(int64_t)(taps - 2 - q) * cp + ch], x, acc);
        if (owner) hout[(int64_t)q * cp + ch] = prev;
        prev = x;
      }
      put(i, acc);
    }
  }
  if (wave == 2) {
    const float t = softplus_f32(ex + dt_bias);
    step[0] = t;
    step[1] = expf(per_head * t);
  } else if (wave == 3) {
    ex = silu_f32(ex);
  }
  asm volatile("" : "+v"(ex));   // (here, not behind the barriers)
  __syncthreads();
  const float dt = step[0], da = step[1];
  float* sout = a.s.state + (int64_t)e.state_out * a.s.pool_stride + so;
#pragma unroll
  for (int vt = 0; vt < VT; ++vt) {
    const float4 x = *reinterpret_cast<const float4*>(xs + vt * 16 + v4);
    float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int n = n0 + i * 64;
      if (n < np) {
        const float db = dt * bc[n], cn = bc[NI * 64 + n];
        float4& s = S[vt][i];
        s = make_float4(fmaf(db, x.x, da * s.x), fmaf(db, x.y, da * s.y), fmaf(db, x.z, da * s.z), fmaf(db, x.w, da * s.w));
        float* at = sout + (vt * np + n) * 16 + v4;
        if constexpr (NT) __builtin_nontemporal_store(f32x4_t{s.x, s.y, s.z, s.w}, reinterpret_cast<f32x4_t*>(at));
        else *reinterpret_cast<float4*>(at) = s;
        y = make_float4(fmaf(cn, s.x, y.x), fmaf(cn, s.y, y.y), fmaf(cn, s.z, y.z), fmaf(cn, s.w, y.w));
      }
    }
    y = make_float4(sum_stride4(y.x), sum_stride4(y.y), sum_stride4(y.z), sum_stride4(y.w));
    if (lane < 4) *reinterpret_cast<float4*>(&red[wave][vt * 16 + v4]) = y;
  }
  __syncthreads();
  if (fin >= 0 && fin < VT * 16) {
    const float yy = fmaf(per_head, xs[fin], (red[0][fin] + red[1][fin]) + (red[2][fin] + red[3][fin]));
    const float g = yy * ex;
    a.g[(int64_t)seq * inner + col] = g;
    float s = g * g;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) s += __shfl_xor(s, o, 16);
    if ((fin & 15) == 0) a.ssq[(int64_t)seq * (inner >> 4) + h * nvs + vs + (fin >> 4)] = s;
  }
  if constexpr (few_taps) {
#pragma unroll
    for (int k = 0; k < NIT; ++k) {
      const int i = tid + k * 256;
      if (i < total && (i >= 2 * np || (blockIdx.y == 0 && vs == 0))) {
        const int ch = channel(i);
#pragma unroll
        for (int q = 0; q < HT; ++q)
          if (q < taps - 1) hout[(int64_t)q * cp + ch] = q == 0 ? cur[k] : x[k][q > 0 ? q - 1 : 0];
      }
    }
  }
}

// ---- gate and norm -----------------------------------------------------------------------------------------------------------------------
// The gated row in LDS; wave w sums the parts w, w + waves, ... (a part is a run of real columns: heads one after the other without their pads)
template <typename T, bool GATED>
__global__ __launch_bounds__(512) void gated_norm_kernel(GatedNormArgs a) {
  extern __shared__ __attribute__((aligned(16))) float row[];   // (inner), then 1 / rms per part
  const int tid = threadIdx.x, inner = a.d.inner(), r = blockIdx.x, parts = a.d.norm_groups, vdim = a.d.vdim, vdp = a.d.vdp;
  float* rinv = row + inner;
  if constexpr (GATED) {
    const float* y = (const float*)a.y + (int64_t)r * a.ldy;
    for (int c = tid * 4; c < inner; c += 2048) *reinterpret_cast<float4*>(row + c) = *reinterpret_cast<const float4*>(y + c);
  } else {
    const T *y = (const T*)a.y + (int64_t)r * a.ldy, *z = (const T*)a.z + (int64_t)r * a.ldz;
    for (int c = tid * 4; c < inner; c += 2048) {
      const float4 yv = Act<T>::ld4(y + c), zv = Act<T>::ld4(z + c);
      *reinterpret_cast<float4*>(row + c) = make_float4(yv.x * silu_f32(zv.x), yv.y * silu_f32(zv.y), yv.z * silu_f32(zv.z), yv.w * silu_f32(zv.w));
    }
  }
  __syncthreads();
  const int gs = a.d.heads * vdim / parts;
  for (int g = tid >> 6; g < parts; g += 8) {
    float s = 0.f;
    for (int k = tid & 63; k < gs; k += 64) {
      const int i = g * gs + k;
      const float v = row[vdim == vdp ? i : i / vdim * vdp + i % vdim];
      s = fmaf(v, v, s);
    }
    s = wave_sum(s);
    if ((tid & 63) == 0) rinv[g] = 1.0f / sqrtf(s / (float)gs + a.eps);
  }
  __syncthreads();
  T* o = (T*)a.out + (int64_t)r * a.ldo;
  for (int c = tid * 4; c < inner; c += 2048) {
    const float4 v = *reinterpret_cast<const float4*>(row + c), w = wbf4(a.w, c);
    const int h = c / vdp, d = c - h * vdp;
    float f[4] = {v.x, v.y, v.z, v.w};
    const float wv[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) f[j] = d + j < vdim ? f[j] * rinv[(h * vdim + d + j) / gs] * wv[j] : 0.f;
    Act<T>::st4(o + c, make_float4(f[0], f[1], f[2], f[3]));
  }
}

// Parts of whole 8-column pieces, no pads between heads: a thread keeps its pieces in registers, their sums of squares meet in LDS
template <typename T, bool GATED, int NP>   // NP x 512 pieces
__global__ __launch_bounds__(512) void gated_norm_pieces_kernel(GatedNormArgs a) {
  extern __shared__ __attribute__((aligned(16))) float sums[];   // per piece, then 1 / rms per part
  const int tid = threadIdx.x, pieces = a.d.inner() >> 3, r = blockIdx.x, parts = a.d.norm_groups, per = pieces / parts;
  float* rinv = sums + pieces;
  float v[NP][8];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int c = (tid + i * 512) * 8;
    if (c < a.d.inner()) {
      if constexpr (GATED) {
        ld8<float>((const float*)a.y + (int64_t)r * a.ldy + c, v[i]);
      } else {
        float z[8];
        ld8<T>((const T*)a.y + (int64_t)r * a.ldy + c, v[i]);
        ld8<T>((const T*)a.z + (int64_t)r * a.ldz + c, z);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] *= silu_rows<T>(z[j]);
      }
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) s = fmaf(v[i][j], v[i][j], s);
      sums[tid + i * 512] = s;
    }
  }
  __syncthreads();
  for (int g = tid >> 6; g < parts; g += 8) {
    float s = 0.f;
    for (int k = tid & 63; k < per; k += 64) s += sums[g * per + k];
    s = wave_sum(s);
    if ((tid & 63) == 0) rinv[g] = 1.0f / sqrtf(s / (float)(per * 8) + a.eps);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int p = tid + i * 512, c = p * 8;
    if (c >= a.d.inner()) continue;
    const float q = rinv[p / per];
    float w[8];
    ld8<bf16_t>((const bf16_t*)a.w + c, w);
    T* o = (T*)a.out + (int64_t)r * a.ldo + c;
    Act<T>::st4(o, make_float4(v[i][0] * q * w[0], v[i][1] * q * w[1], v[i][2] * q * w[2], v[i][3] * q * w[3]));
    Act<T>::st4(o + 4, make_float4(v[i][4] * q * w[4], v[i][5] * q * w[5], v[i][6] * q * w[6], v[i][7] * q * w[7]));
  }
}

}  // namespace

void launch_short_conv(const ShortConvArgs& a, const SeqBatch& b, bool f32, hipStream_t st) {
  if (b.rows <= 0) return;
  const int tile = b.rows >= 2048 ? 16 : b.rows >= 256 ? 8 : 2;
  const int64_t conv_items = (int64_t)((b.rows + tile - 1) / tile) * (a.d.cp() >> 3), items = conv_items + (int64_t)b.rows * a.d.heads;
  const dim3 grid((unsigned)((items + 255) / 256)), block(256);
  auto go = [&](auto t, auto taps) {
    using T = decltype(t);
    hipLaunchKernelGGL((short_conv_kernel<T, decltype(taps)::value>), grid, block, 0, st, a, b, tile, conv_items);
  };
  auto by_taps = [&](auto t) {
    switch (a.d.taps) {
      case 1: go(t, std::integral_constant<int, 1>{}); break;
      case 2: go(t, std::integral_constant<int, 2>{}); break;
      case 3: go(t, std::integral_constant<int, 3>{}); break;
      case 4: go(t, std::integral_constant<int, 4>{}); break;
      default: go(t, std::integral_constant<int, 0>{}); break;
    }
  };
  if (f32) by_taps(float{});
  else by_taps(bf16_t{});
}

void launch_ssm_scan(const SsmScanArgs& a, const SeqBatch& b, bool f32, hipStream_t st) {
  if (b.rows <= 0) return;
  const dim3 grid((unsigned)(a.d.heads * (a.d.vdp >> 4)), (unsigned)b.n), block(256);
  const size_t lds = (size_t)a.d.np * 64;
  auto go = [&](auto k) {
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(k, grid, block, lds, st, a, b);
  };
  if (f32) go(ssm_scan_kernel<float>);
  else go(ssm_scan_kernel<bf16_t>);
}

bool ssm_chunk_ok(const SsmDims& d) { return d.np <= SSM_CHUNK_NP; }

// Columns (16 VT of them) per block and segments per entry of a launch: enough blocks for the chip where the prompt has the chunks, at least two chunks
// per segment
constexpr int SSM_BLOCKS = 1024;
static void ssm_chunk_plan(const SsmDims& d, int n, int max_len, int* vt, int* nseg, int* chunks) {
  const int nvs = d.vdp >> 4, nchunk = (max_len + 63) / 64, most = std::max(1, nchunk / 2);
  *vt = nvs % 4 == 0 && d.np <= 160 ? 4 : nvs % 2 == 0 ? 2 : 1;
  while (*vt > 1 && (int64_t)d.heads * nvs / *vt * n * most < 256) *vt /= 2;
  const int64_t base = (int64_t)d.heads * nvs / *vt * n;
  const int want = (int)std::max<int64_t>(1, std::min<int64_t>(most, SSM_BLOCKS / base));
  *chunks = std::max(1, (nchunk + want - 1) / want);
  *nseg = std::max(1, (nchunk + *chunks - 1) / *chunks);
}
size_t ssm_segment_floats(const SsmDims& d) {   // segments x entries <= SSM_BLOCKS / blocks of one segment, if there are segments
  size_t most = 0;
  const int nvs = d.vdp >> 4;
  for (int vt = 1; vt <= 4; vt *= 2)
    if (nvs % vt == 0) most = std::max(most, (size_t)std::max(1, SSM_BLOCKS / (d.heads * nvs / vt)) * (size_t)(d.state_floats() + d.heads));
  return most;
}

void launch_ssm_chunks(const SsmScanArgs& a, const SeqBatch& b, float* scratch, size_t scratch_floats, hipStream_t st) {
  if (b.rows <= 0) return;
  const int nvs = a.d.vdp >> 4;
  int vt, nseg, chunks;
  ssm_chunk_plan(a.d, b.n, b.max_len, &vt, &nseg, &chunks);
  if ((size_t)b.n * nseg * (size_t)(a.d.state_floats() + a.d.heads) > scratch_floats) {
    nseg = 1;
    chunks = 1 << 24;
  }
  const SsmSegments sg{scratch, scratch + (size_t)b.n * nseg * a.d.state_floats(), nseg, chunks};
  auto go = [&](auto ks, auto v, auto only) {
    constexpr int KS = decltype(ks)::value, VT = decltype(v)::value;
    constexpr bool ONLY = decltype(only)::value;
    constexpr int lds = ssm_chunk_lds<KS, VT>(ONLY);
    auto k = ssm_chunk_kernel<KS, VT, ONLY>;
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    hipLaunchKernelGGL(k, dim3((unsigned)(a.d.heads * nvs / VT), (unsigned)(b.n * nseg)), dim3(256), lds, st, a, b, sg);
  };
  auto by_vt = [&](auto ks) {
    auto both = [&](auto v) {
      if (nseg > 1) {
        go(ks, v, std::true_type{});
        hipLaunchKernelGGL(ssm_segments_kernel, dim3((unsigned)((a.d.state_floats() / 4 + 255) / 256), (unsigned)b.n), dim3(256), 0, st, a, b, sg);
      }
      go(ks, v, std::false_type{});
    };
    if (vt == 4) {
      if constexpr (decltype(ks)::value <= 5) both(std::integral_constant<int, 4>{});
    } else if (vt == 2) {
      both(std::integral_constant<int, 2>{});
    } else {
      both(std::integral_constant<int, 1>{});
    }
  };
  switch (a.d.np >> 5) {
    case 1: by_vt(std::integral_constant<int, 1>{}); break;
    case 2: by_vt(std::integral_constant<int, 2>{}); break;
    case 3: by_vt(std::integral_constant<int, 3>{}); break;
    case 4: by_vt(std::integral_constant<int, 4>{}); break;
    case 5: by_vt(std::integral_constant<int, 5>{}); break;
    case 6: by_vt(std::integral_constant<int, 6>{}); break;
    case 7: by_vt(std::integral_constant<int, 7>{}); break;
    default: by_vt(std::integral_constant<int, 8>{}); break;
  }
}

void launch_ssm_step(const SsmStepArgs& a, const SeqBatch& b, hipStream_t st) {
  if (b.n <= 0) return;
  if (const int most = 65535 / a.d.groups; b.n > most) {   // (the grid's z)
    SsmStepArgs rest = a;
    rest.g += (int64_t)most * a.d.inner();
    rest.ssq += (int64_t)most * (a.d.inner() >> 4);
    SeqBatch first = b, later = b;
    first.n = most;
    later.n -= most;
    later.entries += most;
    launch_ssm_step(a, first, st);
    return launch_ssm_step(rest, later, st);
  }
  const int nvs = a.d.vdp >> 4;
  const bool wide = nvs % 4 == 0 && (int64_t)a.d.heads * nvs / 4 * b.n >= 512;   // B and C of the group once per 64 columns
  // From 16 MB of states per launch on, past the caches: nothing reads them before the next step, and they push out what is read (128 dims of state, 16 MB:
  // 10.4 -> 9.0 us at 4 sequences of the 8B widths, 11.4 -> 10.0 at 16 of the 0.6B ones, in stacks of 2 to 28 layers; 268 MB: 59.7 -> 50.8).  Smaller ones
  // are still there in the next step (2 MB 6.6 against 7.2 us past the caches, 8 MB 7.4 against 8.1).
  const bool past = (int64_t)b.n * a.d.heads * a.d.vdp * a.d.np * 4 >= 16 << 20;
  const int hpg = a.d.heads / a.d.groups;
  const dim3 grid((unsigned)(nvs / (wide ? 4 : 1)), (unsigned)hpg, (unsigned)(a.d.groups * b.n)), block(256);
  const SsmStepLead lead{a.d.np | std::min(a.d.taps, 63) << 10 | hpg << 16, a.d.vdp | a.d.groups << 16};
  auto go = [&](auto ni) {
    constexpr int NI = decltype(ni)::value;
    auto launch = [&](auto ti, auto vt, auto nt, auto form) {
      using TI = decltype(ti);
      constexpr int VT = decltype(vt)::value;
      constexpr bool NT = decltype(nt)::value;
      constexpr int FORM = decltype(form)::value;
      const float *sin = a.s.state, *hin = a.h.hist;
      const TI* in_c = (const TI*)a.in.p + a.in.c_off;
      if (FORM == STEP_ONE) {
        sin += (int64_t)b.one.state_in * a.s.pool_stride;
        hin += (int64_t)b.one.slot * a.h.slot_stride + (int64_t)b.one.hist_in * (a.d.taps - 1) * a.d.cp();
        in_c += (int64_t)b.one.row0 * a.in.ld;
      }
      hipLaunchKernelGGL((ssm_step_kernel<TI, NI, VT, NT, FORM>), grid, block, 0, st, sin, in_c, hin, a.p.conv_w, a.p.conv_b, a.d.inner(), lead.np_taps_hpg, lead.vdp_groups, b.one.pos0, a, b);
    };
    auto run = [&](auto vt, auto nt) {
      auto typed = [&](auto ti) {
        if (a.d.taps < 2 || a.d.taps > 5) launch(ti, vt, nt, std::integral_constant<int, STEP_ANY>{});
        else if (b.has_one) launch(ti, vt, nt, std::integral_constant<int, STEP_ONE>{});
        else launch(ti, vt, nt, std::integral_constant<int, STEP_FEW>{});
      };
      if (a.in_f32) typed(float{});
      else typed(bf16_t{});
    };
    if (!wide) run(std::integral_constant<int, 1>{}, std::false_type{});
    else if (past) run(std::integral_constant<int, 4>{}, std::true_type{});
    else run(std::integral_constant<int, 4>{}, std::false_type{});
  };
  if (a.d.np <= 64) go(std::integral_constant<int, 1>{});
  else if (a.d.np <= 128) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 4>{});
}

void launch_gated_norm(const GatedNormArgs& a, bool f32, hipStream_t st) {
  if (a.rows <= 0) return;
  const int inner = a.d.inner(), gs = a.d.heads * a.d.vdim / a.d.norm_groups;
  auto by_type = [&](auto&& f) {
    if (a.z && f32) f(float{}, std::false_type{});
    else if (a.z) f(bf16_t{}, std::false_type{});
    else if (f32) f(float{}, std::true_type{});
    else f(bf16_t{}, std::true_type{});
  };
  if (a.d.vdim == a.d.vdp && gs % 8 == 0 && inner <= 4 * 4096) {
    const size_t lds = (size_t)(inner / 8 + a.d.norm_groups) * 4;
    by_type([&](auto t, auto gated) {
      using T = decltype(t);
      constexpr bool GATED = decltype(gated)::value;
      auto go = [&](auto np) { hipLaunchKernelGGL((gated_norm_pieces_kernel<T, GATED, decltype(np)::value>), dim3((unsigned)a.rows), dim3(512), lds, st, a); };
      if (inner <= 4096) go(std::integral_constant<int, 1>{});
      else if (inner <= 2 * 4096) go(std::integral_constant<int, 2>{});
      else go(std::integral_constant<int, 4>{});
    });
    return;
  }
  const size_t lds = (size_t)(inner + a.d.norm_groups) * 4;
  by_type([&](auto t, auto gated) {
    auto k = gated_norm_kernel<decltype(t), decltype(gated)::value>;
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(k, dim3((unsigned)a.rows), dim3(512), lds, st, a);
  });
}

}  // namespace aha
