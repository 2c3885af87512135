// Row kernels of the layer-list decoders (layered.hip), each templated on the activation type (bf16 served, float for the 32-bit mode; all
// arithmetic is f32 either way):
//   postnorm_conv_kernel   x = norm(alpha x + y) (or the scaled embedding row), h = x + causal convolution of x
//   final_rows_kernel      the last sublayer's norm and the model's norm on the wanted rows
//   rope_pairs_kernel      (cos, sin) of a step's angles, once for all layers of the same rotation
//   qkv_post_kernel        q / k norm over the whole projection, rotation, value mixing, KV append
//   polynorm_rows_kernel   a N(z) + b N(z^2) + c N(z^3) + e
#include <math.h>

#include <algorithm>

#include <type_traits>

#include "rows_common.h"

namespace aha {

namespace {

constexpr int NT = 256;

// sum over the block; `red` holds 4 floats per call and must not be reused before the next __syncthreads
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// One block walks `tile` consecutive rows in order.  Wave w owns columns (i * waves + w) * 256 .. + 256 of every row (i < NV; ld is a multiple of
// 256, so a column group is in or out of range for a whole wave: loads go out unconditionally at a clamped column, only stores branch).  The
// taps - 1 rows in front of the current one sit in an LDS ring (each thread reads only what it wrote: no barrier).  Rows in front of the tile are
// recomputed when they belong to the same step (x_in is not x_out), and come from the sequence's history otherwise.
template <typename T, int NTH, int NV, bool EMBED>
__global__ __launch_bounds__(NTH) void postnorm_conv_kernel(PostNormArgs a, SeqBatch b, int tile) {
  extern __shared__ __attribute__((aligned(16))) float ring[];   // (taps - 1) x NV * NTH * 4
  __shared__ float red[2][NTH / 64];
  constexpr int CP = NTH * 4, RP = NV * CP;   // columns per pass / per ring row
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), taps = a.conv.taps, nh = taps - 1, ld = (int)a.ld;
  const int r0 = (int)blockIdx.x * tile, r1 = min(r0 + tile, b.rows);
  int flip = 0, ctr = 0;   // ctr: ring slot of the next push; the row `back` tokens ago is slot (ctr - back) mod nh
  auto in = [&](int i) { return i * CP + wave * 256 < ld; };
  auto col = [&](int i) { return min(i * CP + tid * 4, ld - 4); };
  auto slot_of = [&](int c) { return c < 0 ? c + nh : c; };
  auto lds = [&](int slot, int i) { return reinterpret_cast<float4*>(ring + slot * RP + i * CP + tid * 4); };
  auto push = [&](const float4 (&v)[NV]) {
    if (nh == 0) return;
#pragma unroll
    for (int i = 0; i < NV; ++i) *lds(ctr, i) = v[i];
    ctr = ctr + 1 == nh ? 0 : ctr + 1;
  };
  auto load_row = [&](int r, float4 (&v)[NV]) {   // the row's value before its norm; zeros out of range
    if (EMBED) {
      const bf16_t* erow = (const bf16_t*)a.embed + (int64_t)a.ids[r] * ld;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const float4 e = wbf4(erow, col(i));
        const float f = in(i) ? a.embed_scale : 0.f;
        v[i] = make_float4(e.x * f, e.y * f, e.z * f, e.w * f);
      }
      return;
    }
    const float* xr = a.x_in + (int64_t)r * ld;
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = *reinterpret_cast<const float4*>(xr + col(i));
    if (a.y) {
      const T* yr = (const T*)a.y + (int64_t)r * a.ldy;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const float4 y = Act<T>::ld4(yr + col(i));
        v[i] = make_float4(fmaf(a.alpha, v[i].x, y.x), fmaf(a.alpha, v[i].y, y.y), fmaf(a.alpha, v[i].z, y.z), fmaf(a.alpha, v[i].w, y.w));
      }
    } else {
#pragma unroll
      for (int i = 0; i < NV; ++i) v[i] = make_float4(a.alpha * v[i].x, a.alpha * v[i].y, a.alpha * v[i].z, a.alpha * v[i].w);
    }
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (!in(i)) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  };
  auto norm_row = [&](float4 (&v)[NV]) {
    if (EMBED) return;
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) ss += (v[i].x * v[i].x + v[i].y * v[i].y) + (v[i].z * v[i].z + v[i].w * v[i].w);   // (pad columns are zero)
    ss = block_sum_n<NTH>(ss, red[flip]);
    flip ^= 1;
    const float rinv = 1.0f / sqrtf(ss / (float)a.width + a.eps);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const float4 n = wbf4(a.norm_w, col(i));
      v[i] = make_float4(v[i].x * rinv * (1.f + n.x), v[i].y * rinv * (1.f + n.y), v[i].z * rinv * (1.f + n.z), v[i].w * rinv * (1.f + n.w));
    }
  };
  auto hist_of = [&](const SeqEntry& e, int which) { return a.conv.hist + (int64_t)e.slot * a.conv.slot_stride + (int64_t)which * taps * ld; };
  auto push_hist = [&](const SeqEntry& e, int back) {   // the input `back` tokens in front of the entry's first
    float4 v[NV];
    if (e.pos0 - back >= 0) {
      const float* h = hist_of(e, e.hist_in) + (int64_t)(back - 1) * ld;
#pragma unroll
      for (int i = 0; i < NV; ++i) v[i] = *reinterpret_cast<const float4*>(h + col(i));
    } else {
#pragma unroll
      for (int i = 0; i < NV; ++i) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    push(v);
  };

  int ei = entry_of_row(b, r0);
  SeqEntry e = seq_entry_at(b, ei);
  if (nh > 0 && r0 > e.row0) {
    const int hb = min(nh, r0 - e.row0);
    for (int back = nh; back > hb; --back) push_hist(e, back - hb);
    for (int r = r0 - hb; r < r0; ++r) {
      float4 v[NV];
      load_row(r, v);
      norm_row(v);
      push(v);
    }
  }
  float4 v[NV], nxt[NV];
  load_row(r0, v);
  for (int r = r0; r < r1; ++r) {
    if (r > r0 && r == e.row0 + e.len) e = seq_entry_at(b, ++ei);
    if (r == e.row0)
      for (int back = nh; back > 0; --back) push_hist(e, back);
    load_row(min(r + 1, r1 - 1), nxt);
    norm_row(v);
    float* xo = a.x_out + (int64_t)r * ld;
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (in(i)) *reinterpret_cast<float4*>(xo + col(i)) = v[i];
    if (a.h_out) {
      auto tap = [&](float4& s, int j, int i, float4 x) {
        const float4 w = wbf4(a.conv.w, (int64_t)j * ld + col(i));
        s.x = fmaf(w.x, x.x, s.x); s.y = fmaf(w.y, x.y, s.y); s.z = fmaf(w.z, x.z, s.z); s.w = fmaf(w.w, x.w, s.w);
      };
      float4 acc[NV];
#pragma unroll
      for (int i = 0; i < NV; ++i) acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      for (int j = 0; j < nh; ++j) {
        const int slot = slot_of(ctr - (nh - j));
#pragma unroll
        for (int i = 0; i < NV; ++i) tap(acc[i], j, i, *lds(slot, i));
      }
      T* ho = (T*)a.h_out + (int64_t)r * ld;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        tap(acc[i], nh, i, v[i]);
        if (in(i)) Act<T>::st4(ho + col(i), make_float4(v[i].x + acc[i].x, v[i].y + acc[i].y, v[i].z + acc[i].z, v[i].w + acc[i].w));
      }
      if (r == e.row0 + e.len - 1) {   // history for the next step: row k = k + 1 tokens in front of the next token, then their weighted sum
        float* hs = hist_of(e, e.hist_out);
#pragma unroll
        for (int i = 0; i < NV; ++i) acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int k = nh - 1; k >= 1; --k) {
          const int slot = slot_of(ctr - k);
#pragma unroll
          for (int i = 0; i < NV; ++i) {
            const float4 x = *lds(slot, i);
            tap(acc[i], nh - 1 - k, i, x);
            if (in(i)) *reinterpret_cast<float4*>(hs + (int64_t)k * ld + col(i)) = x;
          }
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          if (nh > 0) tap(acc[i], nh - 1, i, v[i]);
          if (in(i)) {
            if (nh > 0) *reinterpret_cast<float4*>(hs + col(i)) = v[i];
            *reinterpret_cast<float4*>(hs + (int64_t)nh * ld + col(i)) = acc[i];
          }
        }
      }
    }
    push(v);
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = nxt[i];
  }
}

// The same where every sequence brings one row, ld <= 4 * NTH: a block per row, a thread its four columns.  Eight rows are eight blocks, so the launch is
// its chain of round trips -- entry, history, and in the general kernel one more per tap, per weight row and behind the norm (6.0 us at 8 rows of 4096
// columns, 3 taps); here everything that the entry does not decide is requested in front of it, the history right behind: 4.1 us.
template <typename T, int NTH, int TAPS, bool EMBED>
__global__ __launch_bounds__(NTH) void postnorm_conv_step_kernel(const float* x_in, const void* yp, const void* norm_w, const void* conv_w, const SeqEntry* entries, int ld_, int64_t ldy, PostNormArgs a,
                                                                  SeqBatch b) {
  constexpr int NH = TAPS - 1;
  // (what the first requests need: in scalar registers at the start, gemv_body.h)
  a.x_in = x_in;
  a.y = yp;
  a.norm_w = norm_w;
  a.conv.w = conv_w;
  a.ld = ld_;
  a.ldy = ldy;
  b.entries = entries;
  __shared__ float red[NTH / 64];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), ld = (int)a.ld, r = (int)blockIdx.x;
  const bool in = wave * 256 < ld;
  const int c = min(tid * 4, ld - 4);
  const SeqEntry e = seq_entry_at(b, r);   // (one row per sequence)
  float4 v, y = make_float4(0.f, 0.f, 0.f, 0.f), nw = y, w[TAPS], hist[NH];
  if (EMBED) {
    v = wbf4((const bf16_t*)a.embed + (int64_t)a.ids[r] * ld, c);
  } else {
    v = *reinterpret_cast<const float4*>(a.x_in + (int64_t)r * ld + c);
    if (a.y) y = Act<T>::ld4((const T*)a.y + (int64_t)r * a.ldy + c);
    nw = wbf4(a.norm_w, c);
  }
#pragma unroll
  for (int j = 0; j < TAPS; ++j) w[j] = wbf4(a.conv.w, (int64_t)j * ld + c);
  float* base = a.conv.hist + (int64_t)e.slot * a.conv.slot_stride + c;
  const float* hi = base + (int64_t)e.hist_in * TAPS * ld;
#pragma unroll
  for (int k = 0; k < NH; ++k) {   // hist[k]: the input k + 1 tokens ago
    hist[k] = *reinterpret_cast<const float4*>(hi + (int64_t)k * ld);
    if (e.pos0 < k + 1) hist[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  if (EMBED) {
    v = make_float4(v.x * a.embed_scale, v.y * a.embed_scale, v.z * a.embed_scale, v.w * a.embed_scale);
    if (!in) v = make_float4(0.f, 0.f, 0.f, 0.f);
  } else {
    v = a.y ? make_float4(fmaf(a.alpha, v.x, y.x), fmaf(a.alpha, v.y, y.y), fmaf(a.alpha, v.z, y.z), fmaf(a.alpha, v.w, y.w))
            : make_float4(a.alpha * v.x, a.alpha * v.y, a.alpha * v.z, a.alpha * v.w);
    if (!in) v = make_float4(0.f, 0.f, 0.f, 0.f);
    const float ss = block_sum_n<NTH>((v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w), red);
    const float rinv = 1.0f / sqrtf(ss / (float)a.width + a.eps);
    v = make_float4(v.x * rinv * (1.f + nw.x), v.y * rinv * (1.f + nw.y), v.z * rinv * (1.f + nw.z), v.w * rinv * (1.f + nw.w));
  }
  if (!in) return;
  auto tap = [](float4& s, float4 t, float4 x) { s.x = fmaf(t.x, x.x, s.x); s.y = fmaf(t.y, x.y, s.y); s.z = fmaf(t.z, x.z, s.z); s.w = fmaf(t.w, x.w, s.w); };
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f), next = acc;   // next: the weighted sum of what the next token finds behind it
#pragma unroll
  for (int j = 0; j < NH; ++j) tap(acc, w[j], hist[NH - 1 - j]);
  tap(acc, w[NH], v);
#pragma unroll
  for (int k = NH - 1; k >= 1; --k) tap(next, w[NH - 1 - k], hist[k - 1]);
  tap(next, w[NH - 1], v);
  *reinterpret_cast<float4*>(a.x_out + (int64_t)r * ld + c) = v;
  Act<T>::st4((T*)a.h_out + (int64_t)r * ld + c, make_float4(v.x + acc.x, v.y + acc.y, v.z + acc.z, v.w + acc.w));
  float* ho = base + (int64_t)e.hist_out * TAPS * ld;
  *reinterpret_cast<float4*>(ho) = v;
#pragma unroll
  for (int k = 1; k < NH; ++k) *reinterpret_cast<float4*>(ho + (int64_t)k * ld) = hist[k - 1];
  *reinterpret_cast<float4*>(ho + (int64_t)NH * ld) = next;
}

// The same for up to four taps, prompt-sized steps: the tile's rows and the TAPS - 1 in front of them in registers at once -- one round of loads,
// one barrier for all the sums -- instead of row by row.  NV = 1: 4 * NTH columns.
template <typename T, int NTH, int TAPS, int TILE>
__global__ __launch_bounds__(NTH) void postnorm_conv_tile_kernel(PostNormArgs a, SeqBatch b) {
  constexpr int NH = TAPS - 1, NR = TILE + NH, NW = NTH / 64;
  __shared__ float red[NR][NW], rms[NR];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ld = (int)a.ld;
  // neighbouring tiles on one XCD: its L2 holds the rows a tile shares with the one before it
  const int nt = (int)gridDim.x, per = (nt + 7) >> 3;
  const int tile = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  const int r0 = tile * TILE;
  if (r0 >= b.rows) return;
  const bool in = wave * 256 < ld;
  const int c = min(tid * 4, ld - 4);
  float4 v[NR];
  const float* xb = a.x_in;
  const T* yb = (const T*)a.y;
  {
    float4 y[NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int64_t r = min(max(r0 - NH + k, 0), b.rows - 1);
      v[k] = *reinterpret_cast<const float4*>(xb + r * ld + c);
      y[k] = Act<T>::ld4(yb + r * a.ldy + c);
    }
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      v[k] = make_float4(fmaf(a.alpha, v[k].x, y[k].x), fmaf(a.alpha, v[k].y, y[k].y), fmaf(a.alpha, v[k].z, y[k].z), fmaf(a.alpha, v[k].w, y[k].w));
      if (!in) v[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  const float4 n = wbf4(a.norm_w, c);
  float4 w[TAPS];
#pragma unroll
  for (int j = 0; j < TAPS; ++j) w[j] = wbf4(a.conv.w, (int64_t)j * ld + c);
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    const float ss = wave_sum((v[k].x * v[k].x + v[k].y * v[k].y) + (v[k].z * v[k].z + v[k].w * v[k].w));
    if (lane == 0) red[k][wave] = ss;
  }
  __syncthreads();
  for (int k = wave; k < NR; k += NW) {   // one wave per row finishes its sum
    const float ss = wave_sum(lane < NW ? red[k][min(lane, NW - 1)] : 0.f);
    if (lane == 0) rms[k] = 1.0f / sqrtf(ss / (float)a.width + a.eps);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    const float rinv = rms[k];
    v[k] = make_float4(v[k].x * rinv * (1.f + n.x), v[k].y * rinv * (1.f + n.y), v[k].z * rinv * (1.f + n.z), v[k].w * rinv * (1.f + n.w));
  }
  int ei = entry_of_row(b, r0);
  SeqEntry e = seq_entry_at(b, ei);
  auto hist_of = [&](int which) { return a.conv.hist + (int64_t)e.slot * a.conv.slot_stride + (int64_t)which * TAPS * ld; };
#pragma unroll
  for (int k = NH; k < NR; ++k) {
    const int r = r0 - NH + k;
    if (r >= b.rows) break;
    if (r == e.row0 + e.len) e = seq_entry_at(b, ++ei);
    const int rel = r - e.row0;
    // inputs 1 .. NH tokens back: rows of this step, of the sequence's history, or nothing
    float4 back[NH];
#pragma unroll
    for (int q = 1; q <= NH; ++q) {
      back[q - 1] = v[k - q];
      if (rel < q) {   // (uniform; the first rows of an entry)
        back[q - 1] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (e.pos0 + rel - q >= 0) back[q - 1] = *reinterpret_cast<const float4*>(hist_of(e.hist_in) + (int64_t)(q - rel - 1) * ld + c);
      }
    }
    float4 acc = make_float4(w[NH].x * v[k].x, w[NH].y * v[k].y, w[NH].z * v[k].z, w[NH].w * v[k].w);
#pragma unroll
    for (int q = 1; q <= NH; ++q) {
      const float4 ww = w[NH - q], x = back[q - 1];
      acc.x = fmaf(ww.x, x.x, acc.x); acc.y = fmaf(ww.y, x.y, acc.y); acc.z = fmaf(ww.z, x.z, acc.z); acc.w = fmaf(ww.w, x.w, acc.w);
    }
    if (in) {
      *reinterpret_cast<float4*>(a.x_out + (int64_t)r * ld + c) = v[k];
      Act<T>::st4((T*)a.h_out + (int64_t)r * ld + c, make_float4(v[k].x + acc.x, v[k].y + acc.y, v[k].z + acc.z, v[k].w + acc.w));
      if (rel == e.len - 1) {   // history for the next step, and its weighted sum
        float* hs = hist_of(e.hist_out);
        float4 nx = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int q = NH - 1; q >= 0; --q) {   // row q = q + 1 tokens in front of the next one
          const float4 x = q == 0 ? v[k] : back[q > 0 ? q - 1 : 0], ww = w[NH - 1 - q];
          *reinterpret_cast<float4*>(hs + (int64_t)q * ld + c) = x;
          nx.x = fmaf(ww.x, x.x, nx.x); nx.y = fmaf(ww.y, x.y, nx.y); nx.z = fmaf(ww.z, x.z, nx.z); nx.w = fmaf(ww.w, x.w, nx.w);
        }
        *reinterpret_cast<float4*>(hs + (int64_t)NH * ld + c) = nx;
      }
    }
  }
}

// A block per row, NV columns a thread, everything asked for at once (8 rows of 4096: 15.9 us with a load at a time, 4.8 so).  A row longer than that goes
// round again from LDS.
// NORM: norm_w and y are there
template <typename T, int NV, bool NORM>
__global__ __launch_bounds__(NT) void final_rows_kernel(FinalRowsArgs a) {
  __shared__ float red[2][4];
  extern __shared__ __attribute__((aligned(16))) float row[];   // (ld): what a row has behind NV * NT columns
  const int r = a.rows ? a.rows[blockIdx.x] : (int)blockIdx.x, tid = (int)threadIdx.x;
  auto value = [&](int c) {
    const float v = a.x[(int64_t)r * a.ld + c];
    if constexpr (NORM) return fmaf(a.alpha, v, Act<T>::ld((const T*)a.y + (int64_t)r * a.ldy + c));
    return a.norm_w ? fmaf(a.alpha, v, a.y ? Act<T>::ld((const T*)a.y + (int64_t)r * a.ldy + c) : 0.f) : v;
  };
  float v[NV], nw[NV], fw[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = min(tid + k * NT, a.width - 1);
    v[k] = value(c);
    nw[k] = NORM || a.norm_w ? bf2f(((const bf16_t*)a.norm_w)[c]) : 0.f;
    fw[k] = bf2f(((const bf16_t*)a.final_w)[c]);
  }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    if (tid + k * NT >= a.width) v[k] = 0.f;
    ss += v[k] * v[k];
  }
  for (int c = tid + NV * NT; c < a.width; c += NT) {
    const float x = value(c);
    row[c] = x;
    ss += x * x;
  }
  if (NORM || a.norm_w) {
    ss = block_sum(ss, red[0]);
    const float rinv = 1.0f / sqrtf(ss / (float)a.width + a.eps);
    ss = 0.f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      v[k] = v[k] * rinv * (1.f + nw[k]);
      ss += v[k] * v[k];
    }
    for (int c = tid + NV * NT; c < a.width; c += NT) {
      const float x = row[c] * rinv * (1.f + bf2f(((const bf16_t*)a.norm_w)[c]));
      row[c] = x;
      ss += x * x;
    }
  }
  ss = block_sum(ss, red[1]);
  const float rinv = 1.0f / sqrtf(ss / (float)a.width + a.eps);
  T* out = (T*)a.out + (int64_t)blockIdx.x * a.ld;
#pragma unroll
  for (int k = 0; k < NV; ++k)
    if (tid + k * NT < a.ld) Act<T>::st(out + tid + k * NT, tid + k * NT < a.width ? v[k] * rinv * (1.f + fw[k]) : 0.f);
  for (int c = tid + NV * NT; c < a.ld; c += NT) Act<T>::st(out + c, c < a.width ? row[c] * rinv * (1.f + bf2f(((const bf16_t*)a.final_w)[c])) : 0.f);
}

__global__ __launch_bounds__(NT) void rope_pairs_kernel(SeqBatch b, double base, int half, float* __restrict__ tab) {
  const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (i >= (int64_t)b.rows * half) return;
  const int r = (int)(i / half), k = (int)(i - (int64_t)r * half);
  const SeqEntry e = seq_entry_at(b, entry_of_row(b, r));
  const double ang = (double)(e.pos0 + r - e.row0) * pow(base, -(double)k / (double)half);   // f64 once per step and pair: no error at far positions
  double s, c;
  sincos(ang, &s, &c);
  reinterpret_cast<float2*>(tab)[i] = make_float2((float)c, (float)s);
}

template <typename T, bool FRAG>
__global__ __launch_bounds__(NT) void qkv_post_kernel(QkvPostArgs a, SeqBatch b) {
  extern __shared__ __attribute__((aligned(16))) float sm[];   // q | k | v of the row, f32
  __shared__ float red[2][4];
  const int r = blockIdx.x, tid = threadIdx.x;
  const SeqEntry e = seq_entry_at(b, entry_of_row(b, r));
  const int pos = e.pos0 + r - e.row0;
  const int nq = a.heads * a.dim, nk = a.kvh * a.dim, nv = a.kvh * a.vdim;
  const T* src = (const T*)a.qkv + (int64_t)r * a.ld;
  const int ko = nq, vo = nq + nk;   // (indices into sm, not pointers: a selected LDS pointer would decay to a flat one)
  float sq = 0.f, sk = 0.f;
  for (int i = tid; i < nq; i += NT) { const float v = Act<T>::ld(src + i) + (a.bias ? a.bias[i] : 0.f); sm[i] = v; sq += v * v; }
  for (int i = tid; i < nk; i += NT) { const float v = Act<T>::ld(src + a.k_off + i) + (a.bias ? a.bias[a.k_off + i] : 0.f); sm[ko + i] = v; sk += v * v; }
  for (int i = tid; i < nv; i += NT) {
    float v = Act<T>::ld(src + a.v_off + i) + (a.bias ? a.bias[a.v_off + i] : 0.f);
    float* vf = a.v_first + (int64_t)r * nv + i;
    if (a.v_store) *vf = v;
    if (a.v_use) v = (1.f - a.lambda) * v + a.lambda * *vf;
    sm[vo + i] = v;
  }
  sq = block_sum(sq, red[0]);
  sk = block_sum(sk, red[1]);   // (its barrier also publishes sm)
  const float rq = 1.0f / sqrtf(sq / (float)nq + a.eps), rk = 1.0f / sqrtf(sk / (float)nk + a.eps);
  const int half = a.rope_dims / 2;
  const float2* cs = reinterpret_cast<const float2*>(a.rope) + (int64_t)r * half;
  auto rotated = [&](bool is_k, int head, int d) {
    const bf16_t* w = (const bf16_t*)(is_k ? a.k_norm : a.q_norm);
    const float rinv = is_k ? rk : rq;
    const int so = is_k ? ko : 0, j = head * a.dim + d;
    const float x = sm[so + j] * rinv * bf2f(w[j]);
    if (d >= a.rope_dims) return x;
    const int pd = d < half ? d + half : d - half, pj = head * a.dim + pd;
    const float y = sm[so + pj] * rinv * bf2f(w[pj]);
    const float2 t = cs[d < half ? d : pd];
    return d < half ? x * t.x - y * t.y : x * t.x + y * t.y;
  };
  const int page = pos / KV_PAGE_TOKENS, tk = pos % KV_PAGE_TOKENS;
  const int dq = a.kv.dq, dv = a.kv.dv;
  T* kp = reinterpret_cast<T*>(a.kv.tab[(int64_t)e.slot * a.kv.ld + page] + a.kv.layer_off);
  T* vp = kp + (int64_t)a.kvh * KV_PAGE_TOKENS * dq;
  if (FRAG) {
    // 8 dims (16 bytes) per item; dq is 32 * a power of two
    const int sh = 31 - __builtin_clz(dq >> 3), np = dq >> 3;
    for (int i = tid; i < (a.heads + a.kvh) * np; i += NT) {
      const int hd = i >> sh, d0 = (i & (np - 1)) * 8;
      const bool is_k = hd >= a.heads;
      float y[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = d0 + j < a.dim ? rotated(is_k, is_k ? hd - a.heads : hd, d0 + j) : 0.f;
      const u32x4_t o = {pack_bf(y[0], y[1]), pack_bf(y[2], y[3]), pack_bf(y[4], y[5]), pack_bf(y[6], y[7])};
      if (is_k) *reinterpret_cast<u32x4_t*>((bf16_t*)kp + (int64_t)(hd - a.heads) * KV_PAGE_TOKENS * dq + kpage_elem(tk, d0, dq >> 5)) = o;
      else *reinterpret_cast<u32x4_t*>((bf16_t*)a.q_out + ((int64_t)r * a.heads + hd) * dq + d0) = o;
    }
    for (int h = tid >> 6; h < a.kvh; h += NT / 64)
      for (int d = tid & 63; d < a.vdim; d += 64) Act<T>::st(vp + (int64_t)h * KV_PAGE_TOKENS * dv + vpage_elem(tk, d), sm[vo + h * a.vdim + d]);
  } else {
    for (int h = tid >> 6; h < a.heads + a.kvh; h += NT / 64) {
      const bool is_k = h >= a.heads;
      for (int d = tid & 63; d < a.dim; d += 64) {
        if (is_k) Act<T>::st(kp + ((int64_t)(h - a.heads) * KV_PAGE_TOKENS + tk) * dq + d, rotated(true, h - a.heads, d));
        else Act<T>::st((T*)a.q_out + ((int64_t)r * a.heads + h) * dq + d, rotated(false, h, d));
      }
    }
    for (int h = tid >> 6; h < a.kvh; h += NT / 64)
      for (int d = tid & 63; d < a.vdim; d += 64) Act<T>::st(vp + ((int64_t)h * KV_PAGE_TOKENS + tk) * dv + d, sm[vo + h * a.vdim + d]);
  }
}

// The same for 32-bit rows on token-major pages whose dims come in fours: the row, the norm weights and the angles are requested 16 bytes at a time before
// anything waits (the loop above is a round trip per 256 columns and one more per pair of heads: 13.9 us at 16 + 2 x 8 heads x 128, 4.8).
// Q4 groups of four columns per thread hold the row (4096 of 4 * NT * Q4 at most); a thread's piece of a head is dims d .. d + 3 with their partners half a
// rotation further, or four dims behind the rotated ones.
constexpr int QF_NT = 512, QF_Q4 = 4;
__global__ __launch_bounds__(QF_NT) void qkv_post_f32_kernel(const float* qkv, const float* bias, const float* rope, const bf16_t* q_norm, const bf16_t* k_norm, int ld, int heads_kvh, QkvPostArgs a,
                                                             SeqBatch b) {
  extern __shared__ __attribute__((aligned(16))) float sm[];   // q | k of the row
  __shared__ float red[2][QF_NT / 64];
  const int r = blockIdx.x, tid = threadIdx.x;
  const int heads = heads_kvh >> 16, kvh = heads_kvh & 0xffff;
  const int nq = heads * a.dim, nk = kvh * a.dim, nv = kvh * a.vdim, n = nq + nk + nv;
  float4 v[QF_Q4], bi[QF_Q4], first[QF_Q4];
#pragma unroll
  for (int j = 0; j < QF_Q4; ++j) {
    const int i = min((tid + j * QF_NT) * 4, n - 4);
    const int at = i < nq ? i : i < nq + nk ? i - nq + a.k_off : i - nq - nk + a.v_off;
    v[j] = *reinterpret_cast<const float4*>(qkv + (int64_t)r * ld + at);
    bi[j] = bias ? *reinterpret_cast<const float4*>(bias + at) : make_float4(0.f, 0.f, 0.f, 0.f);
    first[j] = a.v_use && i >= nq + nk ? *reinterpret_cast<const float4*>(a.v_first + (int64_t)r * nv + i - nq - nk) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  // this thread's pieces of the heads: at most QF_Q4 of them (two quarters of the row's columns per piece where all dims rotate)
  const int half = a.rope_dims >> 1, hp = half >> 2, per = (a.dim >> 2) - hp, np = (heads + kvh) * per;
  uint2 wx[QF_Q4], wy[QF_Q4];
  float4 cs[QF_Q4][2];
#pragma unroll
  for (int j = 0; j < QF_Q4; ++j) {
    const int it = min(tid + j * QF_NT, np - 1), hd = it / per, p = it - hd * per, d = p < hp ? p * 4 : a.rope_dims + (p - hp) * 4;
    const bf16_t* w = hd < heads ? q_norm + hd * a.dim : k_norm + (hd - heads) * a.dim;
    wx[j] = *reinterpret_cast<const uint2*>(w + d);
    wy[j] = *reinterpret_cast<const uint2*>(w + (p < hp ? d + half : d));
    const float4* t = reinterpret_cast<const float4*>(rope + ((int64_t)r * half + (p < hp ? d : 0)) * 2);
    cs[j][0] = hp > 0 ? t[0] : make_float4(1.f, 0.f, 1.f, 0.f);
    cs[j][1] = hp > 0 ? t[1] : make_float4(1.f, 0.f, 1.f, 0.f);
  }
  const SeqEntry e = seq_entry_at(b, entry_of_row(b, r));
  const int pos = e.pos0 + r - e.row0, page = pos / KV_PAGE_TOKENS, tk = pos % KV_PAGE_TOKENS, dq = a.kv.dq, dv = a.kv.dv;
  float* kp = reinterpret_cast<float*>(a.kv.tab[(int64_t)e.slot * a.kv.ld + page] + a.kv.layer_off);
  float* vp = kp + (int64_t)kvh * KV_PAGE_TOKENS * dq;
  float sq = 0.f, sk = 0.f;
#pragma unroll
  for (int j = 0; j < QF_Q4; ++j) {
    const int i = (tid + j * QF_NT) * 4;
    if (i >= n) continue;
    const float4 x = make_float4(v[j].x + bi[j].x, v[j].y + bi[j].y, v[j].z + bi[j].z, v[j].w + bi[j].w);
    if (i < nq + nk) {
      *reinterpret_cast<float4*>(sm + i) = x;
      (i < nq ? sq : sk) += (x.x * x.x + x.y * x.y) + (x.z * x.z + x.w * x.w);
      continue;
    }
    const int iv = i - nq - nk, h = iv / a.vdim, d = iv - h * a.vdim;
    if (a.v_store) *reinterpret_cast<float4*>(a.v_first + (int64_t)r * nv + iv) = x;
    const float4 f = a.v_store ? x : first[j];   // (stored and used at once: the value itself)
    float4 y = x;
    if (a.v_use) {
      const float k0 = 1.f - a.lambda, k1 = a.lambda;
      y = make_float4(k0 * x.x + k1 * f.x, k0 * x.y + k1 * f.y, k0 * x.z + k1 * f.z, k0 * x.w + k1 * f.w);
    }
    *reinterpret_cast<float4*>(vp + ((int64_t)h * KV_PAGE_TOKENS + tk) * dv + d) = y;
  }
  sq = block_sum_n<QF_NT>(sq, red[0]);
  sk = block_sum_n<QF_NT>(sk, red[1]);   // (its barrier also publishes sm)
  const float rq = 1.0f / sqrtf(sq / (float)nq + a.eps), rk = 1.0f / sqrtf(sk / (float)nk + a.eps);
#pragma unroll
  for (int j = 0; j < QF_Q4; ++j) {
    const int it = tid + j * QF_NT;
    if (it >= np) continue;
    const int hd = it / per, p = it - hd * per, d = p < hp ? p * 4 : a.rope_dims + (p - hp) * 4;
    const float rinv = hd < heads ? rq : rk;
    float* dst = hd < heads ? (float*)a.q_out + ((int64_t)r * heads + hd) * dq : kp + ((int64_t)(hd - heads) * KV_PAGE_TOKENS + tk) * dq;
    const float4 s = *reinterpret_cast<const float4*>(sm + hd * a.dim + d);
    const float x[4] = {s.x * rinv * lo_bf(wx[j].x), s.y * rinv * hi_bf(wx[j].x), s.z * rinv * lo_bf(wx[j].y), s.w * rinv * hi_bf(wx[j].y)};
    if (p >= hp) {
      *reinterpret_cast<float4*>(dst + d) = make_float4(x[0], x[1], x[2], x[3]);
      continue;
    }
    const float4 t = *reinterpret_cast<const float4*>(sm + hd * a.dim + d + half);
    const float y[4] = {t.x * rinv * lo_bf(wy[j].x), t.y * rinv * hi_bf(wy[j].x), t.z * rinv * lo_bf(wy[j].y), t.w * rinv * hi_bf(wy[j].y)};
    const float co[4] = {cs[j][0].x, cs[j][0].z, cs[j][1].x, cs[j][1].z}, si[4] = {cs[j][0].y, cs[j][0].w, cs[j][1].y, cs[j][1].w};
    *reinterpret_cast<float4*>(dst + d) = make_float4(x[0] * co[0] - y[0] * si[0], x[1] * co[1] - y[1] * si[1], x[2] * co[2] - y[2] * si[2], x[3] * co[3] - y[3] * si[3]);
    *reinterpret_cast<float4*>(dst + d + half) = make_float4(y[0] * co[0] + x[0] * si[0], y[1] * co[1] + x[1] * si[1], y[2] * co[2] + x[2] * si[2], y[3] * co[3] + x[3] * si[3]);
  }
}

// The same for bf16 rows whose head dims, value dims and rotated half come in eights (16-byte pieces, fragment-major pages): blocks [0, rows)
// norm and rotate the q and k heads of a row, an eight-dim piece per thread and step; the first v_blocks mix the values and write the V pages
// (few blocks with a long chain each: first, so that they are no tail), a thread gathering eight token slots x eight dims (the slots of a piece are contiguous in the page).
__global__ __launch_bounds__(1024) void qkv_post_frag_kernel(QkvPostArgs a, SeqBatch b, int pages_per_entry, int v_blocks) {
  const int tid = threadIdx.x, nth = blockDim.x, dq = a.kv.dq, dv = a.kv.dv;
  auto unpack = [](u32x4_t w, float (&f)[8]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) { f[2 * j] = lo_bf(w[j]); f[2 * j + 1] = hi_bf(w[j]); }
  };
  auto piece = [&](const bf16_t* row, int c, float (&f)[8]) {   // eight columns of a row, bias added
    unpack(ld16(row + c), f);
    if (a.bias) {
      const float4 lo = *reinterpret_cast<const float4*>(a.bias + c), hi = *reinterpret_cast<const float4*>(a.bias + c + 4);
      f[0] += lo.x; f[1] += lo.y; f[2] += lo.z; f[3] += lo.w; f[4] += hi.x; f[5] += hi.y; f[6] += hi.z; f[7] += hi.w;
    }
  };
  if ((int)blockIdx.x >= v_blocks) {
    __shared__ float red[2][16];
    const int r = (int)blockIdx.x - v_blocks;
    const SeqEntry e = seq_entry_at(b, entry_of_row(b, r));
    const int pos = e.pos0 + r - e.row0, nq = a.heads * a.dim, nk = a.kvh * a.dim;
    const bf16_t* row = (const bf16_t*)a.qkv + (int64_t)r * a.ld;
    const int half = a.rope_dims / 2, sh = 31 - __builtin_clz(dq >> 3), np = dq >> 3, items = (a.heads + a.kvh) * np;
    const float* cs = a.rope + (int64_t)r * half * 2;
    // an item: eight dims d0 .. of head hd (q heads, then k heads); everything it needs but the two sums is requested before they are known
    struct Item { float x[8], y[8], t[16]; u32x4_t g, gp; };
    auto split_item = [&](int i, int* h, int* d0) {
      const int hd = i >> sh;
      *d0 = (i & (np - 1)) * 8;
      const bool is_k = hd >= a.heads;
      *h = is_k ? hd - a.heads : hd;
      return is_k;
    };
    auto fetch = [&](int i, Item& it) {
      int h, d0;
      const bool is_k = split_item(i, &h, &d0);
      if (d0 >= a.dim) return;
      const int w0 = h * a.dim + d0, off = is_k ? a.k_off : 0;
      const bf16_t* w = (const bf16_t*)(is_k ? a.k_norm : a.q_norm);
      piece(row, off + w0, it.x);
      it.g = ld16(w + w0);
      if (d0 < a.rope_dims) {
        const int pd = d0 < half ? half : -half, t0 = d0 < half ? d0 : d0 - half;
        piece(row, off + w0 + pd, it.y);
        it.gp = ld16(w + w0 + pd);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float4 v = *reinterpret_cast<const float4*>(cs + t0 * 2 + j * 4);
          it.t[4 * j] = v.x; it.t[4 * j + 1] = v.y; it.t[4 * j + 2] = v.z; it.t[4 * j + 3] = v.w;
        }
      }
    };
    Item first;
    if (tid < items) fetch(tid, first);
    float sq = 0.f, sk = 0.f;
    for (int i = tid; i < items; i += nth) {
      int h, d0;
      const bool is_k = split_item(i, &h, &d0);
      if (d0 >= a.dim) continue;
      float f[8], s = 0.f;
      if (i != tid) piece(row, (is_k ? a.k_off : 0) + h * a.dim + d0, f);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float v = i == tid ? first.x[j] : f[j];
        s = fmaf(v, v, s);
      }
      if (is_k) sk += s;
      else sq += s;
    }
    sq = wave_sum(sq);
    sk = wave_sum(sk);
    if ((tid & 63) == 0) { red[0][tid >> 6] = sq; red[1][tid >> 6] = sk; }
    __syncthreads();
    sq = sk = 0.f;
    for (int w = 0; w < nth / 64; ++w) { sq += red[0][w]; sk += red[1][w]; }
    const float rq = 1.0f / sqrtf(sq / (float)nq + a.eps), rk = 1.0f / sqrtf(sk / (float)nk + a.eps);
    bf16_t* kp = reinterpret_cast<bf16_t*>(a.kv.tab[(int64_t)e.slot * a.kv.ld + pos / KV_PAGE_TOKENS] + a.kv.layer_off);
    auto finish = [&](int i, const Item& it) {
      int h, d0;
      const bool is_k = split_item(i, &h, &d0);
      const float rinv = is_k ? rk : rq;
      u32x4_t o = {0u, 0u, 0u, 0u};
      if (d0 < a.dim) {
        float x[8], g[8];
        unpack(it.g, g);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = it.x[j] * rinv * g[j];
        if (d0 < a.rope_dims) {
          const bool lo = d0 < half;
          unpack(it.gp, g);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float z = it.y[j] * rinv * g[j];
            x[j] = fmaf(x[j], it.t[2 * j], (lo ? -z : z) * it.t[2 * j + 1]);
          }
        }
        o = u32x4_t{pack_bf(x[0], x[1]), pack_bf(x[2], x[3]), pack_bf(x[4], x[5]), pack_bf(x[6], x[7])};
      }
      if (is_k) *reinterpret_cast<u32x4_t*>(kp + (int64_t)h * KV_PAGE_TOKENS * dq + kpage_elem(pos % KV_PAGE_TOKENS, d0, dq >> 5)) = o;
      else *reinterpret_cast<u32x4_t*>((bf16_t*)a.q_out + ((int64_t)r * a.heads + h) * dq + d0) = o;
    };
    if (tid < items) finish(tid, first);
    for (int i = tid + nth; i < items; i += nth) {
      Item it;
      fetch(i, it);
      finish(i, it);
    }
    return;
  }
  // ---- V pages: unit = (entry, page of the entry, kv head), dv threads per unit (dv is 32, 64, 128 or 256)
  const int64_t u = (int64_t)blockIdx.x * nth + tid;
  const int lu = (int)(u & (dv - 1)), nd = dv >> 3;
  int unit = (int)(u >> (31 - __builtin_clz(dv)));
  const int h = unit % a.kvh;
  unit /= a.kvh;
  const int ent = unit / pages_per_entry;
  if (ent >= b.n) return;
  const SeqEntry e = seq_entry_at(b, ent);
  const int page = e.pos0 / KV_PAGE_TOKENS + unit % pages_per_entry;
  const int dchunk = lu & (nd - 1), g8 = lu >> (31 - __builtin_clz(nd)), kk = g8 >> 2, G = g8 & 3, d0 = dchunk * 8;
  if (page > (e.pos0 + e.len - 1) / KV_PAGE_TOKENS || d0 >= a.vdim) return;
  const int nv = a.kvh * a.vdim;
  uint32_t in[8][4];
  bool ok[8], all = true;
#pragma unroll
  for (int s = 0; s < 8; ++s) {   // slot order inside the piece: s = sub1 * 4 + j  <->  token kk * 32 + sub1 * 16 + G * 4 + j
    const int rel = page * KV_PAGE_TOKENS + kk * 32 + (s >> 2) * 16 + G * 4 + (s & 3) - e.pos0;
    ok[s] = rel >= 0 && rel < e.len;
    all &= ok[s];
    const int64_t r = e.row0 + min(max(rel, 0), e.len - 1);
    float v[8];
    piece((const bf16_t*)a.qkv + r * a.ld, a.v_off + h * a.vdim + d0, v);
    float* vf = a.v_first + r * nv + h * a.vdim + d0;
    if (a.v_store && ok[s]) {
      *reinterpret_cast<float4*>(vf) = make_float4(v[0], v[1], v[2], v[3]);
      *reinterpret_cast<float4*>(vf + 4) = make_float4(v[4], v[5], v[6], v[7]);
    }
    if (a.v_use) {
      const float4 lo = *reinterpret_cast<const float4*>(vf), hi = *reinterpret_cast<const float4*>(vf + 4);
      const float m = a.lambda, c = 1.f - a.lambda;
      v[0] = fmaf(m, lo.x, c * v[0]); v[1] = fmaf(m, lo.y, c * v[1]); v[2] = fmaf(m, lo.z, c * v[2]); v[3] = fmaf(m, lo.w, c * v[3]);
      v[4] = fmaf(m, hi.x, c * v[4]); v[5] = fmaf(m, hi.y, c * v[5]); v[6] = fmaf(m, hi.z, c * v[6]); v[7] = fmaf(m, hi.w, c * v[7]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) in[s][j] = pack_bf(v[2 * j], v[2 * j + 1]);
  }
  bf16_t* vb = reinterpret_cast<bf16_t*>(a.kv.tab[(int64_t)e.slot * a.kv.ld + page] + a.kv.layer_off) + (int64_t)a.kvh * KV_PAGE_TOKENS * dq + (int64_t)h * dv * KV_PAGE_TOKENS;
#pragma unroll
  for (int dd = 0; dd < 8; ++dd) {
    const int d = d0 + dd;
    u32x4_t o;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const uint32_t a0 = in[2 * w][dd >> 1], a1 = in[2 * w + 1][dd >> 1];
      o[w] = (dd & 1) ? ((a0 >> 16) | (a1 & 0xffff0000u)) : ((a0 & 0xffffu) | (a1 << 16));
    }
    bf16_t* dst = vb + ((((d >> 4) * 2 + kk) * 64 + G * 16 + (d & 15)) << 3);
    if (all) {
      *reinterpret_cast<u32x4_t*>(dst) = o;
    } else {
#pragma unroll
      for (int s = 0; s < 8; ++s)
        if (ok[s]) dst[s] = (bf16_t)((s & 1) ? (o[s >> 1] >> 16) : (o[s >> 1] & 0xffffu));
    }
  }
}

// NVZ * 4 * NTH columns of the row in registers (NVZ = 0: any width, the row is read twice)
template <typename T, int NTH, int NVZ>
__global__ __launch_bounds__(NTH) void polynorm_rows_kernel(const void* zp, int64_t ldz, PolyNormArgs a) {
  a.z = zp;   // (what the first requests need: in scalar registers at the start, gemv_body.h)
  a.ld = ldz;
  __shared__ float red[3][NTH / 64];
  constexpr bool REGS = NVZ > 0;
  const T* z = (const T*)a.z + (int64_t)blockIdx.x * a.ld;
  T* o = (T*)a.out + (int64_t)blockIdx.x * a.ld;
  const int tid = threadIdx.x, ld = (int)a.ld;
  float4 v[REGS ? NVZ : 1];
  float s1 = 0.f, s2 = 0.f, s3 = 0.f;
  auto add = [&](float x) {
    const float v2 = x * x, v4 = v2 * v2;
    s1 += v2;
    s2 += v4;
    s3 = fmaf(v4, v2, s3);
  };
  auto add4 = [&](float4 x) { add(x.x); add(x.y); add(x.z); add(x.w); };   // (pad columns are zero)
  if constexpr (REGS) {
#pragma unroll
    for (int i = 0; i < NVZ; ++i) v[i] = Act<T>::ld4(z + min((i * NTH + tid) * 4, ld - 4));
#pragma unroll
    for (int i = 0; i < NVZ; ++i) {
      if ((i * NTH + tid) * 4 >= ld) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      add4(v[i]);
    }
  } else {
    for (int c = tid * 4; c < ld; c += NTH * 4) add4(Act<T>::ld4(z + c));
  }
  s1 = block_sum_n<NTH>(s1, red[0]);
  s2 = block_sum_n<NTH>(s2, red[1]);
  s3 = block_sum_n<NTH>(s3, red[2]);
  const float inv = 1.0f / (float)a.ff;
  const float r1 = a.coef[0] / sqrtf(s1 * inv + a.eps), r2 = a.coef[1] / sqrtf(s2 * inv + a.eps), r3 = a.coef[2] / sqrtf(s3 * inv + a.eps);
  auto act = [&](float x) { return fmaf(x, fmaf(x, fmaf(x, r3, r2), r1), a.coef[3]); };
  auto put = [&](int c, float4 x) {
    Act<T>::st4(o + c, make_float4(c < a.ff ? act(x.x) : 0.f, c + 1 < a.ff ? act(x.y) : 0.f, c + 2 < a.ff ? act(x.z) : 0.f, c + 3 < a.ff ? act(x.w) : 0.f));
  };
  if constexpr (REGS) {
#pragma unroll
    for (int i = 0; i < NVZ; ++i)
      if ((i * NTH + tid) * 4 < ld) put((i * NTH + tid) * 4, v[i]);
  } else {
    for (int c = tid * 4; c < ld; c += NTH * 4) put(c, Act<T>::ld4(z + c));
  }
}

template <typename T, bool EMBED>
void postnorm_conv_t(const PostNormArgs& a, const SeqBatch& b, hipStream_t st) {
  // rows per block: a tile repeats the norm of its taps - 1 preceding rows, a short grid leaves CUs idle
  using std::integral_constant;
  if (b.max_len == 1 && a.h_out && a.conv.taps >= 2 && a.conv.taps <= 4 && a.ld <= 4096) {
    auto step = [&](auto nth, auto taps) {
      constexpr int NTH = decltype(nth)::value, TAPS = decltype(taps)::value;
      hipLaunchKernelGGL((postnorm_conv_step_kernel<T, NTH, TAPS, EMBED>), dim3((unsigned)b.rows), dim3(NTH), 0, st, a.x_in, a.y, a.norm_w, a.conv.w, b.entries, (int)a.ld, a.ldy, a, b);
    };
    auto by_taps = [&](auto nth) {
      if (a.conv.taps == 2) step(nth, integral_constant<int, 2>{});
      else if (a.conv.taps == 3) step(nth, integral_constant<int, 3>{});
      else step(nth, integral_constant<int, 4>{});
    };
    if (a.ld <= 1024) by_taps(integral_constant<int, 256>{});
    else if (a.ld <= 2048) by_taps(integral_constant<int, 512>{});
    else by_taps(integral_constant<int, 1024>{});
    return;
  }
  if constexpr (!EMBED) {
    if (b.max_len > 1 && a.y && a.h_out && a.conv.taps >= 2 && a.conv.taps <= 4 && a.ld <= 4096) {
      auto tiled = [&](auto nth, auto taps, auto tl) {
        constexpr int NTH = decltype(nth)::value, TAPS = decltype(taps)::value, TILE = decltype(tl)::value;
        const int nt = ((b.rows + TILE - 1) / TILE + 7) / 8 * 8;   // (whole rounds over the XCDs: the tile order needs them)
        hipLaunchKernelGGL((postnorm_conv_tile_kernel<T, NTH, TAPS, TILE>), dim3((unsigned)nt), dim3(NTH), 0, st, a, b);
      };
      auto by_rows = [&](auto nth, auto taps) {
        if (b.rows >= 4096) tiled(nth, taps, integral_constant<int, 8>{});
        else if (b.rows >= 1024) tiled(nth, taps, integral_constant<int, 4>{});
        else tiled(nth, taps, integral_constant<int, 2>{});
      };
      auto by_taps = [&](auto nth) {
        if (a.conv.taps == 2) by_rows(nth, integral_constant<int, 2>{});
        else if (a.conv.taps == 3) by_rows(nth, integral_constant<int, 3>{});
        else by_rows(nth, integral_constant<int, 4>{});
      };
      if (a.ld <= 1024) by_taps(integral_constant<int, 256>{});
      else if (a.ld <= 2048) by_taps(integral_constant<int, 512>{});
      else by_taps(integral_constant<int, 1024>{});
      return;
    }
  }
  const int tile = b.max_len == 1 ? 1 : b.rows >= 4096 ? 8 : b.rows >= 1024 ? 4 : 2;
  auto go = [&](auto nth, auto nv) {
    constexpr int NTH = decltype(nth)::value, NV = decltype(nv)::value;
    const size_t lds = a.h_out ? (size_t)(a.conv.taps - 1) * NV * NTH * 16 : 0;
    hipLaunchKernelGGL((postnorm_conv_kernel<T, NTH, NV, EMBED>), dim3((unsigned)((b.rows + tile - 1) / tile)), dim3(NTH), lds, st, a, b, tile);
  };
  if (a.ld <= 1024) go(integral_constant<int, 256>{}, integral_constant<int, 1>{});
  else if (a.ld <= 2048) go(integral_constant<int, 512>{}, integral_constant<int, 1>{});
  else if (a.ld <= 4096) go(integral_constant<int, 1024>{}, integral_constant<int, 1>{});
  else go(integral_constant<int, 1024>{}, integral_constant<int, 2>{});
}

}  // namespace

void launch_postnorm_conv(const PostNormArgs& a, const SeqBatch& b, bool f32, hipStream_t st) {
  if (b.rows <= 0) return;
  if (a.embed) {
    if (f32) postnorm_conv_t<float, true>(a, b, st);
    else postnorm_conv_t<bf16_t, true>(a, b, st);
  } else {
    if (f32) postnorm_conv_t<float, false>(a, b, st);
    else postnorm_conv_t<bf16_t, false>(a, b, st);
  }
}

void launch_final_rows(const FinalRowsArgs& a, bool f32, hipStream_t st) {
  if (a.n <= 0) return;
  const size_t lds = (size_t)a.ld * 4;
  auto go = [&](auto k) { hipLaunchKernelGGL(k, dim3((unsigned)a.n), dim3(NT), lds, st, a); };
  const bool norm = a.norm_w && a.y;
  if (a.ld <= 4 * NT) f32 ? norm ? go(final_rows_kernel<float, 4, true>) : go(final_rows_kernel<float, 4, false>) : norm ? go(final_rows_kernel<bf16_t, 4, true>) : go(final_rows_kernel<bf16_t, 4, false>);
  else f32 ? norm ? go(final_rows_kernel<float, 16, true>) : go(final_rows_kernel<float, 16, false>) : norm ? go(final_rows_kernel<bf16_t, 16, true>) : go(final_rows_kernel<bf16_t, 16, false>);
}

void launch_rope_pairs(const SeqBatch& b, double base, int dims, float* tab, hipStream_t st) {
  const int64_t n = (int64_t)b.rows * (dims / 2);
  if (n > 0) hipLaunchKernelGGL(rope_pairs_kernel, dim3((unsigned)((n + NT - 1) / NT)), dim3(NT), 0, st, b, base, dims / 2, tab);
}

void launch_qkv_post(const QkvPostArgs& a, const SeqBatch& b, bool f32, hipStream_t st) {
  if (b.rows <= 0) return;
  const size_t lds = (size_t)((a.heads + a.kvh) * a.dim + a.kvh * a.vdim) * 4;
  const dim3 grid((unsigned)b.rows), block(NT);
  if (!f32 && a.kv.frag && a.dim % 8 == 0 && a.vdim % 8 == 0 && a.rope_dims % 16 == 0) {
    const int pages = (b.max_len + KV_PAGE_TOKENS - 1) / KV_PAGE_TOKENS + 1;   // pages one entry's rows can touch
    const int64_t vt = (int64_t)b.n * pages * a.kvh * a.kv.dv;
    const int nth = 256, vb = (int)((vt + nth - 1) / nth);
    hipLaunchKernelGGL(qkv_post_frag_kernel, dim3((unsigned)(vb + b.rows)), dim3(nth), 0, st, a, b, pages, vb);
    return;
  }
  const int n = (a.heads + a.kvh) * a.dim + a.kvh * a.vdim;
  const bool fours = ((a.dim | a.vdim | a.k_off | a.v_off | a.kv.dq | a.kv.dv) & 3) == 0 && (a.ld & 3) == 0 && a.rope_dims % 8 == 0 && a.heads < 32768 && a.ld < (1 << 30) &&
                     (((uintptr_t)a.qkv | (uintptr_t)a.bias | (uintptr_t)a.rope | (uintptr_t)a.q_norm | (uintptr_t)a.k_norm | (uintptr_t)a.v_first | (uintptr_t)a.q_out) & 15) == 0;
  const int pieces = (a.heads + a.kvh) * ((a.dim >> 2) - (a.rope_dims >> 3));
  if (f32 && fours && n <= 4 * QF_NT * QF_Q4 && pieces <= QF_NT * QF_Q4) {
    hipLaunchKernelGGL(qkv_post_f32_kernel, grid, dim3(QF_NT), (size_t)(a.heads + a.kvh) * a.dim * 4, st, (const float*)a.qkv, a.bias, a.rope, (const bf16_t*)a.q_norm, (const bf16_t*)a.k_norm,
                       (int)a.ld, a.heads << 16 | a.kvh, a, b);
    return;
  }
  if (f32) hipLaunchKernelGGL((qkv_post_kernel<float, false>), grid, block, lds, st, a, b);
  else if (a.kv.frag) hipLaunchKernelGGL((qkv_post_kernel<bf16_t, true>), grid, block, lds, st, a, b);
  else hipLaunchKernelGGL((qkv_post_kernel<bf16_t, false>), grid, block, lds, st, a, b);
}

void launch_polynorm_rows(const PolyNormArgs& a, bool f32, hipStream_t st) {
  if (a.rows <= 0) return;
  auto go = [&](auto k, int nth) { hipLaunchKernelGGL(k, dim3((unsigned)a.rows), dim3(nth), 0, st, a.z, (int64_t)a.ld, a); };
  if (f32) go(polynorm_rows_kernel<float, 256, 0>, 256);
  else if (a.ld <= 4096) go(polynorm_rows_kernel<bf16_t, 256, 4>, 256);
  else if (a.ld <= 8192) go(polynorm_rows_kernel<bf16_t, 512, 4>, 512);
  else if (a.ld <= 12288) go(polynorm_rows_kernel<bf16_t, 512, 6>, 512);
  else if (a.ld <= 16384) go(polynorm_rows_kernel<bf16_t, 512, 8>, 512);
  else go(polynorm_rows_kernel<bf16_t, 512, 0>, 512);
}

}  // namespace aha
