// D11 on the device: the deterministic half of `sample_and_push` (reference src/models/common/generate.rs:70-86) --
// repeat penalty (src/models/common/sample.rs:41-60 -> candle_transformers::utils::apply_repeat_penalty) and the candidate
// set of candle's LogitsProcessor (Sampling::TopK / TopKThenTopP / TopP, sample.rs:7-38): the k largest penalised logits
// with their vocabulary indices, plus the max and the sum of exp((x - max) / T) over the WHOLE vocabulary, so that the host
// gets the same probabilities candle's full-vocabulary softmax would give those k tokens.  The random draw stays on the host
// (the caller's RNG): 8k + 8 bytes cross PCIe per token instead of the 608 KB logits vector.
//
// HBM-bound integer/compare work: one pass over V f32 logits (608 KB), no LDS staging needed.  Selection is k rounds of
// (wave max, lowest index among the maxima) over register-resident candidates: exact, ordered by (value desc, index asc).
#include "common.h"
#include "kernels.h"

namespace aha {
namespace {

__device__ __forceinline__ unsigned wave_min_u32(unsigned v) {
  {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    v = min(r[0], r[1]);
  }
  {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = min(r[0], r[1]);
  }
  v = min(v, (unsigned)__builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, false));
  v = min(v, (unsigned)__builtin_amdgcn_update_dpp(0, v, 0x124, 0xf, 0xf, false));
  v = min(v, (unsigned)__builtin_amdgcn_update_dpp(0, v, 0x122, 0xf, 0xf, false));
  v = min(v, (unsigned)__builtin_amdgcn_update_dpp(0, v, 0x121, 0xf, 0xf, false));
  return v;
}

constexpr unsigned NO_IDX = 0xffffffffu;

// k rounds over the C candidates each lane holds in registers.  emit(r, value, index) is called by every lane with the
// wave-uniform winner of round r (index NO_IDX once the candidates are exhausted).
template <int C, typename Emit>
__device__ __forceinline__ void wave_topk_rounds(float (&v)[C], unsigned (&id)[C], int k, Emit emit) {
  for (int r = 0; r < k; ++r) {
    float lm = v[0];
    unsigned li = id[0];
#pragma unroll
    for (int j = 1; j < C; ++j) {
      const bool better = v[j] > lm || (v[j] == lm && id[j] < li);
      lm = better ? v[j] : lm;
      li = better ? id[j] : li;
    }
    const float wm = wave_max(lm);
    const unsigned wi = wave_min_u32(lm == wm ? li : NO_IDX);
    emit(r, wm, wi);
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const bool hit = id[j] == wi && wi != NO_IDX;
      v[j] = hit ? -INFINITY : v[j];
      id[j] = hit ? NO_IDX : id[j];
    }
  }
}

// Total order (value desc, index asc) as one integer, larger = earlier; zeros compare equal, NaN and empty slots come last.
__device__ __forceinline__ uint64_t order_key(float v, unsigned id) {
  if (id == NO_IDX || v != v) return 0;
  const unsigned u = __float_as_uint(v + 0.0f), o = u & 0x80000000u ? ~u : u | 0x80000000u;
  return (uint64_t)o << 32 | (NO_IDX - id);
}

// work[t] = penalised logit of every context token t (reads the untouched logits, so duplicates in ctx write the same value:
// the reference applies the penalty once per distinct id through a HashSet).
__global__ void repeat_penalty_kernel(const float* logits, float* work, const uint32_t* ctx, int n, float penalty, int V) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t t = ctx[i];
  if (t >= (uint32_t)V) return;  // `logits.get_mut(token_id)` is None: ignored
  const float x = logits[t];
  work[t] = x >= 0.f ? x / penalty : x * penalty;
}

constexpr int S1_C = 8;                      // elements per lane in stage 1
constexpr int S1_WAVE_ELEMS = 64 * S1_C;     // 512 logits per wave
constexpr int S1_WAVES_PER_BLOCK = 4;

// stage 1: every wave reduces 512 consecutive logits to its k best and its softmax partial (max, sum exp((x - max) * inv_temp))
__global__ __launch_bounds__(64 * S1_WAVES_PER_BLOCK) void topk_stage1_kernel(const float* x, int V, int k, float inv_temp,
                                                                              float* cand_val, unsigned* cand_idx,
                                                                              float* part_m, float* part_s) {
  const int lane = threadIdx.x & 63;
  const int w = blockIdx.x * S1_WAVES_PER_BLOCK + (threadIdx.x >> 6);
  const int base = w * S1_WAVE_ELEMS;
  if (base >= V) return;
  float v[S1_C];
  unsigned id[S1_C];
  float lm = -INFINITY;
#pragma unroll
  for (int j = 0; j < S1_C; ++j) {
    const int i = base + j * 64 + lane;
    const bool ok = i < V;
    v[j] = ok ? x[ok ? i : 0] : -INFINITY;
    id[j] = ok ? (unsigned)i : NO_IDX;
    lm = fmaxf(lm, v[j]);
  }
  const float wm = wave_max(lm);
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < S1_C; ++j)
    if (id[j] != NO_IDX) s += __expf((v[j] - wm) * inv_temp);
  s = wm == -INFINITY ? 0.f : wave_sum(s);   // (a wave of -inf only: nothing, not the NaN of (-inf) - (-inf))
  if (lane == 0) {
    part_m[w] = wm;
    part_s[w] = s;
  }
  wave_topk_rounds<S1_C>(v, id, k, [&](int r, float val, unsigned idx) {
    if (lane == 0) {
      cand_val[(size_t)w * k + r] = val;
      cand_idx[(size_t)w * k + r] = idx;
    }
  });
}

// ---- up to 512 waves of logits (262 144 entries): three launches whose work follows k, not the vocabulary ------------------------------------------
// heads: every wave's largest entry and softmax partial; rounds: the k-th largest head bounds the k-th largest logit from below, so a wave emits only
// while its next entry is not below it (most emit none); final: one block ranks the k to k * k entries that are left by counting.
// Rounds over all waves' candidates, whoever could still win, were 67 us at 151 936 logits and k = 20 (14 + 27 + 25 us of dependent wave reductions);
// 5 + 12 + 6 us here.  Each round is 2.8 us of the call there and 0.2 us here, each wave's head 0.04 us here (every block compares all of them): up to a
// k per 70 waves the rounds are as fast or faster (call of the host in us, rounds / bound: 151 936 logits, k = 1 / 2 / 4: 35.4 / 42.7, 38.2 / 43.3,
// 43.7 / 43.9; 262 144, k = 1 / 7: 38.6 / 52.7, 55.8 / 53.6; 65 536, k = 1 / 2: 35.1 / 36.3, 37.9 / 36.5; 32 768, k = 1: 34.3 / 34.3).
constexpr int HEADS = 512, HEADS_PER_ROUND = 70, FINAL_CAP = 64 * 64;
__global__ __launch_bounds__(64 * S1_WAVES_PER_BLOCK) void topk_heads_kernel(const float* x, int V, float inv_temp, uint64_t* heads, float* part_m, float* part_s) {
  const int lane = threadIdx.x & 63, w = blockIdx.x * S1_WAVES_PER_BLOCK + (threadIdx.x >> 6), base = w * S1_WAVE_ELEMS;
  if (base >= V) return;
  float v[S1_C];
  uint64_t best = 0;
  float lm = -INFINITY;
#pragma unroll
  for (int j = 0; j < S1_C; ++j) {
    const int i = base + j * 64 + lane;
    v[j] = x[min(i, V - 1)];
    if (i >= V) v[j] = -INFINITY;
    const uint64_t k = order_key(v[j], i < V ? (unsigned)i : NO_IDX);
    best = k > best ? k : best;
    lm = fmaxf(lm, v[j]);
  }
  const float wm = wave_max(lm);
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < S1_C; ++j)
    if (base + j * 64 + lane < V) s += __expf((v[j] - wm) * inv_temp);
  s = wm == -INFINITY ? 0.f : wave_sum(s);   // (a wave of -inf only: nothing, not the NaN of (-inf) - (-inf))
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t other = __shfl_xor(best, o, 64);
    best = other > best ? other : best;
  }
  if (lane == 0) {
    part_m[w] = wm;
    part_s[w] = s;
    heads[w] = best;
  }
}

__global__ __launch_bounds__(64 * S1_WAVES_PER_BLOCK) void topk_rounds_kernel(const float* x, int V, int k, const uint64_t* heads, int nw, uint64_t* cand, int* count) {
  __shared__ uint64_t h[HEADS], bound;
  const int tid = threadIdx.x, lane = tid & 63, w = blockIdx.x * S1_WAVES_PER_BLOCK + (tid >> 6), base = w * S1_WAVE_ELEMS;
  float v[S1_C];
#pragma unroll
  for (int j = 0; j < S1_C; ++j) v[j] = x[min(base + j * 64 + lane, V - 1)];
  const int nw8 = (nw + 7) & ~7;
  for (int i = tid; i < nw8; i += 64 * S1_WAVES_PER_BLOCK) h[i] = i < nw ? heads[i] : 0;
  if (tid == 0) bound = 1;   // (fewer than k heads: everything but empty slots)
  __syncthreads();
  for (int i = tid; i < nw; i += 64 * S1_WAVES_PER_BLOCK) {
    const uint64_t mine = h[i];
    int above = 0;
    for (int j = 0; j < nw8; j += 8) {
#pragma unroll
      for (int u = 0; u < 8; ++u) above += h[j + u] > mine;
    }
    if (above == k - 1 && mine != 0) bound = mine;   // (keys are distinct: one thread)
  }
  __syncthreads();
  if (base >= V) return;
  const uint64_t least = bound;
  uint64_t key[S1_C], best = 0;
#pragma unroll
  for (int j = 0; j < S1_C; ++j) {
    const int i = base + j * 64 + lane;
    key[j] = order_key(v[j], i < V ? (unsigned)i : NO_IDX);
    best = key[j] > best ? key[j] : best;
  }
  int n = 0;
  while (n < k) {
    uint64_t m = best;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const uint64_t other = __shfl_xor(m, o, 64);
      m = other > m ? other : m;
    }
    if (m < least) break;
    if (lane == 0) cand[(size_t)w * k + n] = m;
    ++n;
    if (best == m) {   // (one lane: its next entry)
      uint64_t next = 0;
#pragma unroll
      for (int j = 0; j < S1_C; ++j) {
        if (key[j] == m) key[j] = 0;
        next = key[j] > next ? key[j] : next;
      }
      best = next;
    }
  }
  if (lane == 0) count[w] = n;
}

__global__ __launch_bounds__(1024) void topk_final_kernel(const float* x, const uint64_t* cand, const int* count, int nw, int k, const float* part_m, const float* part_s, float inv_temp,
                                                          float* out_val, unsigned* out_idx, float* out_ms) {
  __shared__ uint64_t keys[FINAL_CAP];
  __shared__ int cnt[HEADS], n;
  const int tid = threadIdx.x;
  if (tid == 0) n = 0;
  if (tid < nw) cnt[tid] = count[tid];
  if (tid < k) {
    out_val[tid] = -INFINITY;
    out_idx[tid] = NO_IDX;
  }
  __syncthreads();
  for (int i = tid; i < nw * k; i += 1024) {
    const int w = i / k;
    if (i - w * k < cnt[w]) keys[atomicAdd(&n, 1)] = cand[i];   // (at most k waves hold an entry as large as the k-th head, or fewer than k waves are there)
  }
  if (tid >= 960) {   // the last wave: the softmax partials
    const int lane = tid - 960;
    float m = -INFINITY;
    for (int i = lane; i < nw; i += 64) m = fmaxf(m, part_m[i]);
    const float M = wave_max(m);
    float s = 0.f;
    for (int i = lane; i < nw; i += 64) s += part_s[i] * __expf((part_m[i] - M) * inv_temp);
    s = wave_sum(s);
    if (lane == 0) {
      out_ms[0] = M;
      out_ms[1] = s;
    }
  }
  __syncthreads();
  for (int i = tid; i < n; i += 1024) {
    const uint64_t mine = keys[i];
    int r = 0;
    for (int j = 0; j < n; ++j) r += keys[j] > mine;
    if (r < k) {
      const unsigned id = NO_IDX - (unsigned)mine;
      out_val[r] = x[id];   // (the logit itself: a key has no signed zero)
      out_idx[r] = id;
    }
  }
}

// ---- larger vocabularies, few candidates of many waves: rounds over all candidates ----------------------------------------------------------------
constexpr int S2_WAVES = 16;
constexpr int S2_C = 20;  // 16 waves x 64 lanes x 20 >= 297 stage-1 waves x 64 candidates

// stage 2a (16 one-wave blocks, one per CU -- the rounds are VALU-bound, so the waves must not share a SIMD): each wave
// reduces a contiguous sixteenth of the stage-1 candidates to its k best
__global__ __launch_bounds__(64) void topk_stage2a_kernel(const float* cand_val, const unsigned* cand_idx, int n_cand, int k,
                                                          float* mid_val, unsigned* mid_idx) {
  const int lane = threadIdx.x, wave = blockIdx.x;
  const int chunk = (n_cand + S2_WAVES - 1) / S2_WAVES;
  const int c0 = wave * chunk, c1 = min(c0 + chunk, n_cand);
  float v[S2_C];
  unsigned id[S2_C];
#pragma unroll
  for (int j = 0; j < S2_C; ++j) {
    const int i = c0 + j * 64 + lane;
    const bool ok = i < c1;
    v[j] = ok ? cand_val[ok ? i : 0] : -INFINITY;
    id[j] = ok ? cand_idx[ok ? i : 0] : NO_IDX;
    if (id[j] == NO_IDX) v[j] = -INFINITY;
  }
  wave_topk_rounds<S2_C>(v, id, k, [&](int r, float val, unsigned idx) {
    if (lane == 0) {
      mid_val[wave * k + r] = val;
      mid_idx[wave * k + r] = idx;
    }
  });
}

// stage 2b (one wave): 16 x k -> k in (value desc, index asc) order, and the softmax partials -> (max, sumexp)
__global__ __launch_bounds__(64) void topk_stage2b_kernel(const float* mid_val, const unsigned* mid_idx, const float* part_m,
                                                          const float* part_s, int n_part, int k, float inv_temp,
                                                          float* out_val, unsigned* out_idx, float* out_ms) {
  const int lane = threadIdx.x;
  {
    float m = -INFINITY;
    for (int i = lane; i < n_part; i += 64) m = fmaxf(m, part_m[i]);
    const float M = wave_max(m);
    float s = 0.f;
    for (int i = lane; i < n_part; i += 64) s += part_s[i] * __expf((part_m[i] - M) * inv_temp);
    s = wave_sum(s);
    if (lane == 0) {
      out_ms[0] = M;
      out_ms[1] = s;
    }
  }
  float v[S2_WAVES];
  unsigned id[S2_WAVES];
#pragma unroll
  for (int j = 0; j < S2_WAVES; ++j) {
    const int i = j * 64 + lane;
    const bool ok = i < S2_WAVES * k;
    v[j] = ok ? mid_val[ok ? i : 0] : -INFINITY;
    id[j] = ok ? mid_idx[ok ? i : 0] : NO_IDX;
    if (id[j] == NO_IDX) v[j] = -INFINITY;
  }
  wave_topk_rounds<S2_WAVES>(v, id, k, [&](int r, float val, unsigned idx) {
    if (lane == 0) {
      out_val[r] = val;
      out_idx[r] = idx;
    }
  });
}

}  // namespace

int sample_stage1_waves(int V) { return (V + S1_WAVE_ELEMS - 1) / S1_WAVE_ELEMS; }
// u32 words of launch_topk_candidates' index array, whichever launches it takes
size_t sample_index_words(int V) {
  const size_t nw = sample_stage1_waves(V);
  return nw <= (size_t)HEADS ? 2 * (nw * 64 + HEADS) + HEADS : (nw + 16) * 64;
}
// k <= 64 and the stage-1 candidates within what stage 2a holds in registers (16 waves x 64 lanes x 20)
bool sample_shape_ok(int V, int k) { return V > 0 && k >= 1 && k <= 64 && (int64_t)sample_stage1_waves(V) * k <= S2_WAVES * 64 * S2_C; }

void launch_repeat_penalty(const float* logits, float* work, const uint32_t* ctx, int n, float penalty, int V, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(repeat_penalty_kernel, dim3((n + 255) / 256), dim3(256), 0, st, logits, work, ctx, n, penalty, V);
}

void launch_topk_candidates(const float* x, int V, int k, float inv_temp, float* cand_val, unsigned* cand_idx, float* part_m,
                            float* part_s, float* out_val, unsigned* out_idx, float* out_ms, hipStream_t st) {
  const int nw = sample_stage1_waves(V);
  const dim3 blocks((nw + S1_WAVES_PER_BLOCK - 1) / S1_WAVES_PER_BLOCK), threads(64 * S1_WAVES_PER_BLOCK);
  if (nw <= HEADS && k * HEADS_PER_ROUND > nw) {
    uint64_t* cand = reinterpret_cast<uint64_t*>(cand_idx);   // (sample_index_words: keys of all waves' k best, then heads and counts)
    uint64_t* heads = cand + (size_t)nw * 64;
    int* count = reinterpret_cast<int*>(heads + HEADS);
    hipLaunchKernelGGL(topk_heads_kernel, blocks, threads, 0, st, x, V, inv_temp, heads, part_m, part_s);
    hipLaunchKernelGGL(topk_rounds_kernel, blocks, threads, 0, st, x, V, k, heads, nw, cand, count);
    hipLaunchKernelGGL(topk_final_kernel, dim3(1), dim3(1024), 0, st, x, cand, count, nw, k, part_m, part_s, inv_temp, out_val, out_idx, out_ms);
    return;
  }
  hipLaunchKernelGGL(topk_stage1_kernel, dim3((nw + S1_WAVES_PER_BLOCK - 1) / S1_WAVES_PER_BLOCK), dim3(64 * S1_WAVES_PER_BLOCK), 0,
                     st, x, V, k, inv_temp, cand_val, cand_idx, part_m, part_s);
  // the 16 x k intermediates live right behind the stage-1 candidates (model.hip sizes cand_* as (nw + 16) * 64)
  float* mid_val = cand_val + (size_t)nw * 64;
  unsigned* mid_idx = cand_idx + (size_t)nw * 64;
  hipLaunchKernelGGL(topk_stage2a_kernel, dim3(S2_WAVES), dim3(64), 0, st, cand_val, cand_idx, nw * k, k, mid_val, mid_idx);
  hipLaunchKernelGGL(topk_stage2b_kernel, dim3(1), dim3(64), 0, st, mid_val, mid_idx, part_m, part_s, nw, k, inv_temp, out_val,
                     out_idx, out_ms);
}

}  // namespace aha
