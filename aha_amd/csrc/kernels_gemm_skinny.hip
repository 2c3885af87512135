// Projection GEMM for few rows (M <= 64: batched decode steps, short prompts): C[M,N] = A[M,K] . W[N,K]^T with the epilogues of kernels_gemm.hip.
//
// What bounds it is the weight matrix, read once from HBM; the 128-row tiles of kernels_gemm.hip stage 16 times the rows a batch of eight has and
// need K slices and a reduce pass to fill the chip.  Here a block owns R8 * 8 weight rows and the whole K range, its four waves take the 64-wide
// k chunks in turn, and every wave has a ring of S chunks of its own in LDS that it fills by DMA and drains by itself: no barrier before the sums
// of the four waves are joined, 2 KB to 9 KB of weights per stage in flight per wave.  A DMA request covers eight rows x 128 bytes (whole lines);
// operands that waves load to registers themselves as MFMA fragments touch 16 rows x 64 bytes per request and ran at half the rate (6144 x 4096,
// 8 rows: 17.5 us against 10.4 us).  A's rows go the same way: each block reads all of A, so blocks have as many weight rows as one round over
// the chip allows (gemm_skinny_rows).
// Rows past M, N repeat the last one; what they give is not stored.  Lanes of a fragment that no row backs read whatever LDS holds behind the
// stage: an MFMA's output rows and columns do not mix.
//
// Measured on MI355X, back to back from HBM, 8 rows (in brackets: the split-K ring kernel + its reduce pass it replaces, inside a batched step):
//   6144 x 4096 10.4 us (4.8 TB/s), 4096 x 4096 8.1, 12288 x 4096 18.0 (5.6), 4096 x 12288 17.9 (5.6), 24576 x 4096 33.1 (6.1)
//   [18.1 + 4.6 us on average over the first four]; 32 rows: 12.1, 10.1, 19.7, 25.9, 37.2; 64 rows: 15.5, 13.4, 23.3, 35.5, 45.9
#include "gemm256_body.h"

namespace aha {

namespace {

constexpr int SK_NW = 4;

template <int R8, int M8, int S, bool PAIRS>
__global__ __launch_bounds__(SK_NW * 64) void gemm_skinny_kernel(GemmArgs a) {
  constexpr int NF = (R8 + 1) / 2, MT = (M8 + 1) / 2, PER = R8 + M8;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), G = lane >> 4, c = lane & 15;
  char* ring = gemm_smem + wave * (S * PER * 1024);
  const bf16_t* src[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int local = (r < R8 ? r : r - R8) * 8 + (lane >> 3), slot = ((lane & 7) ^ ((local >> 1) & 7)) * 8;   // (the swizzle of swz())
    if (r >= R8) {
      src[r] = (const bf16_t*)a.A + (int64_t)min(local, a.M - 1) * a.lda + slot;
    } else if (PAIRS) {   // eight gate rows, then the eight up rows of the same columns (16-row blocks alternate in W)
      const int col = ((int)blockIdx.x * (R8 / 2) + r / 2) * 8 + (lane >> 3);
      src[r] = (const bf16_t*)a.W + (int64_t)min((col >> 4) * 32 + (r & 1) * 16 + (col & 15), a.N - 1) * a.ldw + slot;
    } else {
      src[r] = (const bf16_t*)a.W + (int64_t)min((int)blockIdx.x * (R8 * 8) + local, a.N - 1) * a.ldw + slot;
    }
  }
  f32x4_t acc[NF][MT];
#pragma unroll
  for (int r = 0; r < NF; ++r)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[r][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int nc = a.K / 64;
  auto load = [&](int u, int ch) {   // (past the end: the last chunk again, never used)
    const int k = min(ch, nc - 1) * 64;
#pragma unroll
    for (int r = 0; r < R8; ++r) __builtin_amdgcn_global_load_lds((glb_ptr_t)(src[r] + k), (lds_ptr_t)(ring + (u * PER + r) * 1024), 16, 0, 2);   // weights: non-temporal
#pragma unroll
    for (int r = R8; r < PER; ++r) __builtin_amdgcn_global_load_lds((glb_ptr_t)(src[r] + k), (lds_ptr_t)(ring + (u * PER + r) * 1024), 16, 0, 0);
  };
#pragma unroll
  for (int u = 0; u < S; ++u) load(u, wave + u * SK_NW);
  int u = 0;
  for (int ch = wave; ch < nc; ch += SK_NW) {
    constexpr int LEFT = (S - 1) * PER;   // requests of the later stages
    static_assert(LEFT < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (LEFT & 15) | ((LEFT >> 4) << 14));
    __builtin_amdgcn_sched_barrier(0);
    const char *sw = ring + u * PER * 1024, *sa = sw + R8 * 1024;
    bf16x8_t wf[2][NF], af[2][MT];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int r = 0; r < NF; ++r) wf[h][r] = as_frag(*reinterpret_cast<const u32x4_t*>(sw + swz(r * 16 + c, h * 4 + G)));
#pragma unroll
      for (int m = 0; m < MT; ++m) af[h][m] = as_frag(*reinterpret_cast<const u32x4_t*>(sa + swz(m * 16 + c, h * 4 + G)));
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < NF; ++r)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[r][m] = mfma16(wf[h][r], af[h][m], acc[r][m]);
    __builtin_amdgcn_s_waitcnt(0xC07F);   // the stage's fragments are in registers: it may be filled again
    __builtin_amdgcn_sched_barrier(0);
    load(u, ch + S * SK_NW);
    u = u + 1 == S ? 0 : u + 1;
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // no DMA may land in what becomes the sums' space
  __syncthreads();
  auto red = reinterpret_cast<f32x4_t(*)[NF * MT][64]>(gemm_smem);
#pragma unroll
  for (int r = 0; r < NF; ++r)
#pragma unroll
    for (int m = 0; m < MT; ++m) red[wave][r * MT + m][lane] = acc[r][m];
  __syncthreads();
  for (int i = wave; i < NF * MT; i += SK_NW) {
    auto total = [&](int l) {
      f32x4_t s = red[0][i][l];
#pragma unroll
      for (int w = 1; w < SK_NW; ++w) s += red[w][i][l];
      return s;
    };
    const int r = i / MT, m = (i - r * MT) * 16 + c;
    if (m >= a.M) continue;
    if constexpr (PAIRS) {   // rows 0-7 of a fragment: gate, 8-15: up
      if (G >= 2) continue;
      const f32x4_t g = total(lane), p = total(lane + 32);
      const float gt[4] = {g[0], g[1], g[2], g[3]}, up[4] = {p[0], p[1], p[2], p[3]};
      const int oc = ((int)blockIdx.x * (R8 / 2) + r) * 8 + G * 4;
      epi_pairs(a, m, 2 * oc, oc, gt, up);   // (oc < N / 2 decides)
    } else {
      const int local = r * 16 + G * 4, n = (int)blockIdx.x * (R8 * 8) + local;
      if (local >= R8 * 8) continue;   // (odd R8: half a fragment)
      const f32x4_t s = total(lane);
      auto epi = [&](auto act) {
        constexpr int ACT = decltype(act)::value;
        if (a.bias && a.residual) epi_group<ACT, true, true>(a, m, n, s[0], s[1], s[2], s[3]);
        else if (a.bias) epi_group<ACT, true, false>(a, m, n, s[0], s[1], s[2], s[3]);
        else if (a.residual) epi_group<ACT, false, true>(a, m, n, s[0], s[1], s[2], s[3]);
        else epi_group<ACT, false, false>(a, m, n, s[0], s[1], s[2], s[3]);
      };
      if (a.act == ACT_NONE) epi(std::integral_constant<int, ACT_NONE>{});
      else if (a.act == ACT_PARTIAL_F32) epi_group<ACT_PARTIAL_F32, false, false>(a, m, n, s[0], s[1], s[2], s[3]);
      else if (a.act == ACT_GELU_TANH) epi(std::integral_constant<int, ACT_GELU_TANH>{});
      else if (a.act == ACT_GELU_ERF) epi(std::integral_constant<int, ACT_GELU_ERF>{});
      else epi(std::integral_constant<int, ACT_SILU>{});
    }
  }
}

template <int R8, int M8, bool PAIRS>
void launch_one(const GemmArgs& a, hipStream_t st) {
  // three stages hide a request's latency; wide ones have enough in flight with two (and three of them leave one block per CU)
  constexpr int S = R8 + M8 <= 6 ? 3 : 2, PER = R8 + M8;
  constexpr int ring = SK_NW * S * PER * 1024 + 1024;   // (+ the half fragment that odd R8 or M8 reads behind the last stage)
  constexpr int red = SK_NW * ((R8 + 1) / 2) * ((M8 + 1) / 2) * 1024;
  constexpr int lds = ring > red ? ring : red;
  if (lds > 64 * 1024)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_skinny_kernel<R8, M8, S, PAIRS>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  hipLaunchKernelGGL((gemm_skinny_kernel<R8, M8, S, PAIRS>), dim3((unsigned)((a.N + R8 * 8 - 1) / (R8 * 8))), dim3(SK_NW * 64), lds, st, a);
}

template <int R8, bool PAIRS>
void launch_rows(const GemmArgs& a, hipStream_t st) {
  if (a.M <= 8) launch_one<R8, 1, PAIRS>(a, st);
  else if (a.M <= 16) launch_one<R8, 2, PAIRS>(a, st);
  else if (a.M <= 32) launch_one<R8, 4, PAIRS>(a, st);
  else launch_one<R8, 8, PAIRS>(a, st);
}

}  // namespace

// Weight rows per block / 8, and the estimated microseconds.  A block streams its weight rows and, from L2, A's rows (0.4 of the price per byte);
// a CU does ~30 bytes per ns of that mix, and launch, first request and the joined sums cost ~3 us (fitted to 8 .. 64 rows of the shapes above).
double gemm_skinny_plan(const GemmArgs& a, int* r8_out) {
  const int m8 = a.M <= 8 ? 1 : a.M <= 16 ? 2 : a.M <= 32 ? 4 : 8;
  double best = 1e30;
  for (int r8 : {2, 3, 4, 6}) {
    if (a.act == ACT_SILU_MUL_PAIRS && r8 == 3) continue;   // (gate and up rows in eights)
    const double rounds = ceil(((a.N + r8 * 8 - 1) / (r8 * 8)) / 256.0), c = 3.0 + rounds * (r8 + 0.4 * m8) * a.K * 16.0 / 30e3;
    if (c < best) {
      best = c;
      *r8_out = r8;
    }
  }
  return best;
}

bool gemm_skinny_ok(const GemmArgs& a) {
  return a.M >= 1 && a.M <= 64 && a.K >= 64 && a.K % 64 == 0 && a.N % 8 == 0 && a.groups == 1 && (a.act != ACT_SILU_MUL_PAIRS || a.N % 32 == 0);
}

void launch_gemm_skinny(const GemmArgs& a, hipStream_t st) {
  int r8 = 2;
  gemm_skinny_plan(a, &r8);
  if (a.act == ACT_SILU_MUL_PAIRS) {
    if (r8 == 2) launch_rows<2, true>(a, st);
    else if (r8 == 4) launch_rows<4, true>(a, st);
    else launch_rows<6, true>(a, st);
  } else {
    if (r8 == 2) launch_rows<2, false>(a, st);
    else if (r8 == 3) launch_rows<3, false>(a, st);
    else if (r8 == 4) launch_rows<4, false>(a, st);
    else launch_rows<6, false>(a, st);
  }
}

}  // namespace aha
