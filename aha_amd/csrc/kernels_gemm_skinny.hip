// Projection GEMM for few rows (M <= 64: batched decode steps, short prompts; to 256 where row tiles of 64 fit into one round): C[M,N] = A[M,K] . W[N,K]^T with the epilogues of kernels_gemm.hip.
//
// What bounds it is the weight matrix, read once from HBM; the 128-row tiles of kernels_gemm.hip stage 16 times the rows a batch of eight has and
// need K slices and a reduce pass to fill the chip.  Here a block owns R8 * 8 weight rows and the whole K range, its four waves take the 64-wide
// k chunks in turn, and every wave has a ring of S chunks of its own in LDS that it fills by DMA and drains by itself: no barrier before the sums
// of the four waves are joined, two to six stages of 3 KB to 14 KB in flight per wave (skinny_stages).  A DMA request covers eight rows x 128 bytes (whole lines);
// operands that waves load to registers themselves as MFMA fragments touch 16 rows x 64 bytes per request and ran at half the rate (6144 x 4096,
// 8 rows: 17.5 us against 10.4 us).  A's rows go the same way: each block reads all of A, so blocks have as many weight rows as one round over
// the chip allows (gemm_skinny_plan).
// Rows past M, N repeat the last one, lanes of a fragment that no row backs another row; what they give is not stored: an MFMA's output rows and columns
// do not mix.
//
// Up to 64 rows blocks start at different k (skinny_first; row tiles of more rows: no difference, and they keep the common start).
//
// Measured on MI355X, back to back from HBM, 8 rows (in brackets: the split-K ring kernel + its reduce pass it replaces, inside a batched step):
//   6144 x 4096 9.9 us (5.1 TB/s), 4096 x 4096 7.2, 12288 x 4096 17.0 (5.9), 4096 x 12288 16.9 (6.0), 24576 x 4096 31.4 (6.4)
//   [18.1 + 4.6 us on average over the first four]; 32 rows: 11.8, 9.6, 18.1, 25.1, 33.0; 64 rows: 15.7, 13.1, 22.4, 35.3, 43.8
//   64-row tiles, 96 / 128 rows (tiled kernels with their reduce pass): 4096 x 1024 6.2 / 6.4 us (10.7 / 10.7), 6144 x 1024 8.1 / 8.3 (12.1 / 12.9),
//   1024 x 2048 6.6 / 7.1 (11.3 / 12.1), 1024 x 3072 8.7 / 9.7 (12.3 / 13.2); a 0.6B prompt of 96 / 128 / 180 / 250 tokens 1.66 / 1.67 / 1.95 / 2.03 ms
//   (1.97 / 2.06 / 2.07 / 2.14), of 300 2.14 (2.09): 256 rows at most.  The 8B shapes stay on the tiles:
//   their weight rows need more than one round or a longer K than a block streams in the tiles' time (6144 x 4096, 96 rows: 21.3 against 21.0).
#include <algorithm>

#include "gemm256_body.h"
#include "skinny_body.h"

namespace aha {

namespace {

template <int R8, int M8, bool PAIRS, bool DEEP>
__global__ __launch_bounds__(SKINNY_WAVES * 64) void gemm_skinny_kernel(const void* A, const void* W, int M, int N, int K, int64_t lda, int64_t ldw, GemmArgs a) {
  // (what the first requests need: in scalar registers at the start, gemv_body.h)
  a.A = A;
  a.W = W;
  a.M = M;
  a.N = N;
  a.K = K;
  a.lda = lda;
  a.ldw = ldw;
  constexpr int NF = (R8 + 1) / 2, MT = (M8 + 1) / 2, PER = R8 + M8;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), G = lane >> 4, c = lane & 15;
  const char* src[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int local = (r < R8 ? r : r - R8) * 8 + (lane >> 3), piece = skinny_piece(local, lane);
    if (r >= R8) {
      src[r] = (const char*)a.A + (int64_t)min((int)blockIdx.y * 64 + local, a.M - 1) * a.lda * 2 + piece;
    } else if (PAIRS) {   // eight gate rows, then the eight up rows of the same columns (16-row blocks alternate in W)
      const int col = ((int)blockIdx.x * (R8 / 2) + r / 2) * 8 + (lane >> 3);
      src[r] = (const char*)a.W + (int64_t)min((col >> 4) * 32 + (r & 1) * 16 + (col & 15), a.N - 1) * a.ldw * 2 + piece;
    } else {
      src[r] = (const char*)a.W + (int64_t)min((int)blockIdx.x * (R8 * 8) + local, a.N - 1) * a.ldw * 2 + piece;
    }
  }
  skinny_sums<R8, M8, false, DEEP>(src, a.K / 64, a.few_rows_spread && a.M <= 64 ? skinny_first((int)blockIdx.x * (R8 * 8), a.K / 64) : 0, gemm_smem, wave, lane);
  for (int i = wave; i < NF * MT; i += SKINNY_WAVES) {
    const int r = i / MT, m = (int)blockIdx.y * 64 + (i - r * MT) * 16 + c;
    if (m >= a.M) continue;
    if constexpr (PAIRS) {   // rows 0-7 of a fragment: gate, 8-15: up
      if (G >= 2) continue;
      const f32x4_t g = skinny_total<R8, M8>(gemm_smem, i, lane), p = skinny_total<R8, M8>(gemm_smem, i, lane + 32);
      const float gt[4] = {g[0], g[1], g[2], g[3]}, up[4] = {p[0], p[1], p[2], p[3]};
      const int oc = ((int)blockIdx.x * (R8 / 2) + r) * 8 + G * 4;
      epi_pairs(a, m, 2 * oc, oc, gt, up);   // (oc < N / 2 decides)
    } else {
      const int local = r * 16 + G * 4, n = (int)blockIdx.x * (R8 * 8) + local;
      if (local >= R8 * 8) continue;   // (odd R8: half a fragment)
      const f32x4_t s = skinny_total<R8, M8>(gemm_smem, i, lane);
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

template <int R8, int M8, bool PAIRS, bool DEEP = false>
void launch_one(const GemmArgs& a, hipStream_t st) {
  if constexpr (!DEEP && skinny_stages(R8 + M8) != skinny_stages(R8 + M8, true))
    if (gemm_skinny_rounds(a, R8) == 1) return launch_one<R8, M8, PAIRS, true>(a, st);
  constexpr int lds = skinny_lds(R8, M8, false, DEEP);
  if (lds > 64 * 1024)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_skinny_kernel<R8, M8, PAIRS, DEEP>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  hipLaunchKernelGGL((gemm_skinny_kernel<R8, M8, PAIRS, DEEP>), dim3((unsigned)((a.N + R8 * 8 - 1) / (R8 * 8)), (unsigned)((a.M + 63) / 64)), dim3(SKINNY_WAVES * 64), lds, st, a.A, a.W, a.M, a.N, a.K, a.lda,
                     a.ldw, a);
}

template <int R8, bool PAIRS>
void launch_rows(const GemmArgs& a, hipStream_t st) {
  if (a.M <= 8) launch_one<R8, 1, PAIRS>(a, st);
  else if (a.M <= 16) launch_one<R8, 2, PAIRS>(a, st);
  else if (a.M <= 32) launch_one<R8, 4, PAIRS>(a, st);
  else launch_one<R8, 8, PAIRS>(a, st);
}

}  // namespace

int gemm_skinny_rounds(const GemmArgs& a, int r8) { return ((a.N + r8 * 8 - 1) / (r8 * 8) * ((a.M + 63) / 64) + 255) / 256; }

// Weight rows per block / 8, and the estimated microseconds.  One round (a block per CU): a block streams its weight rows and, from L2, A's rows (0.4 of
// the price per byte); a CU does ~30 bytes per ns of that mix, and launch, first request and the joined sums cost ~3 us (fitted to 8 .. 64 rows of the
// shapes above).
// More rounds, up to 64 rows (4096 x 1024, 180 rows, 384 blocks: 12.0 us against 10.9 of the tiles): a CU requests at most 60 bytes of weights per ns and
// the chip delivers at most 8.2 TB/s (32 rows per block that lie whole 256 KB apart: 1.34 times as long, their requests meet in the same channels),
// rounded where the two meet; A's rows at 96 bytes per ns and CU, the last row's repetitions for nothing; a block's first requests and the joined sums
// show where no neighbour on the CU covers them.  Fitted to 23 shapes (512 x 4096 to 151936 x 4096) at 1 to 64 rows with every R8, before the blocks started
// at different k; it is 7 % dear on average since, and 32 rows 256 KB apart are only 10 % slower than others.  The width chosen with it is at most 5 % behind the
// best of the four at 20 shapes (1024 x 2048 to 151936 x 1024) with 3 to 64 rows, but for 16384 x 4096 at 16 and more (26.2 us, 21.7 with 32 weight rows), 6208 x
// 4096 at 8 (10.9, 9.9 with 32) and 32768 x 1024 at 3 (12.8, 11.6 with 16); with 1.1 for 1.34 48 rows of 16384 x 4096 leave the tiles.
// The price of one round times their number said 41 us with 32 rows per block for 32768 x 4096 and 8 rows (57.7; 42.6 with 48) and 76 us for
// 151936 x 1024 and 64 rows (96.6; the tiles 73).
double gemm_skinny_plan(const GemmArgs& a, int* r8_out) {
  const int m8 = a.M <= 8 ? 1 : a.M <= 16 ? 2 : a.M <= 32 ? 4 : 8;
  const double chunk = a.K * 16.0;   // bytes of eight rows
  double best = 1e30;
  for (int r8 : {2, 3, 4, 6}) {
    if (a.act == ACT_SILU_MUL_PAIRS && r8 == 3) continue;   // (gate and up rows in eights)
    const int rounds = gemm_skinny_rounds(a, r8);
    double c = 3.0 + (r8 + 0.4 * m8) * chunk / 30e3;
    if (rounds > 1) {
      if (a.M > 64) continue;
      const int resident = std::min(4, skinny_blocks(r8, m8)), rows8 = (a.M + 7) / 8;
      const double cu = rounds * r8 * chunk / 60e3, chip = a.N / 8 * chunk / 8.2e6 * (r8 == 4 && a.ldw * 64 % (256 << 10) == 0 ? 1.34 : 1.0);
      c = 3.5 + sqrt(cu * cu + chip * chip) + rounds * rows8 * chunk / 96e3 + ((rounds + resident - 1) / resident - 1) * 0.25 * rows8 + 0.075 * rounds * m8;
    }
    if (c < best) {
      best = c;
      *r8_out = r8;
    }
  }
  return best;
}

// K < 768 stays with the tiled kernels: they run unsplit there, so a row's bits do not depend on how many rows share the call (row slices of a
// sequence-parallel prompt), for 1.5 to 4 us more per launch (K = 256: 5.1 against 2.7 us, 512: 6.8 against 3.0, 768: 8.5 against 3.3; 8 rows, 2048
// columns).  So do 33 to 64 rows of a matrix below 2 MB (512 x 1024: 10.2 against 5.2 us) and more rows of one below 4 MB.  Only small models have either -- the full-size ones have
// K >= 768 throughout their text stacks, and their one small matrix, the router, is met by 33 to 64 rows only in that band -- and they keep the
// results they had.
// few_rows = 2: a column block of a projection that takes this kernel as a whole, whatever the block's own size (an element's sum has the same order for
// every R8 and M8).
bool gemm_skinny_ok(const GemmArgs& a) {
  return a.few_rows && a.M >= 1 && a.M <= 256 && a.K >= 768 && a.K % 64 == 0 && a.N % 8 == 0 && a.groups == 1 && (a.act != ACT_SILU_MUL_PAIRS || a.N % 32 == 0) &&
         (a.few_rows == 2 || a.M <= 32 || (int64_t)a.N * a.K >= (a.M <= 64 ? 1 << 20 : 1 << 21));
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
