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
// Up to 64 rows blocks start at different k (skinny_first; row tiles of more rows: no difference in time, and they keep the common start).  The start is a
// rotation of the sum's order, by the weight row in the matrix that the call is given and from K = 2048 on.  So an element is the same sum in a call of 1 to 64 rows and
// another in one of 65 to 256, as it already is where the tiles take over; and a tensor-parallel rank's columns (a matrix of its own, its rows counted from the shard's
// first) are summed in another order than the whole matrix' -- the same rounding, not the same bits.  Row-parallel blocks, cut into columns or not by how
// the collective overlaps, keep the common start (GemmArgs::few_rows_spread).
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

template <int R8, int M8, bool PAIRS, bool DEEP, typename PRO, typename EPI>
__device__ __forceinline__ void skinny_product(const void* A, const void* W, int M, int N, int K, int spread, int64_t lda, int64_t ldw, GemmArgs& a, PRO pro, EPI epilogue) {
  // What the first requests need: in scalar registers at the start (gemv_body.h).  `spread` too: read from `a` in memory it put 0.25 to 0.35 us in front of
  // every product's first request (8 rows: 3072 x 1024 3.33 us, 3.59 so).
  a.A = A;
  a.W = W;
  a.M = M;
  a.N = N;
  a.K = K;
  a.lda = lda;
  a.ldw = ldw;
  constexpr int PER = R8 + M8;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
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
  skinny_sums<R8, M8, false, DEEP>(src, a.K / 64, spread ? skinny_first((int)blockIdx.x * (R8 * 8), K / 64) : 0, gemm_smem, wave, lane, pro);
  epilogue(wave, lane);
}


template <int R8, int M8, bool PAIRS, bool DEEP>
__global__ __launch_bounds__(SKINNY_WAVES * 64) void gemm_skinny_kernel(const void* A, const void* W, int M, int N, int K, int spread, int64_t lda, int64_t ldw, GemmArgs a) {
  skinny_product<R8, M8, PAIRS, DEEP>(A, W, M, N, K, spread, lda, ldw, a, SkinnyPlain{}, [&](int wave, int lane) {
    constexpr int NF = (R8 + 1) / 2, MT = (M8 + 1) / 2;
    const int G = lane >> 4, c = lane & 15;
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
  });
}

// ---- PolyNorm between two few-row products ------------------------------------------------------------------------------------------------
// A launch of its own between an up and a down projection of up to 16 rows is a link of the chain like any other, for 8 x 12288 numbers (4.9 us).  Here the
// first product leaves, beside its bf16 result z, the sums of z^2, z^4 and z^6 over each block's columns, [block][M8 * 8 rows]; the second joins them while its
// first stages are on their way and maps the fragments that it reads from LDS: three fma and a rounding per number, under the wait for the weights.
// 8 rows, 12288 x 4096 and back: 39.3 us in three launches, 38.0 in two (gemm_takes_poly: where it pays); 12 layers of 8B sizes, 8 requests and 32 steps 39.0 -> 38.0 ms.
// The sums' place and number come with the launch, as all that stands in front of the first requests.
constexpr int POLY_PARTS = 256;   // blocks of the first product, at most
template <int M8>
struct SkinnyPolyIn {   // stats, parts: from the leading arguments (skinny_product)
  static constexpr bool ON = true;
  static constexpr int R = M8 * 8, PER = 64 / R, NL = POLY_PARTS / (PER * SKINNY_WAVES);
  static_assert(M8 == 1 || M8 == 2, "one activation fragment");
  const SkinnyPoly& p;
  const float* stats;
  int parts;
  f32x4_t (*red)[16];   // [SKINNY_WAVES]
  f32x4_t v[NL];
  float r1 = 0.f, r2 = 0.f, r3 = 0.f, e = 0.f;
  __device__ __forceinline__ SkinnyPolyIn(const SkinnyPoly& p_, const float* stats_, int parts_, f32x4_t (*red_)[16]) : p(p_), stats(stats_), parts(parts_), red(red_) {}
  __device__ __forceinline__ int part(int j) const { return (j * SKINNY_WAVES + (int)(threadIdx.x >> 6)) * PER + (int)(threadIdx.x & 63) / R; }
  __device__ __forceinline__ void request() {
    const f32x4_t* at = reinterpret_cast<const f32x4_t*>(stats) + (threadIdx.x & (R - 1));
#pragma unroll
    for (int j = 0; j < NL; ++j) v[j] = at[min(part(j), parts - 1) * R];
  }
  __device__ __forceinline__ void join() {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    f32x4_t mine = {0.f, 0.f, 0.f, 0.f};   // (all four, though the last is nothing: a loaded register that nobody reads is taken for something else, behind a wait for its load)
#pragma unroll
    for (int j = 0; j < NL; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) mine[i] += part(j) < parts ? v[j][i] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (R == 8) mine[i] += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(mine[i]), 0x128 /* row_ror:8 */, 0xf, 0xf, false));
      mine[i] = rows_sum(mine[i]);
    }
    // The waves' sums meet in LDS by hand: what the compiler knows to touch LDS it lets wait for every stage on its way (and __syncthreads with it).
    typedef __attribute__((address_space(3))) f32x4_t* lds_t;
    const uint32_t at = (uint32_t)(uintptr_t)(lds_t)&red[0][lane & 15];
    f32x4_t w0, w1, w2, w3;
    asm volatile("ds_write_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::"v"(at + wave * 256), "v"(mine) : "memory");   // (the four lanes of one lane & 15: the same)
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:256\n\tds_read_b128 %2, %4 offset:512\n\tds_read_b128 %3, %4 offset:768\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(w0), "=&v"(w1), "=&v"(w2), "=&v"(w3)
                 : "v"(at)
                 : "memory");
    const f32x4_t t = (w0 + w1) + (w2 + w3);
    r1 = p.coef[0] / sqrtf(t[0] * p.inv_ff + p.eps);
    r2 = p.coef[1] / sqrtf(t[1] * p.inv_ff + p.eps);
    r3 = p.coef[2] / sqrtf(t[2] * p.inv_ff + p.eps);
    e = p.coef[3];
  }
  __device__ __forceinline__ u32x4_t map(u32x4_t x) const {   // (pad columns become e: their weights are zero)
    u32x4_t o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float lo = lo_bf(x[i]), hi = hi_bf(x[i]);
      o[i] = pack_bf(fmaf(lo, fmaf(lo, fmaf(lo, r3, r2), r1), e), fmaf(hi, fmaf(hi, fmaf(hi, r3, r2), r1), e));
    }
    return o;
  }
};
// IN: the second product, else the first.  bf16 results, no bias, residual or activation.
template <int R8, int M8, bool DEEP, bool IN>
__global__ __launch_bounds__(SKINNY_WAVES * 64) __attribute__((amdgpu_waves_per_eu(1, 4))) void gemm_skinny_poly_kernel(const void* A, const void* W, int M, int N, int K, int parts_spread, int64_t lda, int64_t ldw, float* stats, SkinnyPoly p, GemmArgs a) {
  const int spread = parts_spread & 1;
  constexpr int NF = (R8 + 1) / 2, R = M8 * 8;
  __shared__ f32x4_t red[SKINNY_WAVES][16];
  auto epilogue = [&](int wave, int lane) {
    const int G = lane >> 4, c = lane & 15, local = wave * 16 + G * 4, n = (int)blockIdx.x * (R8 * 8) + local;
    float t[3] = {0.f, 0.f, 0.f};
    if (wave < NF) {
      const f32x4_t s = skinny_total<R8, M8>(gemm_smem, wave, lane);
      if (local < R8 * 8) {   // (odd R8: half a fragment)
        if (c < a.M) epi_group<ACT_NONE, false, false>(a, c, n, s[0], s[1], s[2], s[3]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float z = n + j < a.N ? bf2f(f2bf(s[j])) : 0.f, z2 = z * z, z4 = z2 * z2;
          t[0] += z2;
          t[1] += z4;
          t[2] = fmaf(z4, z2, t[2]);
        }
      }
    }
    if constexpr (!IN) {   // (rows past M: the last one's again)
      if (wave < NF) {
#pragma unroll
        for (int i = 0; i < 3; ++i) t[i] = rows_sum(t[i]);
        if (G == 0) red[wave][c] = f32x4_t{t[0], t[1], t[2], 0.f};
      }
      __syncthreads();
      if (threadIdx.x < R) {
        f32x4_t v = red[0][threadIdx.x];
#pragma unroll
        for (int r = 1; r < NF; ++r) v += red[r][threadIdx.x];
        reinterpret_cast<f32x4_t*>(stats)[blockIdx.x * R + threadIdx.x] = v;
      }
    }
  };
  if constexpr (IN) skinny_product<R8, M8, false, DEEP>(A, W, M, N, K, spread, lda, ldw, a, SkinnyPolyIn<M8>(p, stats, parts_spread >> 1, red), epilogue);
  else skinny_product<R8, M8, false, DEEP>(A, W, M, N, K, spread, lda, ldw, a, SkinnyPlain{}, epilogue);
}

int skinny_spread(const GemmArgs& a) { return a.few_rows_spread && a.M <= 64; }

template <int R8, int M8, bool PAIRS, bool DEEP = false>
void launch_one(const GemmArgs& a, hipStream_t st) {
  if constexpr (!DEEP && skinny_stages(R8 + M8) != skinny_stages(R8 + M8, true))
    if (gemm_skinny_rounds(a, R8) == 1) return launch_one<R8, M8, PAIRS, true>(a, st);
  constexpr int lds = skinny_lds(R8, M8, false, DEEP);
  if (lds > 64 * 1024)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_skinny_kernel<R8, M8, PAIRS, DEEP>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  hipLaunchKernelGGL((gemm_skinny_kernel<R8, M8, PAIRS, DEEP>), dim3((unsigned)((a.N + R8 * 8 - 1) / (R8 * 8)), (unsigned)((a.M + 63) / 64)), dim3(SKINNY_WAVES * 64), lds, st, a.A, a.W, a.M, a.N, a.K, skinny_spread(a),
                     a.lda, a.ldw, a);
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

namespace {

template <int R8, int M8, bool IN, bool DEEP = false>
void launch_poly_one(const GemmArgs& a, const SkinnyPoly& p, hipStream_t st) {
  if constexpr (!DEEP && skinny_stages(R8 + M8) != skinny_stages(R8 + M8, true))
    if (gemm_skinny_rounds(a, R8) == 1) return launch_poly_one<R8, M8, IN, true>(a, p, st);
  constexpr int lds = skinny_lds(R8, M8, false, DEEP);
  auto k = gemm_skinny_poly_kernel<R8, M8, DEEP, IN>;
  if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  hipLaunchKernelGGL(k, dim3((unsigned)((a.N + R8 * 8 - 1) / (R8 * 8))), dim3(SKINNY_WAVES * 64), lds, st, a.A, a.W, a.M, a.N, a.K, p.parts << 1 | skinny_spread(a), a.lda, a.ldw, p.stats, p, a);
}

template <bool IN>
void launch_poly(const GemmArgs& a, const SkinnyPoly& p, int r8, hipStream_t st) {
  auto go = [&](auto r) {
    if (a.M <= 8) launch_poly_one<decltype(r)::value, 1, IN>(a, p, st);
    else launch_poly_one<decltype(r)::value, 2, IN>(a, p, st);
  };
  if (r8 == 2) go(std::integral_constant<int, 2>{});
  else if (r8 == 3) go(std::integral_constant<int, 3>{});
  else if (IN || r8 == 4) go(std::integral_constant<int, 4>{});
  else if constexpr (!IN) go(std::integral_constant<int, 6>{});
}

}  // namespace

// K of 24 chunks and more: the deepest ring's first requests (skinny_sums).  A second product of 48 weight rows per block has more than 8192 columns, the
// widest that a layer list can be.
bool gemm_skinny_poly_ok(const GemmArgs& up, const GemmArgs& down) {
  if (up.M > 16 || down.M != up.M || down.K != up.N || down.K < 24 * 64) return false;
  int r8 = 2;
  gemm_skinny_plan(down, &r8);
  if (r8 > 4) return false;
  gemm_skinny_plan(up, &r8);
  return (up.N + r8 * 8 - 1) / (r8 * 8) <= POLY_PARTS;
}
size_t gemm_skinny_poly_floats() { return (size_t)POLY_PARTS * 16 * 4; }

void launch_gemm_skinny_poly(const GemmArgs& up, const GemmArgs& down, SkinnyPoly p, hipStream_t st) {
  int r8 = 2;
  gemm_skinny_plan(up, &r8);
  p.parts = (up.N + r8 * 8 - 1) / (r8 * 8);
  launch_poly<false>(up, p, r8, st);
  gemm_skinny_plan(down, &r8);
  launch_poly<true>(down, p, r8, st);
}

}  // namespace aha
