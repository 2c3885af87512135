// Matrix products of the layer-list decoders' 32-bit mode: C[M,N] f32 = A[M,K] f32 . W[N,K]^T, W bf16, optionally a batch of them (operands sa / sw / sc
// elements behind the first's).
//   gemm_f32_few_kernel   few rows: bound by the weights' stream (skinny_body.h)
//   gemm_f32_kernel       tiles of 16, 32 or 64 rows x 64 columns behind an LDS-DMA ring
//   gemm_f32_any_kernel   K or pitches that 16-byte pieces of 64-wide chunks do not divide, on v_mfma_f32_16x16x4_f32
// The first two multiply on the bf16 units without loss: W is bf16, and an f32 is the sum of three bf16 (split_bf16).  On v_mfma_f32_16x16x4_f32, the bound
// of both before, the same products took 5.3 times the matrix cycles, in more and shorter sums: error against 64 bits 5.7e-7 (K = 1024) and 1.0e-6 (3072) in
// tiles, 2.1e-7 and 3.3e-7 in few rows; now 1.0 to 1.9e-7 and 1.6 to 3.4e-7, 1.0e-7 and 1.6e-7.
#include <math.h>

#include <algorithm>

#include <type_traits>

#include "rows_common.h"
#include "skinny_body.h"

namespace aha {

namespace {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* glb_ptr_t;

struct GemmF32Args {
  const float* A;
  const bf16_t* W;
  float* C;
  int64_t lda, ldw, ldc, sa, sw, sc;
  int M, N, K;
};

// 2 / 32 rows back to back (in brackets: f32 MFMA): 4096 x 1024 4.5 / 5.7 us (4.7 / 6.5), 1024 x 2048 5.1 / 7.6 (6.2 / 9.2), 1024 x 3072 6.2 / 10.2 (8.1 / 12.4),
// 32768 x 1024 12.7 us (19.0): 5.3 TB/s of weights.
template <int R8, int M8>
__global__ __launch_bounds__(SKINNY_WAVES * 64) void gemm_f32_few_kernel(const float* A, const bf16_t* W, int M, int N, int K, int64_t lda, int64_t ldw, GemmF32Args a) {
  // (what the first requests need: in scalar registers at the start, gemv_body.h)
  a.A = A;
  a.W = W;
  a.M = M;
  a.N = N;
  a.K = K;
  a.lda = lda;
  a.ldw = ldw;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int MT = (M8 + 1) / 2, PER = skinny_requests(R8, M8, true);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), G = lane >> 4, c = lane & 15, n0 = (int)blockIdx.x * (R8 * 8);
  const char* src[PER];
#pragma unroll
  for (int r = 0; r < R8; ++r) {
    const int local = r * 8 + (lane >> 3);
    src[r] = (const char*)(a.W + (blockIdx.y > 0 ? blockIdx.y * a.sw : 0) + (int64_t)min(n0 + local, a.N - 1) * a.ldw) + skinny_piece(local, lane);
  }
#pragma unroll
  for (int r = 0; r < 2 * M8; ++r) {
    const int local = r % M8 * 8 + (lane >> 3);
    src[R8 + r] = (const char*)(a.A + (blockIdx.y > 0 ? blockIdx.y * a.sa : 0) + (int64_t)min(local, a.M - 1) * a.lda) + r / M8 * 128 + skinny_piece(local, lane);
  }
  skinny_sums<R8, M8, true>(src, a.K / 64, skinny_first(n0, a.K / 64), smem, wave, lane);
  for (int i = wave; i < (R8 / 2) * MT; i += SKINNY_WAVES) {
    const int f = i / MT, m = (i - f * MT) * 16 + c, n = n0 + f * 16 + G * 4;
    if (m < a.M && n < a.N) *reinterpret_cast<f32x4_t*>(a.C + blockIdx.y * a.sc + (int64_t)m * a.ldc + n) = skinny_total<R8, M8>(smem, i, lane);
  }
}

// WR * 16 rows x 64 columns, WR * WK waves of 16 x 64: WR side by side over the rows, WK over the 64-wide k chunks of a stage (their sums are joined at the
// end).  A stage is requests of 1 KB: per chunk 4 WR of A (rows of 64 k of A are two lines) and 8 of W.  The fragments of a stage are read whole before the next
// requests go out.
// A wave's chunk is 88 instructions of splitting and 24 MFMAs, ~0.42 us, its stage's bytes ~0.35 us: with one wave per SIMD a launch takes their sum times the
// chunks of its longest wave, however few blocks it has.  So the k chunks are dealt to WK waves where blocks are few; four chunks of 16 rows as long as one block
// per CU does it, then 32 rows, of four chunks for one block per CU and of two for two, then 64 rows of one (launch_gemm_f32).  us (in brackets: the tiles of 16
// or 32 rows on the f32 MFMA), 252 rows: 4096 x 1024 11.8 (26.2), 1024 x 2048 10.0 (19.3), 3072 x 1024 9.7 (20.2), 1024 x 3072 13.4 (28.1), 6176 x 1024 17.5 (48.4);
// 66 rows: 7.5 (14.6), 9.1 (18.5), 6.6 (11.0), 11.8 (26.7), 10.5 (15.6); 1000 rows: 35 (93), 20 (48), 27.5 (71), 26.1 (75.6), 61 (144).
// The other shapes at 252 rows, 16 rows x 4 chunks / 32 x 4 / 32 x 2 / 64 x 1: 4096 x 1024 22 / 15.3 / 11.8 / 12.0, 1024 x 2048 10.0 / 10.8 / 12.7 / 19.2.
// Fragments a stage ahead in registers: no difference; 32 rows per wave: slower (a wave's chunk takes twice as long).
constexpr int f_stage(int rows, int wk) { return (rows / 4 + 8) * wk * 1024; }
template <int WR, int WK, int F_S>
__global__ __launch_bounds__(WR * WK * 64) void gemm_f32_kernel(GemmF32Args a, int tiles_m) {
  extern __shared__ __attribute__((aligned(16))) char smem[];   // F_S x [A: chunks x halves x rows | W: chunks x 64 rows]
  constexpr int ROWS = WR * 16, STAGE = f_stage(ROWS, WK), HALF = ROWS * 128, NA = ROWS / 4 * WK, QA = 4, NW = 8 / WR, LEFT = (F_S - 2) * (QA + NW);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), G = lane >> 4, c = lane & 15, wr = wave % WR, wk = wave / WR;
  // the row tiles of a column tile stay on one XCD: its weights leave HBM once
  const int xcd = (int)blockIdx.x & 7, local = (int)blockIdx.x >> 3, n0 = (local / tiles_m * 8 + xcd) * 64, m0 = local % tiles_m * ROWS;
  if (n0 >= a.N) return;
  const float* A = a.A + blockIdx.z * a.sa;
  const bf16_t* W = a.W + blockIdx.z * a.sw;
  const int nc = a.K / 64, nk = (nc + WK - 1) / WK;
  const char *asrc[QA], *wsrc[NW];   // requests wave * QA + j of A, wave * NW + j of W
#pragma unroll
  for (int j = 0; j < QA; ++j) {
    const int q = wave * QA + j, ar = q % (ROWS / 8) * 8 + (lane >> 3);
    asrc[j] = (const char*)(A + (int64_t)min(m0 + ar, a.M - 1) * a.lda) + q % (ROWS / 4) / (ROWS / 8) * 128 + skinny_piece(ar, lane);
  }
#pragma unroll
  for (int j = 0; j < NW; ++j) {
    const int wrow = (wave * NW + j) % 8 * 8 + (lane >> 3);
    wsrc[j] = (const char*)(W + (int64_t)min(n0 + wrow, a.N - 1) * a.ldw) + skinny_piece(wrow, lane);
  }
  auto load = [&](int kt) {   // (past the end: the last chunk again, never used)
    char* st = smem + kt % F_S * STAGE;
#pragma unroll
    for (int j = 0; j < QA; ++j) {
      const int q = wave * QA + j;
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(asrc[j] + min(kt * WK + q / (ROWS / 4), nc - 1) * 256), (lds_ptr_t)(st + q * 1024), 16, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      const int q = wave * NW + j;
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(wsrc[j] + min(kt * WK + q / 8, nc - 1) * 128), (lds_ptr_t)(st + (NA + q) * 1024), 16, 0, 0);
    }
  };
  f32x4_t big[4], rest[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) big[r] = rest[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < F_S - 1; ++s) load(s);
  for (int kt = 0; kt < nk; ++kt) {
    __builtin_amdgcn_s_waitcnt(0x0F70 | (LEFT & 15) | ((LEFT >> 4) << 14));   // this wave's part of stage kt is in; behind the barrier everyone's, and stage kt - 1 is read
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const char *sa = smem + kt % F_S * STAGE + wk * (ROWS / 4 * 1024), *sw = smem + kt % F_S * STAGE + (NA + wk * 8) * 1024;
    f32x4_t x[2][2];
    bf16x8_t wf[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int q = 0; q < 2; ++q) x[h][q] = *reinterpret_cast<const f32x4_t*>(sa + h * HALF + skinny_swz(wr * 16 + c, 2 * G + q));
#pragma unroll
      for (int r = 0; r < 4; ++r) wf[h][r] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(sw + skinny_swz(r * 16 + c, h * 4 + G)));
    }
    __builtin_amdgcn_sched_barrier(0);
    load(kt + F_S - 1);
    __builtin_amdgcn_sched_barrier(0);
    if (WK == 1 || kt * WK + wk < nc) {   // (K / 64 no multiple of WK: the last stage lacks a chunk)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const SplitBf16x8 p = split_bf16(x[h][0], x[h][1]);
#pragma unroll
        for (int r = 0; r < 4; ++r) big[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][r], p.hi, big[r], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) rest[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][r], p.lo, rest[r], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) rest[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][r], p.mid, rest[r], 0, 0, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // (the surplus requests: LDS may belong to the next block, or to the sums)
  f32x4_t sum[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) sum[r] = split_sum(big[r], rest[r]);
  if constexpr (WK > 1) {   // wave wk = 0 of a row group adds the others' sums in their order
    __syncthreads();
    auto red = reinterpret_cast<f32x4_t(*)[4][64]>(smem);
    if (wk > 0)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave - WR][r][lane] = sum[r];
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int w = 1; w < WK; ++w)
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[r] += red[(w - 1) * WR + wr][r][lane];
  }
  const int m = m0 + wr * 16 + c;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = n0 + r * 16 + G * 4;
    if (m < a.M && n < a.N) *reinterpret_cast<f32x4_t*>(a.C + blockIdx.z * a.sc + (int64_t)m * a.ldc + n) = sum[r];
  }
}

// any K and pitches: 64 x 64 tile, four waves of 16 x 64 on v_mfma_f32_16x16x4_f32 (lane l: row / column l & 15, k = l >> 4)
constexpr int FBK = 32, FPITCH = FBK + 1;
// (blockIdx.z: one of a batch of products, its operands sa / sw / sc elements behind the first's)
__global__ __launch_bounds__(256) void gemm_f32_any_kernel(const float* __restrict__ A, int64_t lda, const bf16_t* __restrict__ W, int64_t ldw,
                                                      float* __restrict__ C, int64_t ldc, int M, int N, int K, int64_t sa, int64_t sw, int64_t sc) {
  A += blockIdx.z * sa;
  W += blockIdx.z * sw;
  C += blockIdx.z * sc;
  __shared__ float as[64 * FPITCH], ws[64 * FPITCH];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, G = lane >> 4;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  f32x4_t acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += FBK) {
#pragma unroll
    for (int i = 0; i < 64 * FBK / 4 / 256; ++i) {
      const int p = tid + i * 256, row = p >> 3, kk = (p & 7) * 4;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f), w = v;
      if (m0 + row < M) v = *reinterpret_cast<const float4*>(A + (int64_t)(m0 + row) * lda + k0 + kk);
      if (n0 + row < N) w = wbf4(W, (int64_t)(n0 + row) * ldw + k0 + kk);
      float *da = as + row * FPITCH + kk, *dw = ws + row * FPITCH + kk;
      da[0] = v.x; da[1] = v.y; da[2] = v.z; da[3] = v.w;
      dw[0] = w.x; dw[1] = w.y; dw[2] = w.z; dw[3] = w.w;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < FBK; k += 4) {
      const float av = as[(wave * 16 + c) * FPITCH + k + G];
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, ws[(j * 16 + c) * FPITCH + k + G], acc[j], 0, 0, 0);
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + j * 16 + c;
    if (n >= N) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + wave * 16 + G * 4 + r;
      if (m < M) C[(int64_t)m * ldc + n] = acc[j][r];
    }
  }
}

}  // namespace

void launch_gemm_f32(const float* A, int64_t lda, const void* W, int64_t ldw, float* C, int64_t ldc, int M, int N, int K, hipStream_t st, int batch,
                     int64_t sa, int64_t sw, int64_t sc) {
  if (M <= 0 || N <= 0 || batch <= 0) return;
  const GemmF32Args a{A, (const bf16_t*)W, C, lda, ldw, ldc, sa, sw, sc, M, N, K};
  const bool pieces = K >= 64 && K % 64 == 0 && ((N | lda | ldc | sa | sc) & 3) == 0 && ((ldw | sw) & 7) == 0 && (((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) & 15) == 0;
  if (!pieces) {
    hipLaunchKernelGGL(gemm_f32_any_kernel, dim3((unsigned)((N + 63) / 64), (unsigned)((M + 63) / 64), (unsigned)batch), dim3(256), 0, st, A, lda, (const bf16_t*)W,
                       ldw, C, ldc, M, N, K, sa, sw, sc);
    return;
  }
  using std::integral_constant;
  // the few-row form: 48 weight rows per block where they still make two blocks per CU (the head), up to 16 rows
  // (32768 x 1024 at 32 rows: 23 us, in tiles 15.4); else 16.  From 33 rows on the tiles are ahead (64 rows, 4096 x 1024: 9.7 / 7.2, 1024 x 3072: 17.7 / 12.4)
  const bool wide = (int64_t)((N + 47) / 48) * batch >= 512;
  if (M > 32 || (M > 16 && wide)) {
    auto tiles = [&](auto wr, auto wk, auto stages) {
      constexpr int WR = decltype(wr)::value, WK = decltype(wk)::value, S = decltype(stages)::value, lds = S * f_stage(WR * 16, WK);
      auto k = gemm_f32_kernel<WR, WK, S>;
      if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      const int tm = (M + WR * 16 - 1) / (WR * 16), tn = ((N + 63) / 64 + 7) / 8 * 8;
      hipLaunchKernelGGL(k, dim3((unsigned)(tm * tn), 1, (unsigned)batch), dim3(WR * WK * 64), lds, st, a, tm);
    };
    const int64_t cols = (int64_t)((N + 63) / 64) * batch, b16 = (M + 15) / 16 * cols, b32 = (M + 31) / 32 * cols;   // (kernel's comment)
    if (b16 <= 256) tiles(integral_constant<int, 1>{}, integral_constant<int, 4>{}, integral_constant<int, 3>{});
    else if (b32 <= 256) tiles(integral_constant<int, 2>{}, integral_constant<int, 4>{}, integral_constant<int, 2>{});
    else if (b32 <= 512) tiles(integral_constant<int, 2>{}, integral_constant<int, 2>{}, integral_constant<int, 2>{});
    else tiles(integral_constant<int, 4>{}, integral_constant<int, 1>{}, integral_constant<int, 3>{});
    return;
  }
  auto go = [&](auto r8, auto m8) {
    constexpr int R8 = decltype(r8)::value, M8 = decltype(m8)::value, lds = skinny_lds(R8, M8, true);
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_f32_few_kernel<R8, M8>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    hipLaunchKernelGGL((gemm_f32_few_kernel<R8, M8>), dim3((unsigned)((N + R8 * 8 - 1) / (R8 * 8)), (unsigned)batch), dim3(SKINNY_WAVES * 64), lds, st, a.A,
                       a.W, a.M, a.N, a.K, a.lda, a.ldw, a);
  };
  if (M <= 8) wide ? go(integral_constant<int, 6>{}, integral_constant<int, 1>{}) : go(integral_constant<int, 2>{}, integral_constant<int, 1>{});
  else if (M <= 16) wide ? go(integral_constant<int, 6>{}, integral_constant<int, 2>{}) : go(integral_constant<int, 2>{}, integral_constant<int, 2>{});
  else go(integral_constant<int, 2>{}, integral_constant<int, 4>{});
}

}  // namespace aha
