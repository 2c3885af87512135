// Matrix products of the layer-list decoders' 32-bit mode: C[M,N] f32 = A[M,K] f32 . W[N,K]^T, W bf16 (widened exactly), on v_mfma_f32_16x16x4_f32,
// optionally a batch of them (operands sa / sw / sc elements behind the first's).
//   gemm_f32_few_kernel   up to 64 rows: bound by the weights' stream (skinny_body.h)
//   gemm_f32_kernel       32 x 64 tiles behind an LDS-DMA ring: bound by the f32 MFMA
//   gemm_f32_any_kernel   K or pitches that 16-byte pieces of 64-wide chunks do not divide
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

// A decoding step's products had one 64 x 64 tile per 64 columns (64 blocks for 4096 x 1024, every k step a load's latency): 80 us on average at 2
// rows of the 0.6B widths, 6.4 us here; its 32768-column head 21 us (67 MB: 3.1 TB/s).
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
  skinny_sums<R8, M8, true>(src, a.K / 64, smem, wave, lane);
  for (int i = wave; i < (R8 / 2) * MT; i += SKINNY_WAVES) {
    const int f = i / MT, m = (i - f * MT) * 16 + c, n = n0 + f * 16 + G * 4;
    if (m < a.M && n < a.N) *reinterpret_cast<f32x4_t*>(a.C + blockIdx.y * a.sc + (int64_t)m * a.ldc + n) = skinny_total<R8, M8>(smem, i, lane);
  }
}

// WM * 16 rows x 64 columns, 64-wide k stages; WM = 2: four waves of 16 x 32, WM = 1: of 16 x 16.  A stage is requests of 1 KB (rows of 64 k of A are
// two lines: 4 WM of them; 8 of W), a quarter per wave; three stages keep two in flight under the one that multiplies, one barrier per stage.  The tile is
// this small so that a prompt of a few hundred rows still makes two to three blocks per CU: the f32 MFMA (32 cycles for 16 x 16 x 4) is the bound, idle
// SIMDs are the loss.
// 300 rows of the 0.6B widths: 87 us on average (64 x 64 tiles, one stage, through registers) -> 36 us.
// A wave of the wider tile multiplies for 0.43 us per stage, so a launch takes that times K / 64 however few blocks it has, and few blocks are spread over
// the CUs better in halves: 16 rows below 736 blocks of 32.  Blocks of 32 rows: us with 32 / 16 rows, K = 2048: 160: 30.6 / 24.9, 320: 44.9 / 33.8,
// 400: 45.1 / 33.8, 480: 45.2 / 42.6, 640: 60.2 / 55.3, 672: 60.8 / 55.9, 760 (nearly three for every CU): 60.6 / 62.7.  The sums' order is the same.
constexpr int F_S = 3;
constexpr int f_stage(int wm) { return (4 * wm + 8) * 1024; }
template <int WM>
__global__ __launch_bounds__(256) void gemm_f32_kernel(GemmF32Args a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];   // F_S x [A first halves | A second halves | W]
  constexpr int STAGE = f_stage(WM), HALF = WM * 2048, NA = WM, NR = WM, LEFT = (F_S - 2) * (NA + 2);   // A requests per wave, 16-column groups per wave
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), G = lane >> 4, c = lane & 15, wm = WM == 2 ? wave >> 1 : 0, wn = WM == 2 ? wave & 1 : wave;
  const int n0 = (int)blockIdx.y * 64, m0 = (int)blockIdx.x * (WM * 16);   // (consecutive blocks share the weights' tile)
  const float* A = a.A + blockIdx.z * a.sa;
  const bf16_t* W = a.W + blockIdx.z * a.sw;
  const char *asrc[NA], *wsrc[2];   // requests wave * NA + j of A, wave * 2 + j of W
#pragma unroll
  for (int j = 0; j < NA; ++j) {
    const int q = wave * NA + j, ar = q % (2 * WM) * 8 + (lane >> 3);
    asrc[j] = (const char*)(A + (int64_t)min(m0 + ar, a.M - 1) * a.lda) + q / (2 * WM) * 128 + skinny_piece(ar, lane);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int wr = (wave * 2 + j) * 8 + (lane >> 3);
    wsrc[j] = (const char*)(W + (int64_t)min(n0 + wr, a.N - 1) * a.ldw) + skinny_piece(wr, lane);
  }
  const int nk = a.K / 64;
  auto load = [&](int kt) {   // (past the end: the last stage again, never used)
    const int k = min(kt, nk - 1) * 128;
    char* st = smem + kt % F_S * STAGE;
#pragma unroll
    for (int j = 0; j < NA; ++j) __builtin_amdgcn_global_load_lds((glb_ptr_t)(asrc[j] + 2 * k), (lds_ptr_t)(st + (wave * NA + j) * 1024), 16, 0, 0);
#pragma unroll
    for (int j = 0; j < 2; ++j) __builtin_amdgcn_global_load_lds((glb_ptr_t)(wsrc[j] + k), (lds_ptr_t)(st + (4 * WM + wave * 2 + j) * 1024), 16, 0, 0);
  };
  f32x4_t acc[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) acc[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < F_S - 1; ++s) load(s);
  for (int kt = 0; kt < nk; ++kt) {
    __builtin_amdgcn_s_waitcnt(0x0F70 | (LEFT & 15) | ((LEFT >> 4) << 14));   // this wave's part of stage kt is in; behind the barrier everyone's, and stage kt - 1 is read
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    load(kt + F_S - 1);
    const char* st = smem + kt % F_S * STAGE;
    u32x4_t wf[2][NR];
    f32x4_t af[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int r = 0; r < NR; ++r) wf[h][r] = *reinterpret_cast<const u32x4_t*>(st + 2 * HALF + skinny_swz(wn * (NR * 16) + r * 16 + c, h * 4 + G));
#pragma unroll
      for (int q = 0; q < 2; ++q) af[h][q] = *reinterpret_cast<const f32x4_t*>(st + h * HALF + skinny_swz(wm * 16 + c, 2 * G + q));
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int r = 0; r < NR; ++r)
          acc[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(j & 1 ? hi_bf(wf[h][r][j >> 1]) : lo_bf(wf[h][r][j >> 1]), af[h][j >> 2][j & 3], acc[r], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // (the surplus requests: LDS may belong to the next block)
  const int m = m0 + wm * 16 + c;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int n = n0 + wn * (NR * 16) + r * 16 + G * 4;
    if (m < a.M && n < a.N) *reinterpret_cast<f32x4_t*>(a.C + blockIdx.z * a.sc + (int64_t)m * a.ldc + n) = acc[r];
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
  if (M > 64) {
    const unsigned tn = (unsigned)((N + 63) / 64);
    if ((int64_t)((M + 31) / 32) * tn * batch < 736) hipLaunchKernelGGL(gemm_f32_kernel<1>, dim3((unsigned)((M + 15) / 16), tn, (unsigned)batch), dim3(256), F_S * f_stage(1), st, a);
    else hipLaunchKernelGGL(gemm_f32_kernel<2>, dim3((unsigned)((M + 31) / 32), tn, (unsigned)batch), dim3(256), F_S * f_stage(2), st, a);
    return;
  }
  auto go = [&](auto r8, auto m8) {
    constexpr int R8 = decltype(r8)::value, M8 = decltype(m8)::value, lds = skinny_lds(R8, M8, true);
    if (lds > 64 * 1024) (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_f32_few_kernel<R8, M8>), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    hipLaunchKernelGGL((gemm_f32_few_kernel<R8, M8>), dim3((unsigned)((N + R8 * 8 - 1) / (R8 * 8)), (unsigned)batch), dim3(SKINNY_WAVES * 64), lds, st, a.A,
                       a.W, a.M, a.N, a.K, a.lda, a.ldw, a);
  };
  using std::integral_constant;
  // 48 weight rows per block where they still make two blocks per CU (the head); f32 rows take twice the LDS, so more than 32 of them leave room for 16
  const bool wide = (int64_t)((N + 47) / 48) * batch >= 512;
  if (M <= 8) wide ? go(integral_constant<int, 6>{}, integral_constant<int, 1>{}) : go(integral_constant<int, 2>{}, integral_constant<int, 1>{});
  else if (M <= 16) wide ? go(integral_constant<int, 6>{}, integral_constant<int, 2>{}) : go(integral_constant<int, 2>{}, integral_constant<int, 2>{});
  else if (M <= 32) wide ? go(integral_constant<int, 6>{}, integral_constant<int, 4>{}) : go(integral_constant<int, 2>{}, integral_constant<int, 4>{});
  else go(integral_constant<int, 2>{}, integral_constant<int, 8>{});
}

}  // namespace aha
