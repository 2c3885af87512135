// Shared device code of the few-row products (kernels_gemm_skinny.hip: dense; kernels_moe.hip: experts with few slots).  A block of four waves owns
// R8 * 8 weight rows, M8 * 8 activation rows and the whole K range; why and what it measured: kernels_gemm_skinny.hip.
#pragma once
#include <type_traits>

#include "common.h"

namespace aha {

namespace {

constexpr int SKINNY_WAVES = 4;
// Stages of a wave's ring.  Where blocks share a CU: three up to six requests each, two of wider ones.  Two to four blocks then hide each other's latency;
// more stages take the LDS that a neighbour needs (blocks of 16 weight rows: 151936 x 1024, 8 rows, 47.6 us with three stages, 60.0 with six; 32 bits,
// 12288 x 4096, 2 rows, 20.4 with three, 29.6 with five and one block per CU).  DEEP, a block that has its CU to itself: as many as cover a request's
// latency at a CU's share of HBM's rate, ~50 KB (8 rows: 4096 x 4096 8.0 us against 8.1 with three, 2048 x 4096 6.1 against 6.3).  Nothing is requested
// past the end.
constexpr int skinny_stages(int requests, bool deep = false) {
  if (deep) return requests <= 3 ? 6 : requests == 4 ? 5 : requests == 5 ? 4 : requests <= 8 ? 3 : 2;
  return requests <= 6 ? 3 : 2;
}
constexpr int skinny_requests(int r8, int m8, bool f32) { return r8 + (f32 ? 2 : 1) * m8; }
constexpr int skinny_lds(int r8, int m8, bool f32 = false, bool deep = false) {
  const int per = skinny_requests(r8, m8, f32);
  const int ring = SKINNY_WAVES * skinny_stages(per, deep) * per * 1024;
  const int sums = SKINNY_WAVES * ((r8 + 1) / 2) * ((m8 + 1) / 2) * 1024;
  return ring > sums ? ring : sums;
}

constexpr int skinny_blocks(int r8, int m8, bool f32 = false) { return 160 * 1024 / skinny_lds(r8, m8, f32); }   // per CU
static_assert(skinny_blocks(2, 1) == 4 && skinny_blocks(2, 2) == 3 && skinny_blocks(3, 1) == 3 && skinny_blocks(2, 1, true) == 3, "narrow stages: room for three and more blocks");
static_assert(skinny_blocks(2, 4) == 2 && skinny_blocks(2, 8) == 2 && skinny_blocks(3, 4) == 2 && skinny_blocks(4, 2) == 2 && skinny_blocks(6, 4) == 2 && skinny_blocks(6, 2, true) == 2,
              "up to ten requests: two");

// 16-byte piece `slot` of row `row` inside a stage's [rows][64] bf16 image
__device__ __forceinline__ int skinny_swz(int row, int slot) { return row * 128 + ((slot ^ ((row >> 1) & 7)) << 4); }
// the byte offset inside its 128-byte line that lane `lane` of a request fetches (a request: eight rows, eight lanes each)
__device__ __forceinline__ int skinny_piece(int local_row, int lane) { return ((lane & 7) ^ ((local_row >> 1) & 7)) * 16; }

// Where a block starts in K.  All blocks stream at one pace, so from a common start their requests at any moment lie in one narrow band of columns of all
// weight rows -- one value of the address bits below the row pitch, a few of the memory's channels.  The blocks of 96 weight rows (whole blocks of 16, 24, 32
// and 48: an element's sum has the same order for every R8 and M8) start four chunks behind their neighbours: 8 rows, 12288 x 4096 17.5 -> 16.4 us (6.1 TB/s),
// 4096 x 4096 8.0 -> 7.0, 4096 x 12288 17.7 -> 16.6, 6144 x 4096 10.6 -> 9.8; 32 rows, 4096 x 8192 17.8 -> 15.9, 24576 x 4096 35.0 -> 32.7; 48 weight rows, 5 % in
// the mean of 14 shapes.  One or nine chunks behind: 2 and 0 %.  K < 2048: no difference.
__device__ __forceinline__ int skinny_first(int weight_row, int nc) {
  return nc < 32 ? 0 : weight_row / 96 * 4 & ((1 << (31 - __builtin_clz(nc))) - 1);   // (below the largest power of two in nc)
}

// A float as the sum of three bf16 (its 24 significant bits cut 8 / 8 / 8: exact unless the parts fall below bf16's range, 2^-133), eight floats at a time in the
// order of an MFMA operand.  With weights that are bf16 themselves all three products are exact and nothing is left out, so a product on the bf16 units has
// an f32 unit's error (the sums are f32) at three sixteenths of its matrix cycles.
struct SplitBf16x8 { bf16x8_t hi, mid, lo; };
__device__ __forceinline__ SplitBf16x8 split_bf16(const f32x4_t& x0, const f32x4_t& x1) {
  u32x4_t p[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = i < 2 ? x0[2 * i] : x1[2 * i - 4], b = i < 2 ? x0[2 * i + 1] : x1[2 * i - 3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const unsigned ua = __builtin_bit_cast(unsigned, a), ub = __builtin_bit_cast(unsigned, b);
      p[k][i] = __builtin_amdgcn_perm(ub, ua, 0x07060302u);   // the upper halves
      a -= __builtin_bit_cast(float, ua & 0xffff0000u);
      b -= __builtin_bit_cast(float, ub & 0xffff0000u);
    }
  }
  return {__builtin_bit_cast(bf16x8_t, p[0]), __builtin_bit_cast(bf16x8_t, p[1]), __builtin_bit_cast(bf16x8_t, p[2])};
}
// the upper parts' sums and the others'.  An infinity's rest is NaN (inf - inf), so where the upper parts' sum is not finite it is the result, as it would
// be without the split
__device__ __forceinline__ f32x4_t split_sum(const f32x4_t& big, const f32x4_t& rest) {
  f32x4_t s;
#pragma unroll
  for (int i = 0; i < 4; ++i) s[i] = fabsf(big[i]) < INFINITY ? big[i] + rest[i] : big[i];
  return s;
}

// What a product does to its bf16 activations on the way from LDS: nothing
struct SkinnyPlain {
  static constexpr bool ON = false;
  __device__ __forceinline__ void request() {}
  __device__ __forceinline__ void join() {}
  __device__ __forceinline__ u32x4_t map(u32x4_t x) const { return x; }
};

// src[r]: where this lane's piece of request r starts at k = 0 -- R8 weight groups (bf16), then M8 activation groups (bf16); F32: activations are f32,
// a row's 64 k are two requests, the first halves of all groups before the second halves, and the activations' parts (split_bf16) multiply in turn.
// nc: 64-wide k chunks, first: the chunk that wave 0 starts at (skinny_first), wrapping round behind the last.
// On return the waves' sums of the 16 x 16 fragments (weight fragment r, activation fragment m) lie in LDS and every wave may read them
// (skinny_total).
// pro: request() in front of the ring's first requests, join() behind them (with pro all of them are made: nc >= S * SKINNY_WAVES), map() on every fragment.
template <int R8, int M8, bool F32 = false, bool DEEP = false, typename PRO = SkinnyPlain>
__device__ __forceinline__ void skinny_sums(const char* (&src)[skinny_requests(R8, M8, F32)], int nc, int first, char* smem, int wave, int lane, PRO pro = {}) {
  typedef __attribute__((address_space(3))) void* lds_t;
  typedef const __attribute__((address_space(1))) void* glb_t;
  constexpr int NF = (R8 + 1) / 2, MT = (M8 + 1) / 2, PER = skinny_requests(R8, M8, F32), S = skinny_stages(PER, DEEP);
  constexpr int LEFT = (S - 1) * PER;   // requests of the later stages
  static_assert(LEFT < 64, "vmcnt has six bits");
  // Eight rows that are mapped: a fragment's columns 0-7 are their first 32 k of a chunk and columns 8-15 the second 32, so that nothing is mapped twice; what a
  // product gives for the columns of the other half is nobody's, and the second half's sums move by eight lanes at the end.
  constexpr bool HALVES = PRO::ON && M8 == 1;
  const int G = lane >> 4, c = lane & 15;
  char* ring = smem + wave * (S * PER * 1024);
  f32x4_t acc[2][NF][MT];   // the two halves of a chunk (F32: the upper parts and the others) in chains of their own: half the dependent steps, half the roundings in a row
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < NF; ++r)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[h][r][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int end = nc * 128;
  int k = (first + wave < nc ? first + wave : first + wave - nc) * 128;   // the next chunk to request, in bytes of a weight row
  auto load = [&](int u) {
    const int ka = F32 ? 2 * k : k;
#pragma unroll
    for (int r = 0; r < R8; ++r) __builtin_amdgcn_global_load_lds((glb_t)(src[r] + k), (lds_t)(ring + (u * PER + r) * 1024), 16, 0, 2);   // weights: non-temporal
#pragma unroll
    for (int r = R8; r < PER; ++r) __builtin_amdgcn_global_load_lds((glb_t)(src[r] + ka), (lds_t)(ring + (u * PER + r) * 1024), 16, 0, 0);
    k += SKINNY_WAVES * 128;
    k -= k < end ? 0 : end;
  };
  // an odd count leaves half a fragment without rows: its lanes read the other half's again (behind the last stage there may be no LDS)
  const int cw = R8 % 2 ? c & 7 : c, ca = M8 % 2 ? c & 7 : c;   // (of the last fragment)
  auto consume = [&](int u) {
    const char *sw = ring + u * PER * 1024, *sa = sw + R8 * 1024;
    u32x4_t wf[2][NF];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < NF; ++r) wf[h][r] = *reinterpret_cast<const u32x4_t*>(sw + skinny_swz(r * 16 + (r + 1 == NF ? cw : c), h * 4 + G));
    if constexpr (F32) {
      f32x4_t af[2][MT][2];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int q = 0; q < 2; ++q) af[h][m][q] = *reinterpret_cast<const f32x4_t*>(sa + h * (M8 * 1024) + skinny_swz(m * 16 + (m + 1 == MT ? ca : c), 2 * G + q));
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const SplitBf16x8 x = split_bf16(af[h][m][0], af[h][m][1]);
#pragma unroll
          for (int r = 0; r < NF; ++r) acc[0][r][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[h][r]), x.hi, acc[0][r][m], 0, 0, 0);
#pragma unroll
          for (int r = 0; r < NF; ++r) acc[1][r][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[h][r]), x.lo, acc[1][r][m], 0, 0, 0);
#pragma unroll
          for (int r = 0; r < NF; ++r) acc[1][r][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[h][r]), x.mid, acc[1][r][m], 0, 0, 0);
        }
    } else {
      bf16x8_t af[2][MT];
      if constexpr (HALVES) af[0][0] = af[1][0] = __builtin_bit_cast(bf16x8_t, pro.map(*reinterpret_cast<const u32x4_t*>(sa + skinny_swz(c & 7, (c >> 3) * 4 + G))));
#pragma unroll
      for (int h = 0; h < (HALVES ? 0 : 2); ++h)
#pragma unroll
        for (int m = 0; m < MT; ++m) af[h][m] = __builtin_bit_cast(bf16x8_t, pro.map(*reinterpret_cast<const u32x4_t*>(sa + skinny_swz(m * 16 + (m + 1 == MT ? ca : c), h * 4 + G))));
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < NF; ++r)
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[h][r][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[h][r]), af[h][m], acc[h][r][m], 0, 0, 0);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);   // the stage's fragments are in registers: it may be filled again
    __builtin_amdgcn_sched_barrier(0);
  };
  int u = 0, ch = wave;
  pro.request();
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (PRO::ON || wave + s * SKINNY_WAVES < nc) load(s);
  if constexpr (PRO::ON) __builtin_amdgcn_sched_barrier(0);
  pro.join();
  for (; ch + S * SKINNY_WAVES < nc; ch += SKINNY_WAVES) {   // S stages are on their way: the oldest is in when the later ones' requests are left
    __builtin_amdgcn_s_waitcnt(0x0F70 | (LEFT & 15) | ((LEFT >> 4) << 14));
    __builtin_amdgcn_sched_barrier(0);
    consume(u);
    load(u);
    u = u + 1 == S ? 0 : u + 1;
  }
  for (; ch < nc; ch += SKINNY_WAVES) {   // the last ones: as many behind this one as there are chunks left
    const int later = (nc - 1 - ch) / SKINNY_WAVES;
    auto wait = [&](auto n) {
      constexpr int L = decltype(n)::value * PER;
      if constexpr (decltype(n)::value < S)
        if (later == decltype(n)::value) __builtin_amdgcn_s_waitcnt(0x0F70 | (L & 15) | ((L >> 4) << 14));
    };
    wait(std::integral_constant<int, 0>{});
    wait(std::integral_constant<int, 1>{});
    wait(std::integral_constant<int, 2>{});
    wait(std::integral_constant<int, 3>{});
    wait(std::integral_constant<int, 4>{});
    wait(std::integral_constant<int, 5>{});
    static_assert(S <= 6, "a wait for every number of later stages");
    __builtin_amdgcn_sched_barrier(0);
    consume(u);
    u = u + 1 == S ? 0 : u + 1;
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // no DMA may land in what becomes the sums' space
  __syncthreads();
  auto red = reinterpret_cast<f32x4_t(*)[NF * MT][64]>(smem);
  if constexpr (HALVES)
#pragma unroll
    for (int r = 0; r < NF; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[1][r][0][i] = __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(acc[1][r][0][i]), 0x128 /* row_ror:8 */, 0xf, 0xf, false));
#pragma unroll
  for (int r = 0; r < NF; ++r)
#pragma unroll
    for (int m = 0; m < MT; ++m) red[wave][r * MT + m][lane] = F32 ? split_sum(acc[0][r][m], acc[1][r][m]) : acc[0][r][m] + acc[1][r][m];
  __syncthreads();
}

// the four waves' sums of fragment pair i = r * MT + m for lane l: weight rows r * 16 + (l >> 4) * 4 .. + 4, activation row m * 16 + (l & 15)
template <int R8, int M8>
__device__ __forceinline__ f32x4_t skinny_total(const char* smem, int i, int l) {
  auto red = reinterpret_cast<const f32x4_t(*)[((R8 + 1) / 2) * ((M8 + 1) / 2)][64]>(smem);
  static_assert(SKINNY_WAVES == 4, "joined in pairs");
  return (red[0][i][l] + red[1][i][l]) + (red[2][i][l] + red[3][i][l]);
}

}  // namespace

}  // namespace aha
