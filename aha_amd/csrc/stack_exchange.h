// Blocks of one launch that hand vectors to each other (kernels_decode_stack.hip, kernels_prenorm_stack.hip): a value travels with its tag in one dword (bf16 and the
// low half of the tag) or two (f32 and the tag), written by one block and polled past the L1 by others.
#pragma once
#include "common.h"

namespace aha {
namespace stack {

constexpr uint32_t NOWHERE = 0x7fffffffu;   // past every descriptor's range: the store is dropped

constexpr int AUX_NT = 2, AUX_SC1 = 16;   // a load past the L1; a store through to memory

typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;
constexpr u32x4_t NO_SPLIT = {0xff800000u, 0u, 0u, 0u};   // what a split of the attention leaves that has no keys: its maximum (-inf) and its sum, each with its tag
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
#define IN_ORDER __builtin_amdgcn_sched_barrier(0)   // of requests and results, as written
__device__ __forceinline__ float silu_of(float x) { return x / (1.0f + expf(-x)); }
// LDS of this wave written and read, everybody here; requests of weights stay in flight
__device__ __forceinline__ void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Eight products: what a stage takes in is bf16, as the weights are, so v_dot2_f32_bf16 adds two exact products at a time.  Against 64 bits its sums are as close as
// those of an fma chain (1024 columns of weights and activations, rms over the sum of the products' sizes: 3.36e-9 and 3.37e-9; over 24 octaves 1.34e-8 and 1.27e-8, at 3072
// columns 0.99e-8 and 1.03e-8: the unit drops, downwards, what lies far below the largest of its three addends), at a quarter of the instructions: a SIMD has one of these
// waves, and the 500 instructions of gate and up were 1.3 us.
__device__ __forceinline__ float dot8_bf(u32x4_t h, u32x4_t w, float s) {
#pragma unroll
  for (int j = 0; j < 4; ++j) s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, (uint32_t)h[j]), __builtin_bit_cast(bf16x2_t, (uint32_t)w[j]), s, false);
  return s;
}
// a in the lower half of the wave, b in the upper one: each the sum of its two halves
__device__ __forceinline__ float halves(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// a in the even rows of 16 lanes, b in the odd ones: each the sum of a pair of rows
__device__ __forceinline__ float quarters(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// row G of 16 lanes: the sum of y[G] over the wave
__device__ __forceinline__ float four_sums(float y0, float y1, float y2, float y3) { return row_sum(quarters(halves(y0, y2), halves(y1, y3))); }
__device__ __forceinline__ void nap(int n) {
  for (int i = 0; i < n; ++i) __builtin_amdgcn_s_sleep(1);
}
// an address from memory, in the address space that it is in (a generic one would make flat loads)
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(1))) T* global_at(const void* p) { return (const __attribute__((address_space(1))) T*)(uintptr_t)p; }
// A wave that waits for values.  One that has given up goes on with none() instead of what it last found: parts of other steps need not fit together (splits that
// nobody ever wrote have the sum 0), and what such a step and the ones queued behind it append to the cache must be numbers, since the step that is run again
// reads it with weight zero.
struct Poller {
  __amdgpu_buffer_rsrc_t ex;
  int left;   // polls in vain that this wave still makes
  template <class Load, class None>   // load(): requests, and says whether everything is there
  __device__ __forceinline__ void until(bool ok, Load&& load, None&& none) {
    for (;;) {
      if (!ok) ok = load();
      asm volatile("" ::: "memory");
      if (__all(ok)) return;
      if (left <= 0) return none();
      --left;
    }
  }
  // behind the last wait: the launch is marked where this wave gave up (and no earlier one had been)
  __device__ __forceinline__ void report(bool failed, unsigned* fail_dev, unsigned* fail_host, uint32_t epoch) const {
    if (left > 0 || failed || (threadIdx.x & 63)) return;
    __hip_atomic_store(fail_dev, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(fail_host, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  // four values (of a lane that takes part)
  __device__ __forceinline__ u32x4_t values(bool part, uint32_t at, uint32_t t16) {
    u32x4_t v = {0u, 0u, 0u, 0u};
    until(!part, [&] {
      v = __builtin_amdgcn_raw_buffer_load_b128(ex, at, 0, AUX_SC1);
      return (((v[0] ^ t16) | (v[1] ^ t16) | (v[2] ^ t16) | (v[3] ^ t16)) & 0xffffu) == 0;
    }, [&] { v = u32x4_t{0u, 0u, 0u, 0u}; });
    return v;
  }
  // `row` (a lane's, the same in both halves of the wave): the sum of what the eight XCDs left at `at`, (XCD, PITCH) f32 with their tags
  template <int PITCH>
  __device__ __forceinline__ float sum_parts(uint32_t at, int row, uint32_t tag) {
    const uint32_t off = at + (((threadIdx.x & 63) >> 5) * 4 * PITCH + row) * 8;
    u32x2_t p[4] = {};
    until(false, [&] {
      uint32_t bad = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) p[i] = __builtin_amdgcn_raw_buffer_load_b64(ex, off + i * (PITCH * 8), 0, AUX_SC1);
#pragma unroll
      for (int i = 0; i < 4; ++i) bad |= p[i][1] ^ tag;
      return bad == 0;
    }, [&] { p[0] = p[1] = p[2] = p[3] = u32x2_t{0u, 0u}; });
    const float y = (__uint_as_float(p[0][0]) + __uint_as_float(p[1][0])) + (__uint_as_float(p[2][0]) + __uint_as_float(p[3][0]));
    return halves(y, y);
  }
};
__device__ __forceinline__ uint2 pack4(u32x4_t v) { return make_uint2((v[0] >> 16) | (v[1] & 0xffff0000u), (v[2] >> 16) | (v[3] & 0xffff0000u)); }

}  // namespace stack
}  // namespace aha
