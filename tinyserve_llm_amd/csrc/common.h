// Shared device helpers for the gfx950 kernels: storage types, conversions, wave reductions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "entry_points.h"

#define TS_WAVE 64

typedef uint16_t bf16_t;  // bfloat16 stored as its 16 raw bits

__device__ __forceinline__ float bf2f(bf16_t h) { return __uint_as_float(((uint32_t)h) << 16); }

// round to nearest even; NaN stays NaN
__device__ __forceinline__ bf16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16_t)(u >> 16);
}

template <typename T> struct Num;
template <> struct Num<float> {
  static __device__ __forceinline__ float ld(const float* p) { return *p; }
  static __device__ __forceinline__ void st(float* p, float v) { *p = v; }
  static __device__ __forceinline__ float round(float v) { return v; }
};
template <> struct Num<bf16_t> {
  static __device__ __forceinline__ float ld(const bf16_t* p) { return bf2f(*p); }
  static __device__ __forceinline__ void st(bf16_t* p, float v) { *p = f2bf(v); }
  static __device__ __forceinline__ float round(float v) { return bf2f(f2bf(v)); }
};

// 16 bytes that one workgroup reads once and no other soon after (a weight's, a cache's): told so, the caches do not put other lines out for them.
typedef uint32_t stream_u32x4_t __attribute__((ext_vector_type(4)));
template <typename V = uint4> __device__ __forceinline__ V load_once(const void* p) {
  static_assert(sizeof(V) == 16, "16 bytes");
  return __builtin_bit_cast(V, __builtin_nontemporal_load((const stream_u32x4_t*)p));
}
// The same for what is written and not read again soon (a state, until the next step).
template <typename V> __device__ __forceinline__ void store_once(void* p, const V& v) {
  static_assert(sizeof(V) == 16, "16 bytes");
  __builtin_nontemporal_store(__builtin_bit_cast(stream_u32x4_t, v), (stream_u32x4_t*)p);
}

// A kernel's arguments lie in memory that no cache holds when the kernel starts, and the compiler fetches them
// as the code comes to need them: a long argument block is then waited for two or three times, a trip to
// memory each, before the first load of the operands can go out. This asks for one word of each 64 bytes of
// the block at the very start, so that all of it arrives in one trip and every later fetch finds it in the
// scalar cache.
template <int BYTES>
__device__ __forceinline__ void ts_fetch_arguments() {
  typedef const uint32_t __attribute__((address_space(4))) * args_t;
  const args_t block = (args_t)__builtin_amdgcn_kernarg_segment_ptr();
  uint32_t seen = 0;
#pragma unroll
  for (int at = 0; at < BYTES; at += 64) seen |= block[at / 4];
  asm volatile("" ::"s"(seen));
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = TS_WAVE / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, TS_WAVE);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = TS_WAVE / 2; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, TS_WAVE));
  return v;
}

// The first key that the query at position `pos` sees (it sees up to `pos`). `window` > 0: the last `window`
// positions, itself included (a sliding window); `window` < 0: the positions of its own chunk of -window
// positions, chunks counted from position 0 of the request; 0: every key before it.
__device__ __forceinline__ int ts_first_key(int pos, int window) {
  if (window > 0) return pos - window + 1 > 0 ? pos - window + 1 : 0;
  if (window < 0) return pos - pos % (-window);
  return 0;
}

// Orders shared-memory writes of a wavefront before the reads of its other lanes.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

static inline int ts_check_launch() {
  return hipGetLastError() == hipSuccess ? TS_OK : TS_LAUNCH_FAILED;
}
