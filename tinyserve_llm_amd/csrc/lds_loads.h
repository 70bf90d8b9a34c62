// Loads that go from memory straight into shared memory, and the waits that belong to them.
#pragma once
#include "attention_mfma.h"

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));   // (a plain vector: arrays of it stay in registers)
typedef __attribute__((address_space(3))) void* lds_ptr_t;

static __device__ __forceinline__ float4_t mfma32v(u32x4_t a, u32x4_t b, float4_t acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), acc, 0, 0, 0);
}

// Where loads are aimed: byte offsets from `base`, below 2 GB.
static __device__ __forceinline__ __amdgpu_buffer_rsrc_t load_base(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0x7fffffff, 0x20000);
}

// 1 KB from memory straight into LDS: lane l's 16 bytes at voffset + soffset land at lds + 16 l
static __device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t rsrc, uint32_t lds, uint32_t voffset, uint32_t soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)(uintptr_t)lds, 16, (int)voffset, (int)soffset, 0, 0);
}

// The same for what is read once: the caches do not put other lines out for it
static __device__ __forceinline__ void load_to_lds_once(__amdgpu_buffer_rsrc_t rsrc, uint32_t lds, uint32_t voffset, uint32_t soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)(uintptr_t)lds, 16, (int)voffset, (int)soffset, 0, 2);
}

// The same with an address of its own for every lane's 16 bytes (rows gathered from anywhere)
static __device__ __forceinline__ void row_to_lds(const void* src, uint32_t lds) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (lds_ptr_t)(uintptr_t)lds, 16, 0, 0);
}

// Waits until at most VM loads and LGKM reads of this wave are under way (vmcnt in bits 3:0 and 15:14, lgkmcnt in 11:8).
template <int VM, int LGKM = 15> static __device__ __forceinline__ void wait_for() {
  __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4) | (LGKM << 8));
}
