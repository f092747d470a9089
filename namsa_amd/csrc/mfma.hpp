// What the corrector network's kernels share: operands of
// v_mfma_f32_32x32x16_bf16 and buffer accesses.
//
// Operand layout (lane l, 8 bf16 per operand register set):
//   A: row l%32, k = 8*(l/32) + e      B: column l%32, k = 8*(l/32) + e
//   D: 16 floats, register r holds row 8*(r/4) + 4*(l/32) + r%4, column l%32.
#pragma once

#include <hip/hip_runtime.h>

namespace namsa {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t Rsrc;

constexpr int kRawBuffer = 0x00020000;  // gfx9 raw-buffer resource word 3
constexpr int kNowhere = 0x7ffffffc;    // a byte offset past every buffer: reads there give 0, stores are dropped

__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x16 zero16() {
  f32x16 v;
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = 0.0f;
  return v;
}

__device__ __forceinline__ bf16x8 ld8(const __bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }

// Accesses through a buffer resource at a lane's and a scalar byte offset.
__device__ __forceinline__ Rsrc buffer_of(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, kRawBuffer);
}
__device__ __forceinline__ float load_b32(Rsrc r, int lane_at, int at) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, lane_at, at, 0));
}
__device__ __forceinline__ void store_b32(float v, Rsrc r, int lane_at, int at) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, lane_at, at, 0);
}
__device__ __forceinline__ bf16x8 load_bf8(Rsrc r, int lane_at, int at) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, lane_at, at, 0));
}
// eight consecutive floats, rounded to bf16
__device__ __forceinline__ bf16x8 load_f8(Rsrc r, int lane_at, int at) {
  const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(r, lane_at, at, 0);
  const u32x4 b = __builtin_amdgcn_raw_buffer_load_b128(r, lane_at, at + 16, 0);
  bf16x8 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = __bf16(__builtin_bit_cast(float, static_cast<unsigned>(a[e])));
    v[e + 4] = __bf16(__builtin_bit_cast(float, static_cast<unsigned>(b[e])));
  }
  return v;
}

// Registers 8 s .. 8 s + 7 of a product, rounded, as the operand of a next one
// that sums over its rows 16 s .. 16 s + 15: the halves of the wavefront hold
// rows 0-3, 8-11 and 4-7, 12-15 and exchange half of them to hold 0-7 and 8-15.
__device__ __forceinline__ bf16x8 rows_to_k(bf16x8 v) {
  u32x4 w = __builtin_bit_cast(u32x4, v);
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const auto p = __builtin_amdgcn_permlane32_swap(w[e], w[e + 2], false, false);
    w[e] = p[0];
    w[e + 2] = p[1];
  }
  return __builtin_bit_cast(bf16x8, w);
}

// A wavefront exchanges through its own LDS tile in program order: only the
// compiler has to be held to it.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace namsa
