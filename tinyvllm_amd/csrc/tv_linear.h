// Device helpers shared by the product kernels (dense.hip, tile_linear.hip) and
// the norm / RoPE kernels: argmax keys, SiLU, typed vector access and the MFMA
// step over one pair of 16-byte fragments.
#pragma once

#include "tv_common.h"

namespace tv {

__device__ __forceinline__ unsigned long long argmax_key(float v, int n) {
  // order-preserving map of the float to an unsigned key; ties resolve to the
  // smallest index, as numpy / tinygrad argmax return the first maximum
  uint32_t u = __builtin_bit_cast(uint32_t, v);
  u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  return ((unsigned long long)u << 32) | (0xFFFFFFFFu - (uint32_t)n);
}

__device__ __forceinline__ float silu(float x) { return x / (1.0f + expf(-x)); }

// Two / four consecutive elements of T to and from floats.
template <typename T> __device__ __forceinline__ void store2(void* base, size_t idx, float a, float b) {
  *reinterpret_cast<uint32_t*>(reinterpret_cast<uint16_t*>(base) + idx) = pack2<T>(a, b);
}
template <> __device__ __forceinline__ void store2<float>(void* base, size_t idx, float a, float b) {
  *reinterpret_cast<float2*>(reinterpret_cast<float*>(base) + idx) = float2{a, b};
}
template <typename T> __device__ __forceinline__ void store4(void* base, size_t idx, f32x4 v) {
  *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(base) + idx) = u32x2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
}
template <> __device__ __forceinline__ void store4<float>(void* base, size_t idx, f32x4 v) {
  *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(base) + idx) = v;
}
template <typename T> __device__ __forceinline__ f32x4 load4(const void* base, size_t idx) {
  const u32x2 e = *reinterpret_cast<const u32x2*>(reinterpret_cast<const T*>(base) + idx);
  float a, b, c, d;
  unpack2<T>(e[0], a, b);
  unpack2<T>(e[1], c, d);
  return f32x4{a, b, c, d};
}
template <> __device__ __forceinline__ f32x4 load4<float>(const void* base, size_t idx) {
  return *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(base) + idx);
}

// acc += (16 rows of W) x (16 columns of A^T) over the k range of one pair of
// 16-byte fragments: one v_mfma_f32_16x16x32 for 16-bit T; for fp32 four
// v_mfma_f32_16x16x4_f32, step j taking element j of every lane's fragment
// (lane group g then holds k = 4 g + j in both operands, so the steps cover
// the fragment's 16 k once).
template <typename T> __device__ __forceinline__ f32x4 mfma_frag(u32x4 a, u32x4 b, f32x4 c) {
  return mfma16x16x32<T>(a, b, c);
}
template <> __device__ __forceinline__ f32x4 mfma_frag<float>(u32x4 a, u32x4 b, f32x4 c) {
#pragma unroll
  for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(u32_as_f32(a[j]), u32_as_f32(b[j]), c, 0, 0, 0);
  return c;
}

}  // namespace tv
