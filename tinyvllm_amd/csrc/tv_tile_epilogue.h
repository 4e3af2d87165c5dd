// Epilogue of the tiled products (tile_linear.hip, tile_linear_f32.hip).
#pragma once

#include "tv_dense.h"
#include "tv_linear.h"

namespace tv {

// Eight consecutive outputs of T at out[at]: one (16-bit) or two (fp32) 16-byte stores.
template <typename T> __device__ __forceinline__ void store8(void* out, size_t at, const float (&o)[8]) {
  *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(out) + at) =
      u32x4{pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3]), pack2<T>(o[4], o[5]), pack2<T>(o[6], o[7])};
}
template <> __device__ __forceinline__ void store8<float>(void* out, size_t at, const float (&o)[8]) {
  f32x4* p = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(out) + at);
  p[0] = f32x4{o[0], o[1], o[2], o[3]};
  p[1] = f32x4{o[4], o[5], o[6], o[7]};
}

// A wave's 16 MBW tokens from m_wave by 64 features from nw: lane (g, col) holds
// four consecutive features of token 16 mb + col per (mb, nb) -- features
// 16 nb + 4 g .. + 3, or 16 g + 4 nb .. + 3 for SwiGLU.
template <typename T, int EPI, int MBW>
__device__ __forceinline__ void tile_epilogue(const LinearParams& p, const f32x4 (&acc)[MBW][4], int m_wave, int nw,
                                              int split, int lane) {
  constexpr int NB = 4;
  const int g = lane >> 4;
  const int col = lane & 15;
#pragma unroll
  for (int mb = 0; mb < MBW; ++mb) {
    const int m = m_wave + mb * 16 + col;
    if constexpr (EPI == kEpiPartial) {
      if (m < p.M) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const int n = nw + 16 * nb + 4 * g;
          if (n < p.N) *reinterpret_cast<f32x4*>(p.part + ((size_t)split * p.M + m) * p.N + n) = acc[mb][nb];
        }
      }
    } else if constexpr (EPI == kEpiSwiglu) {
      float o[8];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const f32x4 v = acc[mb][nb];
        o[2 * nb] = silu(v[0]) * v[2];
        o[2 * nb + 1] = silu(v[1]) * v[3];
      }
      const int n = nw + 16 * g;
      const size_t at = (size_t)m * p.ldo + (n >> 1);
      if (m < p.M) {
        if (n + 16 <= p.N && p.ldo % (16 / sizeof(T)) == 0 && ((uintptr_t)p.out & 15) == 0) {
          store8<T>(p.out, at, o);
        } else {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            if (n + 4 * nb < p.N) store2<T>(p.out, at + 2 * nb, o[2 * nb], o[2 * nb + 1]);
        }
      }
    } else {
      unsigned long long best = 0;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int n = nw + 16 * nb + 4 * g;
        const f32x4 v = acc[mb][nb];
        if (n < p.N) {
          if (p.out && m < p.M) *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.out) + (size_t)m * p.ldo + n) = v;
#pragma unroll
          for (int i = 0; i < 4; ++i) best = max(best, argmax_key(v[i], n + i));
        }
      }
      if (p.keys && nw < p.N) {   // one key per token and 64 features: the lanes of a token are 16 apart
#pragma unroll
        for (int off = 16; off <= 32; off <<= 1) {
          const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute((lane ^ off) << 2, (int)(uint32_t)best);
          const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute((lane ^ off) << 2, (int)(uint32_t)(best >> 32));
          best = max(best, ((unsigned long long)hi << 32) | lo);
        }
        if (g == 0 && m < p.M) p.keys[(size_t)(nw / kLinBN) * p.M + m] = best;
      }
    }
  }
}

}  // namespace tv
