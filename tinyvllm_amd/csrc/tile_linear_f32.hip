// Y = A W^T at fp32 for many rows of A (prompt passes), on the bf16 matrix
// cores: every fp32 element is split exactly into three bf16 parts, and six of
// the nine products of parts make the fp32 product (tv_split.h).  The matrix
// unit spends 96 cycles on them where v_mfma_f32_16x16x4_f32 spends 256.
//
// A work-group computes a BM x BN tile of Y, its waves 64 features each.
// Per stage of 32 K elements every thread splits its share of both operands
// (loaded into registers a stage ahead) once for all waves and writes the parts
// as planes of 64-byte LDS rows; the 16-byte chunks of a row are XOR-permuted,
// so fragment reads and writes touch every bank once.
//
// What bounds it: the matrix unit at the rate it sustains (512 x 32000 x 2048:
// 375 us, 1.07 PFLOP/s of bf16; the 16-bit product reaches 1.23), and below
// that size the split, which takes its issue slots (64 x 128 tile: 620 clocks
// of a stage beside 768 of products).  Four work-groups per CU of the smaller
// tile (118 registers) run their splits beside each other's products; two with
// a second stage buffer, split and products interleaved, were 3% slower.
// MI355X, against fp32 products on the skinny kernel: 300 x 11264 x 2048 158 ->
// 117 us, 300 x 2048 x 5632 122 -> 58, 512 x 32000 x 2048 616 -> 375.  Parts that
// are cut off instead of rounded saved 3% and adding products straight into the
// sum 4% more, but then what is left out or lost has the sign of the product
// (error x10 on positive data of K 16384).
// Error against 64 bits (2-norm, K 256 / 2048 / 16384): N(0, 1) 0.7e-7 / 1.6e-7 /
// 4.3e-7, fp32 products 2.9e-7 / 8.2e-7 / 2.3e-6; uniform in [0, 1) 0.5e-7 /
// 1.1e-7 / 3.0e-7 against 2.2e-7 / 6.0e-7 / 1.7e-6; all low bits of every
// operand set 0.5e-7 / 2.2e-7 / 4.2e-7 against 0.5e-7 / 9.7e-6 / 2.9e-5.
#include "tv_split.h"
#include "tv_dense.h"
#include "tv_linear.h"
#include "tv_tile_dma.h"
#include "tv_tile_epilogue.h"

#include <algorithm>

namespace tv {

namespace {

constexpr int kBK = 32;          // K elements per stage
constexpr int kRowBytes = 64;    // of one part's LDS row

// 16-byte chunk c of row r sits at slot c ^ part_row_perm(r): over the 16 rows
// of a fragment read (16 b + i, or SPREAD: 16 a + 4 b + i) the pairs (r & 3,
// slot) are distinct, and four rows cover the banks.
__device__ __forceinline__ int part_row_perm(int r) { return ((r >> 2) ^ (r >> 4)) & 3; }

}  // namespace

// WM x WN waves, each 16 MBW rows of A (tokens) by 64 rows of W (features).
template <int EPI, int MBW, int WM, int WN, int WPE>
__global__ void __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(WPE)))
tile_linear_f32_kernel(const LinearParams p) {
  constexpr int NT = 64 * WM * WN;
  constexpr int BM = 16 * MBW * WM;
  constexpr int BN = 64 * WN;
  constexpr int NB = 4;
  constexpr int LA = BM * 4 / NT;      // 8-element units of A per thread and stage
  constexpr int LW = BN * 4 / NT;
  constexpr int PLANE = (BM + BN) * kRowBytes;
  constexpr bool SPREAD = EPI == kEpiSwiglu;   // tile_linear.hip
  static_assert(LA * NT == BM * 4 && LW * NT == BN * 4, "whole units per thread");
  __shared__ __attribute__((aligned(16))) uint8_t lds[3 * PLANE];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int g = lane >> 4;
  const int col = lane & 15;
  const int wm = wave / WN, wn = wave % WN;

  // work-group -> (split, n tile, m tile), as in tile_linear.hip
  const int mt = (p.M + BM - 1) / BM;
  const int nt = (p.N + BN - 1) / BN;
  const int per = gridDim.x >> 3, rest = gridDim.x & 7;
  const int xcd = blockIdx.x & 7;
  int t = xcd * per + min(xcd, rest) + (blockIdx.x >> 3);
  const int split = t / (mt * nt);
  t -= split * mt * nt;
  constexpr int GM = 8;
  const int grp = t / (GM * nt);
  const int gm = min(GM, mt - grp * GM);
  t -= grp * GM * nt;
  const int ntile = t / gm;
  const int m0 = (grp * GM + t - ntile * gm) * BM;
  const int n0 = ntile * BN;
  const int kb = split * p.k_split;
  const int ke = min(kb + p.k_split, p.K);   // K and k_split are multiples of 32: whole stages
  const int nk = (ke - kb) / kBK;

  // ranges end at the tile's last row: rows past M / N read as zero
  const int rows_a = min(BM, p.M - m0);
  const int rows_w = min(BN, p.N - n0);
  const __amdgpu_buffer_rsrc_t ares = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(reinterpret_cast<const float*>(p.a) + (size_t)m0 * p.lda + kb), 0,
      ((rows_a - 1) * (int)p.lda + ke - kb) * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(reinterpret_cast<const float*>(p.w) + (size_t)n0 * p.K + kb), 0,
      ((rows_w - 1) * p.K + ke - kb) * 4, 0x00020000);
  // Unit i of a thread: row tid / 4 + i NT / 4, chunk tid % 4: elements 4 c .. 4 c
  // + 3 and 16 + 4 c .. of the stage's 32 (any order of K will do that A and W
  // share), so a load covers 64 contiguous bytes of a row.
  const int urow = tid >> 2, uch = tid & 3;
  const int va = urow * (int)p.lda * 4 + uch * 16, sa = NT / 4 * (int)p.lda * 4;
  const int vw = urow * p.K * 4 + uch * 16, sw = NT / 4 * p.K * 4;
  constexpr int LU = LA + LW;
  auto gload = [&](int kt, u32x4 (&r)[LU][2]) {   // stages past the last re-read it
    const int o = min(kt, nk - 1) * kBK * 4;
#pragma unroll
    for (int i = 0; i < LU; ++i)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        r[i][u] = i < LA ? buffer_load16(ares, va + i * sa + 64 * u, o) : buffer_load16(wres, vw + (i - LA) * sw + 64 * u, o);
  };
  // split unit i and write its parts
  auto put = [&](const u32x4 (&r)[LU][2], int i) {
    const int row = i < LA ? urow + i * (NT / 4) : BM + urow + (i - LA) * (NT / 4);
    u32x4 s[3];
    split8(as_f32x4(r[i][0]), as_f32x4(r[i][1]), s);
    uint8_t* d = lds + row * kRowBytes + ((uch ^ part_row_perm(row)) << 4);
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4*>(d + q * PLANE) = s[q];
  };

  f32x4 acc[MBW][NB];
#pragma unroll
  for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int wcol = SPREAD ? 16 * (col >> 2) + (col & 3) : col;   // W row of block nb: wcol + nb * (SPREAD ? 4 : 16)
  int fw_at[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int r = BM + wn * 64 + wcol + nb * (SPREAD ? 4 : 16);
    fw_at[nb] = r * kRowBytes + ((g ^ part_row_perm(r)) << 4);
  }
  int fa_at[MBW];
#pragma unroll
  for (int mb = 0; mb < MBW; ++mb) {
    const int r = (wm * MBW + mb) * 16 + col;
    fa_at[mb] = r * kRowBytes + ((g ^ part_row_perm(r)) << 4);
  }

  u32x4 r[LU][2];
  gload(0, r);
  for (int kt = 0; kt < nk; ++kt) {
    if (kt > 0) lds_barrier();         // the previous stage has been read
#pragma unroll
    for (int i = 0; i < LU; ++i) put(r, i);
    gload(kt + 1, r);                  // in flight while this stage multiplies
    lds_barrier();
    u32x4 fa[MBW][3];
#pragma unroll
    for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
      for (int q = 0; q < 3; ++q) fa[mb][q] = *reinterpret_cast<const u32x4*>(lds + fa_at[mb] + q * PLANE);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      u32x4 fw[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) fw[q] = *reinterpret_cast<const u32x4*>(lds + fw_at[nb] + q * PLANE);
      // A stage's products start from zero and join the sum in one fp32 add:
      // added one by one, the small ones would fall below the rounding of a sum
      // of many stages, and as they have the sign of the product, never cancel.
      f32x4 part[MBW];
#pragma unroll
      for (int q = 0; q < kSplitProducts; ++q)
#pragma unroll
        for (int mb = 0; mb < MBW; ++mb)
          part[mb] = mfma16x16x32<__bf16>(fw[kSplitA[q]], fa[mb][kSplitB[q]], q ? part[mb] : f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int mb = 0; mb < MBW; ++mb) acc[mb][nb] += part[mb];
    }
  }

  // Infinities, NaN, operands of 2^104 and results of 2^80 do not split: a wave
  // with a result that is not finite recomputes its part from fp32 products.
  bool finite = true;
#pragma unroll
  for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
      for (int i = 0; i < 4; ++i) finite = finite && fabsf(acc[mb][nb][i]) < __builtin_inff();
      acc[mb][nb] *= kSplitUnscale;
    }
  if (__builtin_amdgcn_ballot_w64(!finite) != 0) {
#pragma unroll
    for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < ke - kb; k += 4) {
      float w[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        w[nb] = u32_as_f32(__builtin_amdgcn_raw_buffer_load_b32(
            wres, ((wn * 64 + wcol + nb * (SPREAD ? 4 : 16)) * p.K + g) * 4, k * 4, 0));
#pragma unroll
      for (int mb = 0; mb < MBW; ++mb) {
        const float a = u32_as_f32(__builtin_amdgcn_raw_buffer_load_b32(
            ares, (((wm * MBW + mb) * 16 + col) * (int)p.lda + g) * 4, k * 4, 0));
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[nb], a, acc[mb][nb], 0, 0, 0);
      }
    }
  }
  tile_epilogue<float, EPI, MBW>(p, acc, m0 + wm * 16 * MBW, n0 + wn * 64, split, lane);
}

// Time model of a tile shape, in microseconds per stage of 32 K elements with n
// work-groups on a CU: `alone` for one, start + each * n for several.  MI355X,
// K 1024 .. 16384, M 65 .. 512.
struct TileShapeF32 {
  int bm, bn;
  double alone, start, each;
};
constexpr TileShapeF32 kTileShapesF32[] = {{128, 128, 1.68, 0.0, 1.35}, {64, 128, 1.15, 0.25, 0.75}};

static double tile_cost_f32(const TileShapeF32& s, int M, int N, int K, int splits) {
  const long long tiles = (long long)((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn) * splits;
  const double per_cu = (double)((tiles + 255) / 256);
  const double stages = (double)((K / splits + kBK - 1) / kBK) + 2.0;   // + fill and epilogue
  return stages * std::max(s.alone, s.start + s.each * per_cu);
}

int tile_linear_f32_shape(int M, int N, int K, int splits, double* cost) {
  const double a = tile_cost_f32(kTileShapesF32[0], M, N, K, splits);
  const double b = tile_cost_f32(kTileShapesF32[1], M, N, K, splits);
  if (cost) *cost = std::min(a, b);
  return b < a ? 1 : 0;
}

// The same with what lies around the stages (within 15% of the measured time, M 65 .. 512).
double tile_linear_f32_us(int M, int N, int K, int splits) {
  double c;
  tile_linear_f32_shape(M, N, K, splits, &c);
  return 2.1 + 1.15 * c;
}

int tile_linear_f32_k_split(int M, int N, int K) {
  double best = 0.0;
  int ks = (K + 31) / 32 * 32;
  for (int splits = 1; splits <= 8 && (splits == 1 || K / splits >= 256); splits *= 2) {
    double c;
    tile_linear_f32_shape(M, N, K, splits, &c);
    c += (splits - 1) * ((double)M * N * 1e-6 + 0.25);   // the partials, read back by the consumer
    if (splits == 1 || c < best) {
      best = c;
      if (splits > 1) ks = ((K + splits - 1) / splits + 63) / 64 * 64;
    }
  }
  return ks;
}

bool tile_linear_f32_supported(const LinearParams& p) {
  // 32-bit offsets inside a tile, and threads of the grid
  const long long tiles = (long long)((p.M + 63) / 64) * ((p.N + 127) / 128) * ((p.K + p.k_split - 1) / p.k_split);
  return std::max<long long>(p.lda, p.K) * 4 * 128 < (1LL << 31) && tiles <= 1 << 23;
}

template <int MBW, int WM, int WN, int WPE>
static void launch_tile_f32(const LinearParams& p, int epi, int splits, hipStream_t s) {
  constexpr int BM = 16 * MBW * WM, BN = 64 * WN;
  const dim3 grid((unsigned)(((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN) * splits)), block(64 * WM * WN);
  if (epi == kEpiPartial) hipLaunchKernelGGL((tile_linear_f32_kernel<kEpiPartial, MBW, WM, WN, WPE>), grid, block, 0, s, p);
  else if (epi == kEpiSwiglu) hipLaunchKernelGGL((tile_linear_f32_kernel<kEpiSwiglu, MBW, WM, WN, WPE>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((tile_linear_f32_kernel<kEpiLogits, MBW, WM, WN, WPE>), grid, block, 0, s, p);
}

void launch_tile_linear_f32(const LinearParams& p, int epi, hipStream_t s) {
  const int splits = (p.K + p.k_split - 1) / p.k_split;
  if (tile_linear_f32_shape(p.M, p.N, p.K, splits, nullptr) == 0) launch_tile_f32<4, 2, 2, 2>(p, epi, splits, s);   // 48 KB of LDS, two per CU
  else launch_tile_f32<2, 2, 2, 4>(p, epi, splits, s);                                             // 36 KB, four
}

}  // namespace tv
