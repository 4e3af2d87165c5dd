// Y = A W^T for many rows of A (prompt passes): LDS-tiled MFMA product, fp16 / bf16.
//
// Both operands are K-major, as the model stores them.  A work-group computes a
// BM x BN tile of Y; each stage of 128 bytes of K per row is loaded straight
// into LDS (buffer_load ... lds: no staging registers, no LDS writes), S stages
// deep.  LDS rows are 128 bytes and unpadded (such a load writes 1 KB
// contiguously), so the 16-byte chunks of a row are XOR-permuted: fragment
// reads touch every bank once (SQ_LDS_BANK_CONFLICT 0).
//
// What bounds it: a CU reads (BM / 16 MBW-row waves + BN / 64-column waves)
// fragments from LDS per stage and writes the stage itself; for a 256 x 256
// tile by eight 128 x 64 waves that is about 2050 LDS clocks against 2048 of
// matrix work, so the two have to overlap almost perfectly.  Hence the shape
// of a half stage (`half` below): between every NB products stand the reads of
// one or two fragments of the next half stage and one load into LDS, pinned in
// that order, and the barrier is passed with a half stage of products still
// to issue.  MI355X, bf16: 2048 x 32768 x 4096 448 us (1.23 PFLOP/s; 471 us
// with the reads and loads in front of the products, 500 us without fragment
// double buffering); 2048 x 4096 x 16384 in two K splits 217 us.  64-byte
// stage rows with twice the stages (more bytes in flight) were 4% slower for
// this tile and 25% for the smaller ones; starting work-groups at different
// stages, to spread the channels they read, was 2-5% slower.
#include "tv_common.h"
#include "tv_dense.h"
#include "tv_linear.h"
#include "tv_tile_dma.h"
#include "tv_tile_epilogue.h"

#include <algorithm>

namespace tv {

namespace {

constexpr int kStageBytes = 128;   // K bytes of one row per stage

// 16-byte chunk c of tile row r sits at slot c ^ tile_row_perm(r).  Two rows
// cover the 64 banks; over the 16 rows of a fragment read (plain: rows
// 16 b .. 16 b + 15; SPREAD: rows 16 a + 4 b + i, a and i = 0..3) the pairs
// (r & 1, perm) are distinct.
template <bool SPREAD> __device__ __forceinline__ int tile_row_perm(int r) {
  if constexpr (SPREAD) return ((r >> 1) & 1) | (((r >> 4) & 3) << 1);
  else return (r >> 1) & 7;
}

}  // namespace

// WM x WN waves, each 16 MBW rows of A (tokens) by 64 rows of W (features).
template <typename T, int EPI, int MBW, int WM, int WN, int S>
__global__ void __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(2)))
tile_linear_kernel(const LinearParams p) {
  constexpr int NW = WM * WN;
  constexpr int BM = 16 * MBW * WM;
  constexpr int BN = 64 * WN;
  constexpr int NB = 4;                // 16-feature blocks of a wave
  constexpr int ES = (int)sizeof(T);
  constexpr int BK = kStageBytes / ES;
  constexpr int LA = BM / 8 / NW;      // A loads per wave and stage (8 rows each)
  constexpr int LW = BN / 8 / NW;
  constexpr int L = LA + LW;
  constexpr int STAGE = (BM + BN) * kStageBytes;
  // SwiGLU: MFMA row 4 a + i of block nb is W row 16 a + 4 nb + i of the wave's
  // 64, so a lane ends up with 16 consecutive features: one 16-byte store.
  constexpr bool SPREAD = EPI == kEpiSwiglu;
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "whole loads per wave");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[S * STAGE];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int g = lane >> 4;
  const int col = lane & 15;
  const int wm = wave / WN, wn = wave % WN;

  // Work-group -> (split, n tile, m tile).  Work-groups are dealt to the 8 XCDs
  // round-robin; each XCD takes a contiguous run of tiles, m tiles innermost
  // (up to 8), so the work-groups that share rows of W share an L2.
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
  const int ke = min(kb + p.k_split, p.K);
  const int nk = (ke - kb + BK - 1) / BK;

  // Loads past a resource's range return zeros: rows past M / N and K past the
  // split are sent out of range by bit 31 of their offset (a tile spans less
  // than 2^31 bytes, tile_linear_supported).
  const int rows_a = min(BM, p.M - m0);
  const int rows_w = min(BN, p.N - n0);
  const u32x4 ares = rsrc_words(reinterpret_cast<const T*>(p.a) + (size_t)m0 * p.lda + kb,
                                (unsigned long long)((long long)(rows_a - 1) * p.lda + (ke - kb)) * ES);
  const u32x4 wres = rsrc_words(reinterpret_cast<const T*>(p.w) + (size_t)n0 * p.K + kb,
                                (unsigned long long)((long long)(rows_w - 1) * p.K + (ke - kb)) * ES);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;

  // load i of a wave covers tile rows 8 (wave + NW i) .. + 7: lane -> row
  // lane / 8, slot lane % 8
  uint32_t va[LA], vw[LW];
  const int lrow = lane >> 3;
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int row = 8 * (wave + NW * i) + lrow;
    va[i] = (uint32_t)(row * (int)p.lda * ES + 16 * ((lane & 7) ^ tile_row_perm<false>(row)));
    if (row >= rows_a) va[i] |= 0x80000000u;
  }
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int row = 8 * (wave + NW * i) + lrow;
    vw[i] = (uint32_t)(row * p.K * ES + 16 * ((lane & 7) ^ tile_row_perm<SPREAD>(row)));
    if (row >= rows_w) vw[i] |= 0x80000000u;
  }
  // Before the load of a short last stage, and of stages past the last: send
  // the chunks past the K range out of range.
  const int tail = (ke - kb) % BK * ES / 16;   // 16-byte chunks of a short last stage (0: whole)
  int issued = 0;                              // stages requested so far
  auto clip = [&]() {
    if (issued < nk - (tail ? 1 : 0)) return;
    const int limit = issued < nk ? tail : 0;
#pragma unroll
    for (int i = 0; i < LA; ++i)
      if (((lane & 7) ^ tile_row_perm<false>(8 * (wave + NW * i) + lrow)) >= limit) va[i] |= 0x80000000u;
#pragma unroll
    for (int i = 0; i < LW; ++i)
      if (((lane & 7) ^ tile_row_perm<SPREAD>(8 * (wave + NW * i) + lrow)) >= limit) vw[i] |= 0x80000000u;
  };
  // load i (of L) of the next stage into the stage buffer at `stage`
  auto load = [&](uint32_t stage, int i) {
    const uint32_t base = lds0 + stage + wave * 1024;
    if (i < LA) {
      load_lds16(ares, base + NW * 1024 * i, va[i]);
      va[i] += kStageBytes;
    } else if (i < L) {
      load_lds16(wres, base + BM * kStageBytes + NW * 1024 * (i - LA), vw[i - LA]);
      vw[i - LA] += kStageBytes;
    }
  };

  f32x4 acc[MBW][NB];
#pragma unroll
  for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};

  // fragment i of a half stage ks: the NB blocks of W, then the MBW blocks of A
  const int wrow = SPREAD ? 16 * (col >> 2) + (col & 3) : col;
  int oa[2], ow[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    oa[ks] = (wm * 16 * MBW + col) * kStageBytes + (((4 * ks + g) ^ tile_row_perm<false>(col)) << 4);
    ow[ks] = (BM + wn * 64 + wrow) * kStageBytes + (((4 * ks + g) ^ tile_row_perm<SPREAD>(wrow)) << 4);
  }
  auto read = [&](uint32_t stage, int ks, int i, u32x4 (&fw)[NB], u32x4 (&fa)[MBW]) {
    const uint8_t* st = lds + stage;
    if (i < NB) fw[i] = *reinterpret_cast<const u32x4*>(st + ow[ks] + i * (SPREAD ? 4 : 16) * kStageBytes);
    else if (i < NB + MBW) fa[i - NB] = *reinterpret_cast<const u32x4*>(st + oa[ks] + (i - NB) * 16 * kStageBytes);
  };
  // The products of one half stage in MBW groups; in front of each group a
  // share of the next half stage's fragment reads and (LOAD) of the loads that
  // refill the buffer `fill`.
  auto half = [&](auto loads, const u32x4 (&fw)[NB], const u32x4 (&fa)[MBW], uint32_t next, int ks,
                  u32x4 (&fwn)[NB], u32x4 (&fan)[MBW], uint32_t fill) {
    constexpr bool LOAD = decltype(loads)::value;
    constexpr int RG = (NB + MBW + MBW - 1) / MBW;
    constexpr int LG = (L + MBW - 1) / MBW;
#pragma unroll
    for (int mb = 0; mb < MBW; ++mb) {
#pragma unroll
      for (int j = 0; j < RG; ++j) read(next, ks, mb * RG + j, fwn, fan);
      if constexpr (LOAD) {
#pragma unroll
        for (int j = 0; j < LG; ++j) load(fill, mb * LG + j);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = mfma_frag<T>(fw[nb], fa[mb], acc[mb][nb]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (LOAD) ++issued;
  };

#pragma unroll
  for (int i = 0; i < S; ++i) {
    clip();
#pragma unroll
    for (int j = 0; j < L; ++j) load(i * STAGE, j);
    ++issued;
  }
  wait_vmcnt<(S - 1) * L>();
  lds_barrier();
  u32x4 fw0[NB], fa0[MBW], fw1[NB], fa1[MBW];
#pragma unroll
  for (int i = 0; i < NB + MBW; ++i) read(0, 0, i, fw0, fa0);
  // Stage kt: its first half multiplies while its second half is read; then
  // every wave has read the stage (lds_barrier waits for the reads) and stage
  // kt + 1 has landed, so the second half multiplies while the buffer is
  // refilled with stage kt + S and the next stage's first half is read.
  uint32_t cur = 0;
  for (int kt = 0; kt < nk; ++kt) {
    clip();
    half(std::false_type{}, fw0, fa0, cur, 1, fw1, fa1, 0);
    wait_vmcnt<(S - 2) * L>();
    lds_barrier();
    const uint32_t next = cur == (S - 1) * STAGE ? 0 : cur + STAGE;
    half(std::true_type{}, fw1, fa1, next, 0, fw0, fa0, cur);
    cur = next;
  }
  wait_vmcnt<0>();   // loads still under way write (zeros) to this work-group's LDS

  tile_epilogue<T, EPI, MBW>(p, acc, m0 + wm * 16 * MBW, n0 + wn * 64, split, lane);
}

// Time model of a tile shape, in microseconds (MI355X, fp16 / bf16): a stage of
// a lone work-group on its CU takes `alone`, of several resident ones `shared`
// each.  From products timed alone at K 2048 .. 16384 with 30 to 4096 tiles.  Over
// 225 products (M 65 .. 2048, N 512 .. 32768, K 256 .. 16384, weights from HBM) what
// it picks is within 6% of the fastest shape and split for 92%, at worst 1.4x
// (777 x 2816 x 1024, 192 x 11264 x 2048).  Inside a prompt pass the same products
// take longer than alone (1000 rows, TinyLlama: QKV 31 us, Wo 17, W2 42, W13 55, by
// the model 22, 12, 31 and 49).
struct TileShape {
  int bm, bn;
  double alone, shared;
};
constexpr TileShape kTileShapes[] = {{256, 256, 1.35, 1.45}, {128, 128, 0.62, 0.50}, {64, 128, 0.34, 0.34}};
constexpr int kTileCus = 256;

static double tile_cost(const TileShape& s, int M, int N, int K, int splits) {
  const long long tiles = (long long)((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn) * splits;
  const double per_cu = (double)((tiles + kTileCus - 1) / kTileCus);
  const double stages = (double)((K / splits + 63) / 64) + 4.0;   // + pipeline fill and epilogue
  return stages * std::max(s.alone, s.shared * per_cu);
}

int tile_linear_shape(int M, int N, int K, int splits, double* cost) {
  int best = 0;
  double bc = 0.0;
  for (int i = 0; i < 3; ++i) {
    const double c = tile_cost(kTileShapes[i], M, N, K, splits);
    if (i == 0 || c < bc) best = i, bc = c;
  }
  if (cost) *cost = bc;
  return best;
}

// The same with what lies around the stages (most within 15% of the measured time, M 65 .. 2048).
double tile_linear_us(int M, int N, int K, int splits) {
  double c;
  tile_linear_shape(M, N, K, splits, &c);
  return 2.4 + 1.2 * c;
}

// Splits of K for a product whose consumer sums partials: the cheapest of 1, 2,
// 4 and 8 with at least four stages each, charged with the fp32 partials that
// the consumer reads back (about 4 TB/s) and half a microsecond per doubling.
int tile_linear_k_split(int M, int N, int K) {
  double best = 0.0;
  int ks = (K + 31) / 32 * 32;
  for (int splits = 1; splits <= 8 && (splits == 1 || K / splits >= 256); splits *= 2) {
    double c;
    tile_linear_shape(M, N, K, splits, &c);
    c += (splits - 1) * ((double)M * N * 1e-6 + 0.25);
    if (splits == 1 || c < best) {
      best = c;
      if (splits > 1) ks = ((K + splits - 1) / splits + 63) / 64 * 64;
    }
  }
  return ks;
}

// 32-bit offsets inside a tile, and threads of the grid.
bool tile_linear_supported(const LinearParams& p) {
  const long long tiles = (long long)((p.M + 63) / 64) * ((p.N + 127) / 128) * ((p.K + p.k_split - 1) / p.k_split);
  return std::max<long long>(p.lda, p.K) * 2 * 256 < (1LL << 31) && tiles <= 1 << 23;
}

template <typename T, int MBW, int WM, int WN, int S>
static void launch_tile(const LinearParams& p, int epi, int splits, hipStream_t s) {
  constexpr int BM = 16 * MBW * WM, BN = 64 * WN;
  const dim3 grid((unsigned)(((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN) * splits)), block(64 * WM * WN);
  switch (epi) {
    case kEpiPartial:
      hipLaunchKernelGGL((tile_linear_kernel<T, kEpiPartial, MBW, WM, WN, S>), grid, block, 0, s, p);
      break;
    case kEpiSwiglu:
      hipLaunchKernelGGL((tile_linear_kernel<T, kEpiSwiglu, MBW, WM, WN, S>), grid, block, 0, s, p);
      break;
    default: hipLaunchKernelGGL((tile_linear_kernel<T, kEpiLogits, MBW, WM, WN, S>), grid, block, 0, s, p);
  }
}

template <typename T> static void launch_tile_t(const LinearParams& p, int epi, hipStream_t s) {
  const int splits = (p.K + p.k_split - 1) / p.k_split;
  switch (tile_linear_shape(p.M, p.N, p.K, splits, nullptr)) {
    case 0: launch_tile<T, 8, 2, 4, 2>(p, epi, splits, s); break;   // 256 x 256, 128 KB of LDS, one per CU
    case 1: launch_tile<T, 4, 2, 2, 2>(p, epi, splits, s); break;   // 128 x 128, 64 KB, two per CU
    default: launch_tile<T, 2, 2, 2, 3>(p, epi, splits, s);         // 64 x 128, 72 KB, two per CU
  }
}

void launch_tile_linear(const LinearParams& p, int epi, int dtype, hipStream_t s) {
  if (dtype == kF16) launch_tile_t<_Float16>(p, epi, s);
  else launch_tile_t<__bf16>(p, epi, s);
}

}  // namespace tv
