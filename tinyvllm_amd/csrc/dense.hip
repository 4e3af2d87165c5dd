// Dense kernels of the batched decode step (gfx950): the weight-streaming
// products, RMSNorm with the residual add, RoPE with the K/V cache write, and
// greedy sampling.  Semantics follow tinyvllm/model/llama.py:
//   RMSNorm          x * rsqrt(mean(x^2) + eps) * w              llama.py:14-23
//   RoPE table       cos/sin(p * theta^(-2i/D))                  llama.py:26-31
//   RoPE             interleaved pairs (2i, 2i+1)                llama.py:34-55
//   SwiGLU           w2(silu(w1 x) * w3 x)                       llama.py:220-221
//   greedy sampling  argmax over the vocabulary (first maximum)  sampling.py:131-134
//
// linear_kernel computes Y = A W^T for a skinny A (the decode batch, 64 rows per
// work-group; at most 16 rows: few_linear_kernel; more than 64: mostly
// tile_linear.hip, tile_linear_f32.hip) against a weight matrix W [N, K] that is
// streamed from HBM once per 64 rows.  Each of the 4 waves of a work-group owns 16 rows of W and all
// 64 rows of A; A is staged in LDS per 512-byte-wide K chunk (256 fp16/bf16 or
// 128 fp32 elements) and shared by the waves.  fp32 runs the same byte layout
// on v_mfma_f32_16x16x4_f32, four of them per 16-byte fragment pair.  W rows are the MFMA A operand (lane = output feature), A^T the B
// operand (lane = token), so a lane ends up holding 4 consecutive output
// features of one token: the layout the fused epilogues want.
#include "tv_common.h"
#include "tv_dense.h"
#include "tv_linear.h"
#include "tv_tile_dma.h"

#include <algorithm>

namespace tv {

// ---------------------------------------------------------------------------
// Y = A W^T
// ---------------------------------------------------------------------------

constexpr int kLinearMinBlocks = 1;    // occupancy hint of the product kernel
constexpr int kLinearWStages = 2;      // W chunks in registers: in flight + the one multiplied
// A chunks requested ahead of the one being multiplied.  Two ahead measured
// slower for every product of the TinyLlama batch-64 decode step (64-step
// graph: 1468 us/step at one ahead; two ahead for the SwiGLU product 1488, for
// the split-K partial products 1485, for both 1505), so one it is.
constexpr int kLinearAStages = 1;

constexpr int gcd_c(int a, int b) { return b == 0 ? a : gcd_c(b, a % b); }
constexpr int lcm3(int a, int b, int c) {
  const int ab = a / gcd_c(a, b) * b;
  return ab / gcd_c(ab, c) * c;
}

// Epilogue of the skinny products: lane (wave, g, col) holds acc[mb][i] =
// Y[m0 + 16 mb + col][n_wave + 4 g + i].  sk: 2 KB of LDS per 16 rows for the
// argmax exchange (logits), free to reuse once every wave reaches this point.
template <typename T, int EPI, int MB>
__device__ __forceinline__ void linear_epilogue(const LinearParams& p, const f32x4 (&acc)[MB], int n_wave, int m0,
                                                int split, int ntile, int wave, int tid, unsigned long long* sk) {
  constexpr int ROWS = 16 * MB;
  const int lane = tid & 63;
  const int g = lane >> 4;
  const int col = lane & 15;
  const int n = n_wave + 4 * g;
  if constexpr (EPI == kEpiPartial) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int m = m0 + mb * 16 + col;
      if (m < p.M && n < p.N)
        *reinterpret_cast<f32x4*>(p.part + ((size_t)split * p.M + m) * p.N + n) = acc[mb];
    }
  } else if constexpr (EPI == kEpiSwiglu) {
    // rows 4j, 4j+1 of W are w1 rows 2j, 2j+1; rows 4j+2, 4j+3 the matching w3 rows
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int m = m0 + mb * 16 + col;
      if (m < p.M && n < p.N) {
        const f32x4 v = acc[mb];
        store2<T>(p.out, (size_t)m * p.ldo + (n >> 1), silu(v[0]) * v[2], silu(v[1]) * v[3]);
      }
    }
  } else {
    lds_barrier();   // sk reuses LDS of the main loop: [16 (wave, g)][ROWS]
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int m = m0 + mb * 16 + col;
      const f32x4 v = acc[mb];
      if (p.out && m < p.M && n < p.N)
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.out) + (size_t)m * p.ldo + n) = v;
      unsigned long long best = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n + i < p.N) best = max(best, argmax_key(v[i], n + i));
      sk[(wave * 4 + g) * ROWS + mb * 16 + col] = best;
    }
    lds_barrier();
    if (tid < ROWS && p.keys && m0 + tid < p.M) {
      unsigned long long best = sk[tid];
#pragma unroll
      for (int j = 1; j < 16; ++j) best = max(best, sk[j * ROWS + tid]);
      p.keys[(size_t)ntile * p.M + m0 + tid] = best;
    }
  }
}

// TAIL: K ranges that end inside a chunk.  What lies past them in W's rows (other
// splits, the next row) is then not read: a product with a zero of A would make
// NaN of an infinity or NaN there.
template <typename T, int EPI, bool TAIL>
__global__ void __launch_bounds__(256, kLinearMinBlocks) linear_kernel(const LinearParams p) {
  // LDS in 16-bit units; a chunk row is 512 bytes of K at a 544-byte pitch (an
  // odd multiple of 32 modulo 256: conflict-free 16-byte reads)
  constexpr int KP = 256 + 16;
  constexpr int KC = 512 / (int)sizeof(T);   // K elements per chunk
  constexpr int VE = 16 / (int)sizeof(T);    // K elements per 16-byte vector
  __shared__ __attribute__((aligned(16))) uint16_t sa[2][kLinBM * KP];   // A chunk, double-buffered

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform: W resource in SGPRs
  const int lane = tid & 63;
  const int g = lane >> 4;
  const int col = lane & 15;
  // grid (splits, n tiles, m tiles): consecutive work-groups take different
  // K splits of one n tile, and each n tile starts its chunk sequence at a
  // different chunk, so the work-groups in flight read different column
  // ranges of W.  (With the row pitch of W a power of two, work-groups that
  // march through the same columns in step all hit the same HBM channels.)
  const int split = blockIdx.x;
  const int ntile = blockIdx.y;
  const int n_wave = ntile * kLinBN + wave * 16;
  const int m0 = blockIdx.z * kLinBM;
  const int kb = split * p.k_split;
  const int ke = min(kb + p.k_split, p.K);
  const int nc = (ke - kb + KC - 1) / KC;
  const int rot = ntile % nc;
  auto chunk_of = [&](int i) { const int c = i + rot; return c < nc ? c : c - nc; };

  // Buffer loads: reads past the end of W (rows >= N) or of A (rows >= M)
  // return zero in hardware, so no address is clamped.  The row part of every
  // offset goes in the VGPR offset: the hardware range check covers the VGPR
  // and instruction offsets, not the scalar one.
  // (16 rows of W, so that offsets from 2^31 on are past its range)
  const unsigned w_rows = __builtin_amdgcn_readfirstlane(min(max(p.N - n_wave, 0), 16));
  const __amdgpu_buffer_rsrc_t wres = make_rsrc(reinterpret_cast<const T*>(p.w) + (size_t)min(n_wave, p.N) * p.K,
                                                (unsigned long long)w_rows * (unsigned)p.K * sizeof(T));
  const __amdgpu_buffer_rsrc_t ares = make_rsrc(reinterpret_cast<const T*>(p.a) + (size_t)m0 * p.lda,
                                                (unsigned long long)max(p.M - m0, 0) * p.lda * sizeof(T));
  const int w_voff = (col * p.K + kb) * (int)sizeof(T) + 16 * g;
  const int a_voff = ((tid >> 5) * (int)p.lda + kb) * (int)sizeof(T) + 16 * (tid & 31);
  const int a_rows8 = 8 * (int)p.lda * (int)sizeof(T);   // byte step between the 8 rows a thread loads

  // W: lane (row col, k group g) reads 16 bytes per 64-byte k step.
  // i is the position in this work-group's chunk sequence; positions past the
  // last chunk load zeros, so padding steps add nothing.
  auto loadW = [&](int i, u32x4 (&r)[8]) {
    const int c = chunk_of(min(i, nc - 1));
    const int off = i < nc ? w_voff + c * 512 : (int)0x80000000;
    const int left = (ke - kb) * (int)sizeof(T) - c * 512;   // bytes of a row from this chunk on
#pragma unroll
    for (int s = 0; s < 8; ++s) r[s] = buffer_load16(wres, !TAIL || 64 * s < left ? off + 64 * s : (int)0x80000000, 0);
  };
  // A chunk: 64 rows x 32 vectors of 16 bytes; thread tid loads vector
  // tid % 32 of rows tid / 32 + 8 i.  Columns past the split are zeroed when
  // stored to LDS (not at load time, so the loads stay in flight while the
  // previous chunk computes).
  auto loadA = [&](int i, u32x4 (&r)[8], bool& valid) {
    const int c = chunk_of(min(i, nc - 1));
    valid = i < nc && kb + c * KC + VE * (tid & 31) < ke;
    const int off = a_voff + c * 512;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = buffer_load16(ares, off + i * a_rows8, 0);   // row in the range-checked offset
  };
  auto storeA = [&](const u32x4 (&r)[8], bool valid, int buf) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      *reinterpret_cast<u32x4*>(&sa[buf][((tid >> 5) + 8 * i) * KP + 8 * (tid & 31)]) = valid ? r[i] : u32x4{0, 0, 0, 0};
  };

  f32x4 acc[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  // All 8 k steps run even on a partial chunk: the A rows there are zero.
  // The B fragments of step s + 1 are read from LDS while step s multiplies.
  auto compute = [&](const u32x4 (&r)[8], int buf) {
    u32x4 b[2][4];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) b[0][mb] = *reinterpret_cast<const u32x4*>(&sa[buf][(mb * 16 + col) * KP + 8 * g]);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      if (s + 1 < 8) {
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
          b[(s + 1) & 1][mb] = *reinterpret_cast<const u32x4*>(&sa[buf][(mb * 16 + col) * KP + 32 * (s + 1) + 8 * g]);
      }
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) acc[mb] = mfma_frag<T>(r[s], b[s & 1][mb], acc[mb]);
    }
  };

  constexpr int NWS = kLinearWStages;
  constexpr int NAS = kLinearAStages;     // A chunks in flight in registers
  constexpr int U = lcm3(NWS, NAS, 2);     // loop unroll: every stage / buffer index compile-time
  u32x4 w[NWS][8], ar[NAS][8];
  bool av[NAS];
  if (nc == 1) {
    loadW(0, w[0]);
    loadA(0, ar[0], av[0]);
    storeA(ar[0], av[0], 0);
    lds_barrier();
    compute(w[0], 0);
  } else if (NWS >= 2 && nc == 2) {
    // both chunks requested at once, one in each LDS buffer: one round trip
    // instead of the pipeline's two (the Wqkv product of the decode step)
    u32x4 a1[8];
    bool v1;
    loadW(0, w[0]);
    loadW(1, w[1 % NWS]);
    loadA(0, ar[0], av[0]);
    loadA(1, a1, v1);
    storeA(ar[0], av[0], 0);
    storeA(a1, v1, 1);
    lds_barrier();
    compute(w[0], 0);
    compute(w[1 % NWS], 1);
  } else {
#pragma unroll
    for (int i = 0; i < NWS - 1; ++i) loadW(i, w[i]);
#pragma unroll
    for (int i = 0; i < NAS; ++i) loadA(i, ar[i], av[i]);
    // Step j multiplies chunk j: W of chunks j + 1 .. j + NWS - 1 and A of
    // chunks j + 1 .. j + NAS are in flight meanwhile.  A goes through two
    // LDS buffers, so one barrier per step orders both its store and the
    // reuse of the buffer two steps later.  The loads are unconditional and
    // the step count is padded to a multiple of U (padding steps multiply
    // zero A rows), so the loop body has no exit and the compiler waits for
    // exactly the chunk it needs.  (sched_barrier keeps each prefetch issued
    // before the waits that follow.)
    const int ncp = (nc + U - 1) / U * U;
    for (int c = 0; c < ncp; c += U) {
#pragma unroll
      for (int j = 0; j < U; ++j) {
        loadW(c + j + NWS - 1, w[(j + NWS - 1) % NWS]);
        __builtin_amdgcn_sched_barrier(0);
        storeA(ar[j % NAS], av[j % NAS], j & 1);
        lds_barrier();
        loadA(c + j + NAS, ar[j % NAS], av[j % NAS]);
        __builtin_amdgcn_sched_barrier(0);
        compute(w[j % NWS], j & 1);
      }
    }
  }

  linear_epilogue<T, EPI, 4>(p, acc, n_wave, m0, split, ntile, wave, tid, reinterpret_cast<unsigned long long*>(&sa[0][0]));
}


// The product for at most kFewRows rows of A, where the time should be the
// stream of W.  Every wave has a ring of S stages in LDS, each 512 bytes of 16
// rows of W and of RA rows of A, filled by direct loads (512 contiguous bytes
// per row and instruction).  The ring is private to the wave, so no barrier
// stands between its loads.  KW = 4: a unit is 16 rows of W, whose stages the
// waves take in turn and sum through LDS, so even a product of 2048 features
// has a unit for every CU with few splits.  KW = 1: 64 rows, 16 per wave (the
// logits, whose argmax keys cover 64 features).  One work-group per CU walks
// the units; its loads run ahead across them.  The 64-row kernel spent its
// time on products for rows that are not there (fp32) and on one 64-row tile
// per work-group, 176 of them on 256 CUs.  W is read once and non-temporally:
// from HBM 3-8% faster (32000 x 2048 fp32 48.4 -> 43.7 us; fp16, 4 rows, 2560 x
// 2048 5.5 -> 5.1, 2048 x 5632 7.1 -> 6.6); weights that all stay in the 256 MB
// last-level cache (models of a few layers) lose 2-5% at 4 rows, up to 20% at 16.  MI355X, 4 rows, against the
// 64-row kernel: 11264 x 2048 fp32 47 -> 19.0 us (4.9 TB/s), 32000 x 2048 87 ->
// 43.7 (6.0), 2048 x 5632 26 -> 11.5; fp16 15.9 -> 10.8, 31.4 -> 22.7, 9.4 ->
// 7.0.  At 16 rows, fp16: 16.4 -> 12.7, 31.7 -> 24.5, 9.9 -> 8.1.  Rejected: A
// held in LDS with W in registers (fp32 25.9 / 62.9 / 12.6 us), both in
// registers (29.1 / 56.0 / 13.8); there an instruction reads 64 bytes of 16 rows.
template <typename T, int EPI, int KW, int RA, int S>
__global__ void __launch_bounds__(256) few_linear_kernel(const LinearParams p) {
  constexpr int ES = (int)sizeof(T);
  constexpr int CB = kFewStage;
  constexpr int LW = 8, LA = RA / 2;   // loads per stage: two rows each
  constexpr int STAGE = (16 + RA) * CB;
  __shared__ __attribute__((aligned(1024))) uint8_t sm[4 * S * STAGE];
  __shared__ f32x4 red[2][256];        // sums of the waves (KW = 4), argmax keys (logits)

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int g = lane >> 4;
  const int col = lane & 15;
  const int kw = KW == 4 ? wave : 0;
  const int ntiles = (p.N + 64 / KW - 1) / (64 / KW);
  const int splits = (p.K + p.k_split - 1) / p.k_split;
  const int units = ntiles * splits;   // consecutive units: the splits of one n tile

  const uint32_t ring0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)sm + wave * S * STAGE;
  const uint8_t* const ring = sm + wave * S * STAGE;
  auto stages_of = [&](int split) {    // of this wave: kw, kw + KW, ...
    const int nc = (min(p.k_split, p.K - split * p.k_split) * ES + CB - 1) / CB;
    return (nc - kw + KW - 1) / KW;
  };

  // the unit that is being loaded
  struct Source {
    u32x4 wres, ares;
    int kbytes, nc, ni, rot, rows_w, i;
  } src;
  int lu = blockIdx.x;
  auto open = [&]() {
    const int ntile = lu / splits, split = lu - ntile * splits;
    const int kb = split * p.k_split;
    const int n_wave = KW == 4 ? ntile * 16 : ntile * 64 + wave * 16;
    src.kbytes = min(p.k_split, p.K - kb) * ES;
    src.nc = (src.kbytes + CB - 1) / CB;
    src.ni = stages_of(split);
    // n tiles start at scattered columns: with rows of W a power of two apart,
    // work-groups in step at one column keep to a few HBM channels (4096 x
    // 16384 fp32: 68.9 us from 16 starting columns, 49.3 from all; 53.7 at a
    // row of 17408, where the start does not matter)
    src.rot = (int)(((((uint32_t)ntile * 0x9E3779B1u) >> 16) * (uint32_t)src.nc) >> 16);
    // ranges end at the wave's last row; everything else (rows past N or M, K
    // past the split, stages past the last) is sent out of range by bit 31 and
    // reads zero
    src.rows_w = min(16, max(p.N - n_wave, 0));
    src.wres = rsrc_words(reinterpret_cast<const T*>(p.w) + (size_t)min(n_wave, p.N) * p.K + kb,
                          src.rows_w ? ((unsigned long long)src.rows_w * p.K - kb) * ES : 0);
    src.ares = rsrc_words(reinterpret_cast<const T*>(p.a) + kb,
                          ((unsigned long long)(p.M - 1) * p.lda + p.K - kb) * ES);
    src.i = 0;
  };
  // Load i of a stage covers rows 2 i and 2 i + 1: lane -> row lane / 32, slot
  // lane % 32; 16-byte chunk c of row r sits at slot c ^ r, so the 16 rows of
  // a fragment read fall on distinct banks.
  const int lrow = lane >> 5;
  auto load = [&](uint32_t base) {
    while (lu < units && src.i >= src.ni) {
      lu += gridDim.x;
      if (lu < units) open();
    }
    int c = kw + KW * src.i + src.rot;
    c = c < src.nc ? c : c - src.nc;
    const int left = lu < units ? src.kbytes - c * CB : 0;   // bytes of this stage
    ++src.i;
#pragma unroll
    for (int t = 0; t < LW; ++t) {
      const int r = 2 * t + lrow, o = 16 * ((lane & 31) ^ r);
      const bool in = o < left && r < src.rows_w;
      load_lds16_nt(src.wres, base + t * 1024, in ? (uint32_t)(r * p.K * ES + c * CB + o) : 0x80000000u);
    }
#pragma unroll
    for (int t = 0; t < LA; ++t) {
      const int r = 2 * t + lrow, o = 16 * ((lane & 31) ^ r);
      const bool in = o < left && r < p.M;
      load_lds16(src.ares, base + (LW + t) * 1024, in ? (uint32_t)(r * (int)p.lda * ES + c * CB + o) : 0x80000000u);
    }
  };

  const int ar = col & (RA - 1);       // columns past RA read copies; columns past M are dropped
  open();
#pragma unroll
  for (int j = 0; j < S; ++j) load(ring0 + j * STAGE);
  int at = 0, parity = 0;
  for (int u = blockIdx.x; u < units; u += gridDim.x) {
    const int ntile = u / splits, split = u - ntile * splits;
    const int ni = stages_of(split);
    f32x4 acc[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
    for (int i = 0; i < ni; ++i) {
      wait_vmcnt<(S - 1) * (LW + LA)>();
      const uint8_t* st = ring + at;
      u32x4 w[8], a[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        w[s] = *reinterpret_cast<const u32x4*>(st + col * CB + 16 * ((4 * s + g) ^ col));
        a[s] = *reinterpret_cast<const u32x4*>(st + (16 + ar) * CB + 16 * ((4 * s + g) ^ ar));
      }
      __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the stage is in registers, its buffer free
      load(ring0 + at);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < 8; ++s) acc[0] = mfma_frag<T>(w[s], a[s], acc[0]);
      at = at == (S - 1) * STAGE ? 0 : at + STAGE;
    }
    if constexpr (KW == 4) {
      // two buffers: a wave passes the next unit's barrier only after wave 0 has read this one's
      red[parity][tid] = acc[0];
      lds_barrier();
      if (wave == 0) {
        acc[0] = (red[parity][lane] + red[parity][64 + lane]) + (red[parity][128 + lane] + red[parity][192 + lane]);
        linear_epilogue<T, EPI, 1>(p, acc, ntile * 16, 0, split, ntile, wave, tid, nullptr);
      }
      parity ^= 1;
    } else {
      linear_epilogue<T, EPI, 1>(p, acc, ntile * 64 + wave * 16, 0, split, ntile, wave, tid,
                                 reinterpret_cast<unsigned long long*>(&red[0][0]));
    }
  }
  wait_vmcnt<0>();                     // loads still under way write zeros to the ring
}

template <typename T, int EPI> static void launch_few(const LinearParams& p, hipStream_t s) {
  constexpr int KW = EPI == kEpiLogits ? 1 : 4;
  const long long units = (long long)((p.N + 64 / KW - 1) / (64 / KW)) * ((p.K + p.k_split - 1) / p.k_split);
  const dim3 grid((unsigned)std::min<long long>(units, kFewWorkGroups));
  if (p.M <= 4) hipLaunchKernelGGL((few_linear_kernel<T, EPI, KW, 4, 3>), grid, dim3(256), 0, s, p);
  else hipLaunchKernelGGL((few_linear_kernel<T, EPI, KW, 16, 2>), grid, dim3(256), 0, s, p);
}

template <typename T, int EPI> static void launch_skinny(const LinearParams& p, hipStream_t s) {
  const dim3 grid((p.K + p.k_split - 1) / p.k_split, (p.N + kLinBN - 1) / kLinBN, (p.M + kLinBM - 1) / kLinBM);
  constexpr int KC = 512 / (int)sizeof(T);
  if (p.K % KC || (p.k_split < p.K && p.k_split % KC))
    hipLaunchKernelGGL((linear_kernel<T, EPI, true>), grid, dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL((linear_kernel<T, EPI, false>), grid, dim3(256), 0, s, p);
}

template <typename T> static void launch_linear_t(const LinearParams& p, int epi, LinearKernel k, hipStream_t s) {
  if (k == kLinearFew) {
    if (epi == kEpiPartial) launch_few<T, kEpiPartial>(p, s);
    else if (epi == kEpiSwiglu) launch_few<T, kEpiSwiglu>(p, s);
    else launch_few<T, kEpiLogits>(p, s);
    return;
  }
  if (epi == kEpiPartial) launch_skinny<T, kEpiPartial>(p, s);
  else if (epi == kEpiSwiglu) launch_skinny<T, kEpiSwiglu>(p, s);
  else launch_skinny<T, kEpiLogits>(p, s);
}

// Work of few_linear_kernel in stages: what the busiest work-group walks (its
// units, each the stages of one wave times four and about three more to start
// and sum), and two more per split for the partials.
static int few_stages(int N, int K, int splits, int es) {
  const int nc = (K * es + kFewStage - 1) / kFewStage;
  const int per = (nc + splits - 1) / splits;
  const long long units = (long long)((N + 15) / 16) * splits;
  return (int)((units + kFewWorkGroups - 1) / kFewWorkGroups) * ((per + 3) / 4 * 4 + 3) + 2 * (splits - 1);
}

// K elements per split of few_linear_kernel: the cheapest of 1 .. 8 splits.
// MI355X, 4 rows, 1 / 2 / 3 / 4 splits: 2048 x 5632 fp32 14.4 / 12.5 / 13.4 /
// 12.1 us (takes 2), fp16 8.8 / 7.3 / 7.9 / 7.6 (2); 2560 x 2048 fp16 5.1 / 5.4 /
// 5.6 / 5.7 (1); 1024 x 2816 fp32 9.0 / 6.7 / 6.1 / 5.9 (3).
static int few_k_split(int N, int K, int es) {
  const int nc = (K * es + kFewStage - 1) / kFewStage;
  int best = 0, chunks = nc;
  for (int s = 1; s <= 8 && s <= nc; ++s) {
    const int cost = few_stages(N, K, s, es);
    if (s == 1 || cost < best) {
      best = cost;
      chunks = (nc + s - 1) / s;
    }
  }
  return (int)std::min<long long>(((long long)K + 31) / 32 * 32, (long long)chunks * (kFewStage / es));
}

// Work-groups a skinny product aims for when it splits K.
constexpr long long kLinearTargetWorkGroups = 192;

// K elements per split of linear_kernel for a product whose consumer sums the
// partials.
static int skinny_k_split(int M, int N, int K) {
  const long long full = ((long long)K + 31) / 32 * 32;
  const long long tiles = ((N + kLinBN - 1) / kLinBN) * (long long)((M + kLinBM - 1) / kLinBM);
  // About three work-groups per four CUs: more splits add partials that the
  // consumer (norm or step attention) reads back, and on the TinyLlama step
  // 192 beat 128, 160, 224 and 256 (1.53 vs 1.55-1.59 ms).
  const long long target = kLinearTargetWorkGroups;
  if (tiles >= target / 2) return (int)full;
  const long long want = (target + tiles - 1) / tiles;
  const long long per = (K + want - 1) / want;
  // whole LDS chunks: a partial chunk still streams the chunk's full width of W
  const long long ks = per >= kLinKC ? (per + kLinKC / 2) / kLinKC * kLinKC : (per + 31) / 32 * 32;
  return (int)std::min(full, std::max(ks, 32LL));
}

// Microseconds of linear_kernel: a start, and per round of work-groups the
// chunks of one (an odd count beyond two runs one more); logits of many rows
// also wait for their scattered stores.  fp32 is bound by its products, so two
// work-groups that share a CU take half a round each.  MI355X, M 65 .. 2048, N
// 512 .. 32768, K 256 .. 16384: most within 15% of the measured time.
static double skinny_us(int M, int N, int K, int k_split, int dtype, bool logits) {
  const int kc = dtype == kF32 ? kLinKC / 2 : kLinKC;
  int chunks = (std::min(k_split, K) + kc - 1) / kc;
  if (chunks > 2) chunks += chunks & 1;
  const long long wgs = (long long)((M + kLinBM - 1) / kLinBM) * ((N + kLinBN - 1) / kLinBN) * ((K + k_split - 1) / k_split);
  const double stores = logits ? 0.6e-6 * M * N : 0.0;
  if (dtype == kF32) return 2.8 + 2.65 * chunks * std::max(1.0, 0.5 * (double)((wgs + 127) / 128)) + stores;
  return (chunks == 1 ? 2.7 : 3.5) + 1.35 * chunks * (double)((wgs + 255) / 256) + stores;
}

// What the consumer of `splits` partials pays for them (about 4 TB/s and a
// quarter of a microsecond each).
static double partials_us(int M, int N, int splits) { return (splits - 1) * ((double)M * N * 1e-6 + 0.25); }

// More than kLinBM rows: the LDS-tiled kernels where their model is the smaller
// one.  They win with many rows, long K or many tiles; where W is small,
// linear_kernel's 64 x 64 tiles and finer splits fill more of the chip.
// MI355X, us, linear_kernel / tiled: 65 rows, fp16 1024 x 1024 4.2 / 5.5, 2048 x
// 2048 9.0 / 7.4; fp32 512 x 512 5.4 / 13.9, 1024 x 4096 (SwiGLU) 86 / 170, 2560 x
// 2048 20.7 / 20.6; 320 rows, fp16 1024 x 512 4.4 / 5.5, 2560 x 2048 16.9 / 12.7;
// fp32 1024 x 1024 13.7 / 14.9, 11264 x 2048 158 / 117.
static double tiled_us(int M, int N, int K, int k_split, int dtype) {
  const int splits = (K + k_split - 1) / k_split;
  return dtype == kF32 ? tile_linear_f32_us(M, N, K, splits) : tile_linear_us(M, N, K, splits);
}

// At most kFewRows rows: microseconds of few_linear_kernel, its share of the
// partials in few_stages.  linear_kernel is the faster one where a work-group
// has one or two chunks: K up to 512 elements under many features (fp16, 4 rows,
// SwiGLU: 32768 x 256 6.1 us against 10.7, 8192 x 256 3.9 / 4.9; fp32 32768 x 128
// 7.6 / 13.3).  Alone it is so too where it splits K that far (fp16, 16 rows:
// 2048 x 2048 4.1 against 5.0 us, 1024 x 2816 3.8 / 4.6), but into 8 and 11 parts
// against 2 and 3, which the next kernel reads: steps of eight TinyLlama layers
// with these products on linear_kernel take 352 us instead of 346 (4 rows), 392
// instead of 388 (16).
static double few_us(int M, int N, int K, int k_split, int dtype) {
  const int stages = few_stages(N, K, (K + k_split - 1) / k_split, dtype == kF32 ? 4 : 2);
  if (dtype == kF32) return 3.0 + 0.18 * stages;
  return M <= 4 ? 3.2 + 0.138 * stages : 4.1 + 0.14 * stages;
}

static bool few_is_faster(int M, int N, int K, int k_split, int dtype, int epi) {
  // one unit of the logits is 64 features: only a single short chunk is faster
  // on 64 x 64 tiles
  if (epi == kEpiLogits) return dtype == kF32 || K > kLinKC || N > 512 * kLinBN;
  return few_us(M, N, K, k_split, dtype) < skinny_us(M, N, K, k_split, dtype, false);
}

// Split of K and kernel of a product whose consumer sums the partials.
struct SplitPlan {
  int k_split;
  LinearKernel kernel;
};
static SplitPlan split_plan(int M, int N, int K, int dtype) {
  const SplitPlan skinny{skinny_k_split(M, N, K), kLinearSkinny};
  if (M > kFewRows && M <= kLinBM) return skinny;
  const double s = skinny_us(M, N, K, skinny.k_split, dtype, false) + partials_us(M, N, (K + skinny.k_split - 1) / skinny.k_split);
  if (M <= kFewRows) {
    const SplitPlan few{few_k_split(N, K, dtype == kF32 ? 4 : 2), kLinearFew};
    return s <= few_us(M, N, K, few.k_split, dtype) ? skinny : few;
  }
  const SplitPlan tiled{dtype == kF32 ? tile_linear_f32_k_split(M, N, K) : tile_linear_k_split(M, N, K), kLinearTiled};
  const double t = tiled_us(M, N, K, tiled.k_split, dtype) + partials_us(M, N, (K + tiled.k_split - 1) / tiled.k_split);
  return s < t ? skinny : tiled;
}

int linear_k_split(int M, int N, int K, int dtype) { return split_plan(M, N, K, dtype).k_split; }

// 32-bit offsets: in the 16 rows that few_linear_kernel addresses, and in the 16
// rows of W and 64 of A (those past M too, which a wrapped offset would bring back
// into range) of linear_kernel.
static bool few_supported(int M, int K, long long lda, int dtype) {
  return M <= kFewRows && std::max<long long>(lda, K) * (dtype == kF32 ? 4 : 2) * 16 < (1LL << 31);
}
static bool skinny_supported(int K, long long lda, int dtype) {
  const long long es = dtype == kF32 ? 4 : 2;
  return K * es * 16 <= (1LL << 32) && lda <= (1LL << 32) / (es * kLinBM);
}
// The tiled kernels' limits lie within linear_kernel's.
bool linear_supported(int M, int K, long long lda, int dtype) {
  return few_supported(M, K, lda, dtype) || skinny_supported(K, lda, dtype);
}

LinearKernel linear_kernel_of(const LinearParams& p, int epi, int dtype) {
  const bool few = few_supported(p.M, p.K, p.lda, dtype);
  if (few && !skinny_supported(p.K, p.lda, dtype)) return kLinearFew;
  const bool tiled = p.M > kLinBM && (dtype == kF32 ? tile_linear_f32_supported(p) : tile_linear_supported(p));
  if (!few && !tiled) return kLinearSkinny;
  if (epi == kEpiPartial) {   // the kernel that a planned split was made for; other splits are the caller's
    const SplitPlan plan = split_plan(p.M, p.N, p.K, dtype);
    if (plan.k_split == p.k_split) return plan.kernel;
  }
  if (few) return few_is_faster(p.M, p.N, p.K, p.k_split, dtype, epi) ? kLinearFew : kLinearSkinny;
  return tiled_us(p.M, p.N, p.K, p.k_split, dtype) <= skinny_us(p.M, p.N, p.K, p.k_split, dtype, epi == kEpiLogits)
             ? kLinearTiled
             : kLinearSkinny;
}

void launch_linear(const LinearParams& p, int epi, int dtype, hipStream_t s) {
  const LinearKernel k = linear_kernel_of(p, epi, dtype);
  if (k == kLinearTiled && dtype == kF32) launch_tile_linear_f32(p, epi, s);
  else if (k == kLinearTiled) launch_tile_linear(p, epi, dtype, s);
  else if (dtype == kF16) launch_linear_t<_Float16>(p, epi, k, s);
  else if (dtype == kBF16) launch_linear_t<__bf16>(p, epi, k, s);
  else launch_linear_t<float>(p, epi, k, s);
}

// ---------------------------------------------------------------------------
// residual add + RMSNorm
// ---------------------------------------------------------------------------

// One work-group per row; thread t holds float4 vectors t + 256 i (VPT of
// them) in registers, so the row is read once: every load (weight, embedding
// or residual, split partials) is issued before the first add, one LDS
// reduction gives the mean square, and the normalised row is written from
// registers.
// MODE: kNormEmb (x = emb[tokens]), kNormPart (x += the split partials) or
// kNormPlain (x as it is).  One instantiation per mode keeps every load of the
// row in one basic block, so the weight, residual and first batch of partials
// are all requested before the first wait.
enum NormMode : int { kNormEmb = 0, kNormPart = 1, kNormPlain = 2 };

template <typename T, int VPT, int MODE>
__global__ void __launch_bounds__(256) norm_kernel(const NormParams p) {
  __shared__ float red[4];
  const int m = blockIdx.x;
  float* x = p.x + (size_t)m * p.dim;
  // SB splits per batch of loads: all of a product's splits in one round trip
  // at the decode step's sizes; indexes past the last split re-read it and are
  // dropped
  constexpr int SB = VPT <= 2 ? 8 : 4;
  f32x4 v[VPT], w[VPT], t[MODE == kNormPart ? SB : 1][VPT];
  int tok = 0;
  if constexpr (MODE == kNormEmb) tok = min(max(p.tokens[m], 0), p.vocab - 1);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int k = min(4 * (threadIdx.x + 256 * i), p.dim - 4);   // clamped: lanes past dim re-read the last vector
    w[i] = *reinterpret_cast<const f32x4*>(p.weight + k);
    if constexpr (MODE == kNormEmb) {
      v[i] = load4<T>(p.emb, (size_t)tok * p.dim + k);
    } else {
      v[i] = *reinterpret_cast<const f32x4*>(x + k);
    }
    if constexpr (MODE == kNormPart) {
      if (p.splits == 1) {   // unsplit producer (prompt passes): one load, not SB copies of it
        t[0][i] = *reinterpret_cast<const f32x4*>(p.part + (size_t)m * p.dim + k);
      } else {
#pragma unroll
        for (int u = 0; u < SB; ++u)
          t[u][i] = *reinterpret_cast<const f32x4*>(p.part + ((size_t)min(u, p.splits - 1) * p.M + m) * p.dim + k);
      }
    }
  }
  if constexpr (MODE == kNormPart) {
#pragma unroll
    for (int u = 0; u < SB; ++u)
      if (u < p.splits) {
#pragma unroll
        for (int i = 0; i < VPT; ++i) v[i] += t[u][i];
      }
    for (int s0 = SB; s0 < p.splits; s0 += SB) {
#pragma unroll
      for (int u = 0; u < SB; ++u)
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
          const int k = min(4 * (threadIdx.x + 256 * i), p.dim - 4);
          t[u][i] = *reinterpret_cast<const f32x4*>(p.part + ((size_t)min(s0 + u, p.splits - 1) * p.M + m) * p.dim + k);
        }
#pragma unroll
      for (int u = 0; u < SB; ++u)
        if (s0 + u < p.splits) {
#pragma unroll
          for (int i = 0; i < VPT; ++i) v[i] += t[u][i];
        }
    }
  }
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int k = 4 * (threadIdx.x + 256 * i);
    if (k < p.dim) {
      if constexpr (MODE != kNormPlain) *reinterpret_cast<f32x4*>(x + k) = v[i];
      ss += v[i][0] * v[i][0] + v[i][1] * v[i][1] + v[i][2] * v[i][2] + v[i][3] * v[i][3];
    }
  }
  ss = group_sum<64>(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  lds_barrier();
  const float r = rsqrtf((red[0] + red[1] + red[2] + red[3]) / (float)p.dim + p.eps);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int k = 4 * (threadIdx.x + 256 * i);
    if (k < p.dim) {
      store4<T>(p.xh, (size_t)m * p.dim + k, v[i] * r * w[i]);
    }
  }
}

template <typename T, int VPT> void launch_norm_v(const NormParams& p, hipStream_t s) {
  if (p.emb) hipLaunchKernelGGL((norm_kernel<T, VPT, kNormEmb>), dim3(p.M), dim3(256), 0, s, p);
  else if (p.part) hipLaunchKernelGGL((norm_kernel<T, VPT, kNormPart>), dim3(p.M), dim3(256), 0, s, p);
  else hipLaunchKernelGGL((norm_kernel<T, VPT, kNormPlain>), dim3(p.M), dim3(256), 0, s, p);
}

template <typename T> void launch_norm_t(const NormParams& p, hipStream_t s) {
  const int vpt = (p.dim + 1023) / 1024;
  if (vpt <= 1) launch_norm_v<T, 1>(p, s);
  else if (vpt <= 2) launch_norm_v<T, 2>(p, s);
  else if (vpt <= 4) launch_norm_v<T, 4>(p, s);
  else launch_norm_v<T, 8>(p, s);
}

void launch_norm(const NormParams& p, int dtype, hipStream_t s) {
  if (dtype == kF16)
    launch_norm_t<_Float16>(p, s);
  else if (dtype == kBF16)
    launch_norm_t<__bf16>(p, s);
  else
    launch_norm_t<float>(p, s);
}

// ---------------------------------------------------------------------------
// QKV: split reduction, RoPE, q store, K/V cache write
// ---------------------------------------------------------------------------

template <typename T>
__global__ void __launch_bounds__(256) qkv_rope_kernel(const QKVParams p) {
  const int qn = p.Hq * p.D;
  const int kn = p.Hkv * p.D;
  const int N = qn + 2 * kn;
  const int half = N >> 1;
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  if (t >= (long long)p.M * half) return;
  const int m = (int)(t / half);
  const int n = 2 * (int)(t - (long long)m * half);
  // SB split partials requested at once with the position (one round trip
  // for the usual split counts); indexes past the last split re-read it and
  // are dropped; the sum runs in split order
  constexpr int SB = 8;
  float2 pv[SB];
  if (p.splits == 1) {   // unsplit producer (prompt passes): one load, not SB copies of it
    pv[0] = *reinterpret_cast<const float2*>(p.part + (size_t)m * N + n);
  } else {
#pragma unroll
    for (int s = 0; s < SB; ++s)
      pv[s] = *reinterpret_cast<const float2*>(p.part + ((size_t)min(s, p.splits - 1) * p.M + m) * N + n);
  }
  const int pos = p.positions ? p.positions[m] : p.pos_base + m;
  float v0 = 0.0f, v1 = 0.0f;
#pragma unroll
  for (int s = 0; s < SB; ++s)
    if (s < p.splits) {
      v0 += pv[s].x;
      v1 += pv[s].y;
    }
  for (int s0 = SB; s0 < p.splits; s0 += SB) {
#pragma unroll
    for (int s = 0; s < SB; ++s)
      pv[s] = *reinterpret_cast<const float2*>(p.part + ((size_t)min(s0 + s, p.splits - 1) * p.M + m) * N + n);
#pragma unroll
    for (int s = 0; s < SB; ++s)
      if (s0 + s < p.splits) {
        v0 += pv[s].x;
        v1 += pv[s].y;
      }
  }
  if (n < qn + kn) {
    const int i = (n % p.D) >> 1;
    const int pr = min(max(pos, 0), p.rope_len - 1);
    const float2 cs = *reinterpret_cast<const float2*>(p.rope + ((size_t)pr * (p.D >> 1) + i) * 2);
    const float a = v0 * cs.x - v1 * cs.y;
    const float b = v0 * cs.y + v1 * cs.x;
    v0 = a;
    v1 = b;
  }
  if (n < qn) {
    store2<T>(p.q, (size_t)m * qn + n, v0, v1);
    return;
  }
  const bool is_k = n < qn + kn;
  const int e = is_k ? n - qn : n - qn - kn;
  void* stage = is_k ? p.k_out : p.v_out;
  if (stage) store2<T>(stage, (size_t)m * kn + e, v0, v1);
  void* cache = is_k ? p.k_cache : p.v_cache;
  const bool report = is_k && e == 0;   // one thread per row reports the slot
  if (!p.block_tables || (!cache && !(report && (p.slots || p.err_count)))) return;
  long long slot = -1;
  if (pos >= 0 && pos / p.block_size < p.bt_width) {
    const int blk = p.block_tables[(size_t)m * p.bt_row_step + pos / p.block_size];
    if (blk >= 0 && blk < p.num_blocks) slot = (long long)blk * p.block_size + pos % p.block_size;
  }
  if (cache && slot >= 0) store2<T>(cache, (size_t)slot * kn + e, v0, v1);
  if (report) {
    if (p.slots) p.slots[m] = (int)slot;
    if (slot < 0 && p.err_count) atomicAdd(p.err_count, 1u);
  }
}

void launch_qkv_rope(const QKVParams& p, int dtype, hipStream_t s) {
  const long long pairs = (long long)p.M * ((p.Hq + 2 * p.Hkv) * p.D / 2);
  const dim3 grid((unsigned)((pairs + 255) / 256));
  if (dtype == kF16)
    hipLaunchKernelGGL(qkv_rope_kernel<_Float16>, grid, dim3(256), 0, s, p);
  else if (dtype == kBF16)
    hipLaunchKernelGGL(qkv_rope_kernel<__bf16>, grid, dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL(qkv_rope_kernel<float>, grid, dim3(256), 0, s, p);
}

__global__ void rope_table_kernel(float* table, int max_pos, int head_dim, float theta) {
  const int half = head_dim >> 1;
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long long)max_pos * half) return;
  const int pos = (int)(idx / half);
  const int i = (int)(idx - (long long)pos * half);
  const float freq = 1.0f / powf(theta, (float)(2 * i) / (float)head_dim);
  const float ang = (float)pos * freq;
  table[2 * idx] = cosf(ang);
  table[2 * idx + 1] = sinf(ang);
}

void launch_rope_table(float* table, int max_pos, int head_dim, float theta, hipStream_t s) {
  const long long n = (long long)max_pos * (head_dim / 2);
  hipLaunchKernelGGL(rope_table_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, table, max_pos,
                     head_dim, theta);
}

// ---------------------------------------------------------------------------
// greedy sampling + position advance
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(64) advance_kernel(const AdvanceParams p) {
  const int m = blockIdx.x;
  const int lane = threadIdx.x;
  unsigned long long best = 0;
  // U keys per lane requested at once (500 per sequence at a 32000 vocabulary:
  // one round trip); indexes past the last key re-read it, which max ignores
  constexpr int U = 8;
  for (int j0 = 0; j0 < p.nparts; j0 += 64 * U) {
    unsigned long long kv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) kv[u] = p.keys[(size_t)min(j0 + lane + 64 * u, p.nparts - 1) * p.M + m];
#pragma unroll
    for (int u = 0; u < U; ++u) best = max(best, kv[u]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute((lane ^ off) << 2, (int)(uint32_t)best);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute((lane ^ off) << 2, (int)(uint32_t)(best >> 32));
    best = max(best, ((unsigned long long)hi << 32) | lo);
  }
  if (lane != 0) return;
  const int tok = (int)(0xFFFFFFFFu - (uint32_t)best);
  p.tokens[m] = tok;
  if (p.positions) {
    const int pos = p.positions[m];
    if (p.history && pos >= 0 && pos + 1 < p.history_len) p.history[(size_t)m * p.history_len + pos + 1] = tok;
    p.positions[m] = pos + 1;
  }
  if (p.context_lens) p.context_lens[m] += 1;
}

void launch_advance(const AdvanceParams& p, hipStream_t s) {
  hipLaunchKernelGGL(advance_kernel, dim3(p.M), dim3(64), 0, s, p);
}

__global__ void __launch_bounds__(256) iota_kernel(int* out, int n, int base) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = base + i;
}

void launch_iota(int* out, int n, int base, hipStream_t s) {
  hipLaunchKernelGGL(iota_kernel, dim3((n + 255) / 256), dim3(256), 0, s, out, n, base);
}

}  // namespace tv
