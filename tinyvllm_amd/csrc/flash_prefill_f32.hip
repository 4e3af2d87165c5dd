// Causal / full prefill attention for fp32 inputs, head_dim 64 or 128, on the
// bf16 matrix cores without giving up fp32 products.
//
// Same semantics as the other prefill kernels (flash_prefill.hip; reference
// tinyvllm/model/llama.py:58-94).  An fp32 number is the exact sum of three
// bf16 numbers, so a product of two is the sum of nine bf16 products, each
// exact in fp32, of which the three smallest are left out (tv_split.h).  Six
// v_mfma_f32_16x16x32_bf16 take 96 cycles where eight v_mfma_f32_16x16x4_f32
// take 256.  Every chain of six starts from zero and joins the score or the
// output in one fp32 add (tile_linear_f32.hip).
//
// A work-group owns 64 query rows of one head, 16 per wave; KS groups of four
// waves share the row block's 32-key tiles (group s takes tiles s + KS j) and
// merge through LDS.  Tiles are loaded a step ahead into registers, split there
// once per work-group and stored as six bf16 planes.  The step itself is the
// 16-bit kernel's (S^T = K Q^T, log2-domain softmax with a lazy rescale, P as
// the B operand of O^T = V^T P^T from registers), with row sums by fp32 adds.
// The split costs about as many issue slots per tile as the products, so
// neither unit is full; two work-groups (or key groups) per CU overlap them.
// MI355X, causal, against one wave per query row on the VALU: Hq 32 / Hkv 4,
// head_dim 64: L 64 8.9 -> 6.5 us, L 512 174 -> 19, L 1500 1347 -> 75; Hkv 8,
// head_dim 128: L 512 354 -> 33, L 1500 2834 -> 148 (125 TFLOP/s of attention).
// Error against 64 bits (2-norm; L 64 / 300 / 700): N(0, 1) 0.8e-7 / 1.1e-7 /
// 1.1e-7, the VALU kernel 1.8e-7 / 3.1e-7 / 3.0e-7; scores of standard deviation
// 6: 1.9e-7 / 2.8e-7 / 3.0e-7 against 4.7e-7 / 9.8e-7 / 8.3e-7.
#include "tv_common.h"
#include "tv_paged_keys.h"
#include "tv_params.h"
#include "tv_split.h"

#include <algorithm>

namespace tv {

namespace {

constexpr int kBM = 64;   // query rows per work-group
constexpr int kBN = 32;   // keys per tile

// Element offset of key j's row in k / v.
template <bool PAGED> __device__ __forceinline__ long long key_row(const PrefillParams& p, int j) {
  if constexpr (!PAGED) return j;
  int b = p.kv_table[j >> p.kv_bs_log2];
  b = (unsigned)b < (unsigned)p.kv_num_blocks ? b : 0;
  return ((long long)b << p.kv_bs_log2) + (j & ((1 << p.kv_bs_log2) - 1));
}

// One query row by one wave in plain fp32 arithmetic, each key's value touched
// only where the key is visible: the rows whose result above is not finite
// (infinities or NaN among the inputs, or values beyond tv_split.h's range).
template <int D, bool PAGED>
__device__ __forceinline__ void exact_row(const PrefillParams& p, int h, int qi, float* sp) {
  const int lane = threadIdx.x & 63;
  const int kvh = h / (p.num_heads / p.num_kv_heads);
  const float* q = reinterpret_cast<const float*>(p.q) + (size_t)qi * p.q_stride + (size_t)h * D;
  const float* kg = reinterpret_cast<const float*>(p.k) + (size_t)kvh * D;
  const float* vg = reinterpret_cast<const float*>(p.v) + (size_t)kvh * D;
  const float c = p.scale * kLog2e;
  const int kend = p.causal ? min(p.kv_len, qi + p.q_pos_offset + 1) : p.kv_len;
  float m = kNegInf, l = 0.0f, acc[D / 64] = {};
  for (int k0 = 0; k0 < kend; k0 += 64) {
    float x = kNegInf;
    if (k0 + lane < kend) {
      const float* kr = kg + key_row<PAGED>(p, k0 + lane) * p.k_stride;
      float dot = 0.0f;
      for (int d = 0; d < D; ++d) dot = fmaf(q[d], kr[d], dot);
      x = dot * c;
    }
    const float mn = fmaxf(m, group_max<64>(x));
    const float mu = mn == kNegInf ? 0.0f : mn;
    const float alpha = fast_exp2(m - mu);
    m = mn;
    const float e = fast_exp2(x - mu);
    l = l * alpha + group_sum<64>(e);
    sp[lane] = e;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int t = 0; t < D / 64; ++t) {
      float a = acc[t] * alpha;
      for (int j = 0; j < min(64, kend - k0); ++j)
        a = fmaf(sp[j], vg[key_row<PAGED>(p, k0 + j) * p.v_stride + lane + 64 * t], a);
      acc[t] = a;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
#pragma unroll
  for (int t = 0; t < D / 64; ++t)
    reinterpret_cast<float*>(p.out)[(size_t)qi * p.out_stride + (size_t)h * D + lane + 64 * t] = acc[t] * (1.0f / l);
}

}  // namespace

template <int D, int KS, bool PAGED>
__global__ void __launch_bounds__(256 * KS) __attribute__((amdgpu_waves_per_eu(2)))
prefill_f32_kernel(const PrefillParams p) {
  constexpr int GT = 256;                 // threads of a key group
  constexpr int KP = D + 16;              // plane row pitch: 32 bytes past a multiple of 128, conflict-free
  constexpr int PLANE = kBN * KP;
  constexpr int TILE = 6 * PLANE;         // K planes, then V planes
  constexpr int KSD = D / 32;
  constexpr int DB = D / 16;
  constexpr int UPR = D / 8;              // 8-float units per row
  constexpr int NV = kBN * UPR / GT;      // units per thread, each of K and V
  constexpr int MP = D + 4;
  constexpr int MERGE = KS > 1 ? KS * kBM * (MP + 2) * 2 : 0;
  constexpr int SMEM = KS * TILE > MERGE ? KS * TILE : MERGE;
  static_assert(NV * GT == kBN * UPR, "tile shape");
  __shared__ __attribute__((aligned(16))) uint16_t smem[SMEM];
  __shared__ float redo[4][64];
  __shared__ int stbl[PAGED ? kPagedTableMax : 1];
  __shared__ int sbad;                    // first table entry that is not a block

  const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x / GT);
  const int tid = threadIdx.x - grp * GT;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4;
  const int col = lane & 15;
  uint16_t* const tile = smem + grp * TILE;

  // heads of a KV group on one XCD; query tiles zig-zag, the longer half first
  const int h = p.xcd_remap ? (blockIdx.x & 7) * (p.num_heads >> 3) + (blockIdx.x >> 3) : blockIdx.x;
  const int kvh = h / (p.num_heads / p.num_kv_heads);
  const int nqt = (p.q_len + kBM - 1) / kBM;
  const int halfq = (nqt + 1) / 2;
  const int qt = (int)blockIdx.y < halfq ? nqt - 1 - (int)blockIdx.y : (int)blockIdx.y - halfq;
  const int qoff = p.q_pos_offset;
  const int kend = prefill_unit_key_end(p.causal != 0, p.kv_len, qt, kBM, qoff);
  const int ntiles = (kend + kBN - 1) / kBN;
  const float c = p.scale * kLog2e;
  const int row0 = qt * kBM + wave * 16;
  const int qi = row0 + col;

  u32x4 qf[KSD][3];
  {
    const float* qg = reinterpret_cast<const float*>(p.q) + (size_t)min(qi, p.q_len - 1) * p.q_stride + (size_t)h * D;
#pragma unroll
    for (int ks = 0; ks < KSD; ++ks)
      split8(*reinterpret_cast<const f32x4*>(qg + ks * 32 + g * 8), *reinterpret_cast<const f32x4*>(qg + ks * 32 + g * 8 + 4),
             qf[ks]);
  }

  const float* kbase = reinterpret_cast<const float*>(p.k) + (size_t)kvh * D;
  const float* vbase = reinterpret_cast<const float*>(p.v) + (size_t)kvh * D;
  int urow[NV], uch[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    urow[i] = (tid + i * GT) / UPR;
    uch[i] = (tid + i * GT) % UPR * 8;
  }
  const int lg = p.kv_bs_log2;
  const int kstage = paged_stage_end(0, kend);
  bool bad = false;
  if constexpr (PAGED) {   // block ids of keys [0, kend); an invalid id reads block 0, and the rows that see it become NaN
    const int nblk = paged_staged_blocks(0, kstage, lg);
    if (threadIdx.x == 0) sbad = 0x7FFFFFFF;
    lds_barrier();
    for (int i = threadIdx.x; i < nblk; i += blockDim.x) {
      const int b = p.kv_table[i];
      const bool ok = (unsigned)b < (unsigned)p.kv_num_blocks;
      stbl[i] = ok ? b : 0;
      if (!ok) atomicMin(&sbad, i);
    }
    lds_barrier();
    bad = sbad <= (p.causal ? min(p.kv_len - 1, qi + qoff) : p.kv_len - 1) >> lg;
  }
  struct Stage {
    u32x4 k[NV][2], v[NV][2];
  } st;
  auto gload = [&](int j) {
    const int t = prefill_group_tile(grp, KS, j, ntiles);
    if constexpr (PAGED) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int key = paged_load_key(0, kstage, t, kBN, urow[i]);
        const long long row = ((long long)stbl[paged_stage_slot(key, 0, lg)] << lg) + (key & ((1 << lg) - 1));
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          st.k[i][u] = *reinterpret_cast<const u32x4*>(kbase + row * p.k_stride + uch[i] + 4 * u);
          st.v[i][u] = *reinterpret_cast<const u32x4*>(vbase + row * p.v_stride + uch[i] + 4 * u);
        }
      }
    } else {
      // range ends at the last key row: rows past it read as zero
      const int last = min(p.kv_len - t * kBN, kBN) - 1;
      const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float*>(kbase + (long long)t * kBN * p.k_stride), 0, (last * (int)p.k_stride + D) * 4, 0x00020000);
      const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float*>(vbase + (long long)t * kBN * p.v_stride), 0, (last * (int)p.v_stride + D) * 4, 0x00020000);
#pragma unroll
      for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          st.k[i][u] = buffer_load16(rk, (urow[i] * (int)p.k_stride + uch[i]) * 4 + 16 * u, 0);
          st.v[i][u] = buffer_load16(rv, (urow[i] * (int)p.v_stride + uch[i]) * 4 + 16 * u, 0);
        }
    }
  };
  auto lstore = [&]() {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      u32x4 s[3];
      uint16_t* d = tile + urow[i] * KP + uch[i];
      split8(as_f32x4(st.k[i][0]), as_f32x4(st.k[i][1]), s);
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4*>(d + q * PLANE) = s[q];
      split8(as_f32x4(st.v[i][0]), as_f32x4(st.v[i][1]), s);
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4*>(d + (3 + q) * PLANE) = s[q];
    }
  };

  f32x4 oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) oacc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  float mref = 0.0f, thr = -__FLT_MAX__, lsum = 0.0f;   // rescale threshold: -FLT_MAX until the first visible key
  float lowest = 0.0f;                                  // smallest score, before scale and mask

  auto compute = [&](int t) {
    const int k0 = t * kBN;
    if (p.causal && k0 > row0 + 15 + qoff) return;      // no visible key for this wave
    f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int ks = 0; ks < KSD; ++ks)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        u32x4 kf[3];
#pragma unroll
        for (int q = 0; q < 3; ++q)
          kf[q] = *reinterpret_cast<const u32x4*>(tile + q * PLANE + (kb * 16 + col) * KP + ks * 32 + g * 8);
        s[kb] += mfma_split(kf, qf[ks], f32x4{0.f, 0.f, 0.f, 0.f});
      }
    // a score of -inf is one whose sum overflowed on its way (the inputs have no
    // infinities, or it would be NaN): its row is repeated in plain fp32
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
      lowest = fminf(lowest, fminf(fminf(s[kb][0], s[kb][1]), fminf(s[kb][2], s[kb][3])));
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[kb][i] = fmaf(s[kb][i] * kSplitUnscale, c, -mref);
    if (!(k0 + kBN <= p.kv_len && (!p.causal || k0 + kBN - 1 <= row0 + qoff))) {
      const int rel = (p.causal ? min(p.kv_len - 1, qi + qoff) : p.kv_len - 1) - (k0 + 4 * g);   // last visible key
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[kb][i] = kb * 16 + i <= rel ? s[kb][i] : kNegInf;
    }
    const float lm = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])),
                           fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
    if (__builtin_amdgcn_ballot_w64(lm > thr) != 0) {
      const float mt = max_over_g(lm);
      const bool need = mt > thr;
      const float delta = need ? mt : 0.0f;
      const float alpha = need && thr > 0.0f ? fast_exp2(-delta) : 1.0f;
#pragma unroll
      for (int db = 0; db < DB; ++db) oacc[db] *= alpha;
      lsum *= alpha;
      s[0] -= delta;
      s[1] -= delta;
      mref += delta;
      thr = need ? 8.0f : thr;
    }
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[kb][i] = fast_exp2(s[kb][i]);
    lsum += ((s[0][0] + s[0][1]) + (s[0][2] + s[0][3])) + ((s[1][0] + s[1][1]) + (s[1][2] + s[1][3]));
    // reduction index 8 g + j: key 4 g + j (j < 4), 16 + 4 g + j - 4
    u32x4 pf[3];
    split8(s[0], s[1], pf);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      u32x4 vf[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const uint16_t* a = tile + (3 + q) * PLANE + (4 * g + (col >> 2)) * KP + db * 16 + 4 * (col & 3);
        const u32x2 lo = lds_read_tr16(a);
        const u32x2 hi = lds_read_tr16(a + 16 * KP);
        vf[q] = u32x4{lo[0], lo[1], hi[0], hi[1]};
      }
      oacc[db] += mfma_split(vf, pf, f32x4{0.f, 0.f, 0.f, 0.f});   // one fp32 add per tile (tile_linear_f32.hip)
    }
  };

  const int nsteps = (ntiles + KS - 1) / KS;
  gload(0);
  for (int j = 0; j < nsteps; ++j) {
    if (j > 0) lds_barrier();             // the previous tile has been read
    lstore();
    gload(j + 1);                         // in flight while this tile multiplies
    lds_barrier();
    if (grp + KS * j < ntiles) compute(grp + KS * j);
  }

  float l = sum_over_g(lowest > kNegInf ? lsum : __builtin_nanf(""));
  if constexpr (KS > 1) {
    float* so = reinterpret_cast<float*>(smem);   // [KS][64 rows][MP]
    float* ssum = so + KS * kBM * MP;             // [KS][64 rows]
    float* smax = ssum + KS * kBM;                // [KS][64 rows]
    const int row = wave * 16 + col;
    lds_barrier();
#pragma unroll
    for (int db = 0; db < DB; ++db) *reinterpret_cast<f32x4*>(&so[(grp * kBM + row) * MP + db * 16 + 4 * g]) = oacc[db];
    if (g == 0) {
      ssum[grp * kBM + row] = l;
      smax[grp * kBM + row] = thr > 0.0f ? mref : kNegInf;
    }
    lds_barrier();
    if (grp != 0) return;
    float M = kNegInf;
#pragma unroll
    for (int s = 0; s < KS; ++s) M = fmaxf(M, smax[s * kBM + row]);
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    l = 0.0f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float ms = smax[s * kBM + row];
      const float f = ms == kNegInf ? 0.0f : fast_exp2(ms - M);
      l = fmaf(ssum[s * kBM + row], f, l);
#pragma unroll
      for (int db = 0; db < DB; ++db)
        oacc[db] += *reinterpret_cast<const f32x4*>(&so[(s * kBM + row) * MP + db * 16 + 4 * g]) * f;
    }
  }

  const float inv = bad ? __builtin_nanf("") : kSplitUnscale / l;
  bool finite = true;
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    oacc[db] *= inv;
#pragma unroll
    for (int i = 0; i < 4; ++i) finite = finite && fabsf(oacc[db][i]) < __builtin_inff();
  }
  if (qi < p.q_len) {
    float* o = reinterpret_cast<float*>(p.out) + (size_t)qi * p.out_stride + (size_t)h * D + 4 * g;
#pragma unroll
    for (int db = 0; db < DB; ++db) *reinterpret_cast<f32x4*>(o + db * 16) = oacc[db];
  }
  unsigned long long again = __builtin_amdgcn_ballot_w64(!finite && qi < p.q_len && !bad);
  if (again) {
    __builtin_amdgcn_s_waitcnt(0);        // the rows' first stores
    again |= again >> 32;
    again |= again >> 16;
    for (int r = 0; r < 16; ++r)
      if (again >> r & 1) exact_row<D, PAGED>(p, h, row0 + r, redo[wave]);
  }
}

bool prefill_f32_supported(const PrefillParams& p, int dtype) {
  return dtype == kF32 && p.out_dtype == kF32 && p.head_dim == p.head_dim_v && (p.head_dim == 64 || p.head_dim == 128) &&
         p.q_stride % 4 == 0 && p.k_stride % 4 == 0 && p.v_stride % 4 == 0 && p.out_stride % 4 == 0 &&
         (((uintptr_t)p.q | (uintptr_t)p.k | (uintptr_t)p.v | (uintptr_t)p.out) & 15) == 0 &&
         p.k_stride < (1 << 22) && p.v_stride < (1 << 22) &&   // 32-bit offsets in a tile
         (p.q_len + kBM - 1) / kBM <= 65535;
}

// A first tile of few keys, or a second one, costs more than the generic kernel's
// one step of 64 keys, whose rows stop at their last key (MI355X, causal, generic
// / here: Hq 32, head_dim 64: L 8 3.6 / 4.1 us, 20 4.2 / 4.2, 32 4.8 / 4.3, 40 5.2
// / 5.7, 48 6.0 / 5.8; Hq 8, head_dim 128: L 8 4.9 / 5.3, 16 5.5 / 5.4, 40 7.3 /
// 7.7, 48 7.8 / 7.8; Hq 32: L 40 8.1 / 7.8; Hq 2, head_dim 64: L 48 5.1 / 5.6).
bool prefill_f32_faster(const PrefillParams& p) {
  const int keys = p.causal ? std::min(p.q_len, p.kv_len) : p.kv_len;
  if (keys <= (p.head_dim == 64 ? 20 : 12)) return false;
  if (!p.causal || keys <= kBN || keys > 2 * kBN) return true;
  const int few = p.head_dim == 64 ? (p.num_heads <= 4 ? kBN : 12) : (p.num_heads <= 16 ? 12 : 0);
  return keys > kBN + few;
}

template <bool PAGED> static void launch_f32(const PrefillParams& p, int ks, hipStream_t s) {
  const dim3 grid(p.num_heads, (p.q_len + kBM - 1) / kBM);
  if (p.head_dim == 64) {
    if (ks == 4) hipLaunchKernelGGL((prefill_f32_kernel<64, 4, PAGED>), grid, dim3(1024), 0, s, p);
    else if (ks == 2) hipLaunchKernelGGL((prefill_f32_kernel<64, 2, PAGED>), grid, dim3(512), 0, s, p);
    else hipLaunchKernelGGL((prefill_f32_kernel<64, 1, PAGED>), grid, dim3(256), 0, s, p);
  } else {
    if (ks >= 2) hipLaunchKernelGGL((prefill_f32_kernel<128, 2, PAGED>), grid, dim3(512), 0, s, p);
    else hipLaunchKernelGGL((prefill_f32_kernel<128, 1, PAGED>), grid, dim3(256), 0, s, p);
  }
}

void launch_prefill_f32(const PrefillParams& p_in, hipStream_t s) {
  PrefillParams p = p_in;
  p.xcd_remap = p.num_heads % 8 == 0;
  // Key groups shorten the chain of the longest row (about 1 us per 32 keys):
  // two beyond 64 keys (MI355X, Hq 32 / Hkv 4, head_dim 64, one / two: L 64 5.9 /
  // 6.1 us, L 300 17.9 / 13.8, L 1024 51.5 / 37.9, L 1500 77 / 72; head_dim 128,
  // Hkv 8: L 512 40.2 / 31.9), but not at head_dim 128 with two to three
  // work-groups per CU, which one-group ones run at once (Hq 32, L 1300 106 / 124, L
  // 1500 148 / 153; Hq 16, L 2500 195 / 207; beyond, Hq 32, L 1700 190 / 180); four
  // at head_dim 64 where the grid leaves CUs with one work-group (L 512 20.2 with
  // two, 18.6; L 300 13.8, 13.7).
  const long long wgs = (long long)p.num_heads * ((p.q_len + kBM - 1) / kBM);
  int ks = 2;
  if (p.kv_len <= 64 || (p.head_dim == 128 && wgs > 512 && wgs <= 768)) ks = 1;
  else if (wgs <= 256 && p.kv_len >= 384) ks = 4;   // (head_dim 128: two)
  if (p.kv_table) launch_f32<true>(p, ks, s);
  else launch_f32<false>(p, ks, s);
}

}  // namespace tv
