"""Prefill attention on the GPU vs the oracle (tinyvllm/model/llama.py:58-94).

Restates tests/test_flash_attention.py of the reference (shapes, GQA, causal
known answers, sequence lengths, head dims, dtypes, TinyLlama shapes) and adds
MFMA-path parity for fp16/bf16 at the benchmark shapes.
Tolerances (max-abs vs the float64 oracle): fp32 1e-4, fp16/bf16 2e-2.
"""

import math

import numpy as np
import pytest
import torch

from oracle.attention import flash_prefill_ref
from tests.random_cases import case_count, case_seed

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-4, torch.float16: 2e-2, torch.bfloat16: 2e-2}


def _op():
    from tinyvllm_amd.attention import flash_prefill_attention
    return flash_prefill_attention


def flash(q, k, v, causal=True):
    """[L, H, D] wrapper like the reference test's (adds and removes the batch dim)."""
    out = _op()(q.unsqueeze(0).cuda(), k.unsqueeze(0).cuda(), v.unsqueeze(0).cuda(), causal)
    torch.cuda.synchronize()
    return out.squeeze(0)


def randn(seed, *shape, dtype=torch.float32):
    rng = np.random.Generator(np.random.PCG64(seed))
    return torch.from_numpy(rng.standard_normal(shape, dtype=np.float32)).to(dtype)


def check(q, k, v, causal=True, tol=None):
    out = flash(q, k, v, causal)
    want = flash_prefill_ref(q.float().numpy()[None], k.float().numpy()[None], v.float().numpy()[None], causal)[0]
    err = np.abs(out.float().cpu().numpy() - want).max()
    tol = TOL[q.dtype] if tol is None else tol
    assert err <= tol, f"max-abs {err} > {tol}"
    return out


# ---- restated reference tests ------------------------------------------------------

def test_output_shape():
    out = flash(randn(0, 16, 8, 64), randn(1, 16, 8, 64), randn(2, 16, 8, 64))
    assert out.shape == (16, 8, 64)


@pytest.mark.parametrize("lq,hq,hkv,d", [(32, 4, 4, 32), (32, 32, 8, 64), (16, 8, 4, 32), (16, 32, 8, 64),
                                          (16, 32, 4, 64), (64, 32, 8, 64), (256, 32, 8, 64)])
def test_matches_standard_attention(lq, hq, hkv, d):
    check(randn(3, lq, hq, d), randn(4, lq, hkv, d), randn(5, lq, hkv, d))


def test_non_causal():
    check(randn(6, 16, 4, 32), randn(7, 16, 4, 32), randn(8, 16, 4, 32), causal=False)


def test_causal_mask_first_token():
    q = torch.zeros(8, 2, 16)
    q[0] = 1.0
    k = randn(9, 8, 2, 16)
    v = torch.eye(8).unsqueeze(1).expand(8, 2, 8).contiguous()     # head_dim_v 8 != head_dim 16
    out = check(q, k, v)
    assert out[0, 0, 0].item() > 0.5


def test_last_token_attends_to_all():
    q = torch.ones(8, 2, 16)
    k = torch.zeros(8, 2, 16)
    v = torch.arange(8).reshape(8, 1, 1).expand(8, 2, 16).float().contiguous()
    out = flash(q, k, v)
    assert abs(out[-1, 0, 0].item() - 3.5) < 1e-2


@pytest.mark.parametrize("q_len", [1, 2, 7, 8, 15, 16, 31, 32, 63, 64, 128])
def test_various_lengths(q_len):
    check(randn(10, q_len, 4, 32), randn(11, q_len, 4, 32), randn(12, q_len, 4, 32))


@pytest.mark.parametrize("head_dim", [32, 64, 128])
def test_various_head_dims(head_dim):
    check(randn(13, 16, 4, head_dim), randn(14, 16, 4, head_dim), randn(15, 16, 4, head_dim))


def test_float16_finite():
    q, k, v = (randn(16 + i, 32, 4, 32, dtype=torch.float16) for i in range(3))
    out = check(q, k, v)
    assert out.shape == (32, 4, 32) and torch.isfinite(out).all()


def test_float32_dtype():
    out = flash(randn(19, 32, 4, 32), randn(20, 32, 4, 32), randn(21, 32, 4, 32))
    assert out.dtype == torch.float32 and out.shape == (32, 4, 32)


# ---- MFMA path (fp16 / bf16, head_dim 64 / 128) --------------------------------------

@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("lq", [1, 15, 64, 65, 200])
@pytest.mark.parametrize("causal", [True, False])
def test_mfma_path(dtype, d, lq, causal):
    hq, hkv = 8, 2
    check(randn(22, lq, hq, d, dtype=dtype), randn(23, lq, hkv, d, dtype=dtype),
          randn(24, lq, hkv, d, dtype=dtype), causal)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("lq,hq,hkv", [(300, 8, 2), (1024, 32, 8)])
def test_peaked_softmax(dtype, d, causal, lq, hq, hkv):
    """q, k ~ N(0, 3^2): scores of tens of units, nearly one-hot softmax rows,
    where any rounding of the scores (or of q * scale) before the softmax shows
    up in the output.  The reference scales after the product (llama.py:84), in
    fp32 here; bar: 2e-2 max-abs against the float64 oracle."""
    q = randn(90, lq, hq, d) * 3
    k = randn(91, lq, hkv, d) * 3
    v = randn(92, lq, hkv, d)
    check(q.to(dtype), k.to(dtype), v.to(dtype), causal)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("lq,lk,scale", [(2048, 2048, 1.0), (2100, 2100, 3.0), (2048, 2500, 1.0)])
def test_long_prompts_head_dim_128(dtype, causal, lq, lk, scale):
    """Prompts of 2048+ rows at head_dim 128 take the 128-row kernel with
    LDS-DMA tiles (flash_prefill_rows.hip): full and partial last query and key
    tiles, Lq != Lk (top-left causal), and peaked scores (q, k ~ N(0, 3^2))."""
    q = randn(93, lq, 8, 128) * scale
    k = randn(94, lk, 2, 128) * scale
    v = randn(95, lk, 2, 128)
    check(q.to(dtype), k.to(dtype), v.to(dtype), causal)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("out_dtype", [None, torch.float32])
def test_split_key_halves_workspace_and_fp32_output(dtype, out_dtype):
    """A causal L 2100 prompt at Hq 8 (17 query tiles of 128 rows, all resident
    at once) runs tiles 8-16 as two key halves each, merged by a second kernel
    (flash_prefill_rows.hip): the workspace is sized for the halves, and the
    merged rows match the oracle in the input type and in fp32."""
    from tinyvllm_amd import _lib
    lib = _lib.load()
    lq = 2100
    assert lib.tv_flash_prefill_workspace_bytes(lq, lq, 8, 128, 128, 1, _lib.dtype_code(dtype), 0) > 0
    assert lib.tv_flash_prefill_workspace_bytes(lq, lq, 8, 128, 128, 0, _lib.dtype_code(dtype), 0) == 0
    q = randn(96, lq, 8, 128).to(dtype)
    k = randn(97, lq, 2, 128).to(dtype)
    v = randn(98, lq, 2, 128).to(dtype)
    out = _op()(q.unsqueeze(0).cuda(), k.unsqueeze(0).cuda(), v.unsqueeze(0).cuda(), True, out_dtype=out_dtype)
    torch.cuda.synchronize()
    assert out.dtype == (dtype if out_dtype is None else out_dtype)
    want = flash_prefill_ref(q.float().numpy()[None], k.float().numpy()[None], v.float().numpy()[None], True)[0]
    err = np.abs(out[0].float().cpu().numpy() - want).max()
    assert err <= TOL[dtype], err


def test_split_key_halves_replay_in_graph():
    """The split launch (halves + merge) captured in a HIP graph: replays, with
    eager work between them, equal the eager launch bit for bit."""
    from tinyvllm_amd.attention import PrefillPlan
    q, k, v = (randn(99 + i, 2048, h, 128, dtype=torch.float16).cuda().unsqueeze(0) for i, h in enumerate((8, 2, 2)))
    plan = PrefillPlan(q, k, v)
    assert plan.ws_bytes > 0
    eager = plan.run().clone()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            plan.run()
    torch.cuda.synchronize()
    for _ in range(3):
        plan.out.zero_()
        junk = torch.randn(1 << 20, device="cuda").sum()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(plan.out, eager)
        del junk


def test_split_shape_without_workspace_runs_unsplit():
    """A prompt that would split its key halves, given no workspace through the
    C ABI, runs unsplit and still matches the oracle; a workspace smaller than
    tv_flash_prefill_workspace_bytes asks for is rejected."""
    import math
    from tinyvllm_amd import _lib
    lib = _lib.load()
    lq, hq, hkv, d = 2048, 8, 2, 128
    q, k, v = (randn(110 + i, lq, h, d, dtype=torch.float16) for i, h in enumerate((hq, hkv, hkv)))
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    need = lib.tv_flash_prefill_workspace_bytes(lq, lq, hq, d, d, 1, _lib.TV_F16, 0)
    assert need > 0
    out = torch.empty((lq, hq, d), dtype=torch.float16, device="cuda")
    stream = _lib.stream_ptr(torch.device("cuda"))
    args = (out.data_ptr(), qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), lq, lq, hq, hkv, d, d, hq * d, hkv * d,
            hkv * d, hq * d, 1, 1.0 / math.sqrt(d), _lib.TV_F16, _lib.TV_F16, 0)
    assert lib.tv_flash_prefill(*args, None, 0, stream) == 0
    torch.cuda.synchronize()
    _check_heads(out, q, k, v, True, [0, hkv - 1], torch.float16)
    small = torch.empty(256, dtype=torch.uint8, device="cuda")
    assert lib.tv_flash_prefill(*args, small.data_ptr(), 256, stream) == _lib.TV_EINVAL
    assert b"workspace" in lib.tv_last_error()


def _check_heads(out, q, k, v, causal, groups, dtype):
    """Oracle rows of the query heads of the listed KV groups only (the float64
    oracle over every head of a large grid would take minutes)."""
    hq, hkv = q.shape[1], k.shape[1]
    g = hq // hkv
    for kvh in groups:
        hs = slice(kvh * g, (kvh + 1) * g)
        want = flash_prefill_ref(q[:, hs].float().numpy()[None], k[:, kvh:kvh + 1].float().numpy()[None],
                                 v[:, kvh:kvh + 1].float().numpy()[None], causal)[0]
        err = np.abs(out[:, hs].float().cpu().numpy() - want).max()
        assert err <= TOL[dtype], (kvh, err)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [True, False])
def test_long_prompt_grid_larger_than_resident(dtype, causal):
    """Hq 48 / Hkv 8 at L 2100: 816 work-groups of the 128-row kernel, more
    than are resident at once, so query tiles are dealt longest first (an odd
    tile count and a partial last tile); rows of two KV groups' query heads
    against the oracle -- the tile order is the same for every head."""
    lq = 2100
    q = randn(140, lq, 48, 128).to(dtype)
    k = randn(141, lq, 8, 128).to(dtype)
    v = randn(142, lq, 8, 128).to(dtype)
    out = flash(q, k, v, causal)
    _check_heads(out, q, k, v, causal, [0, 7], dtype)


def test_varlen_long_prompts_grid_larger_than_resident():
    """Two long prompts packed (Hq 32: grid 32 x 18 x 2 = 1152 work-groups of
    the 128-row kernel, longest-first tiles within each prompt)."""
    from tinyvllm_amd.attention import flash_prefill_varlen
    lens = [2300, 2048]
    tot = sum(lens)
    q, k, v = (randn(143 + i, tot, 32 if i == 0 else 8, 128, dtype=torch.float16) for i in range(3))
    out = flash_prefill_varlen(q.cuda(), k.cuda(), v.cuda(), lens, True)
    torch.cuda.synchronize()
    s = 0
    for n in lens:
        sl = slice(s, s + n)
        _check_heads(out[sl], q[sl], k[sl], v[sl], True, [0, 5], torch.float16)
        s += n


@pytest.mark.parametrize("length", [512, 1024])
def test_tinyllama_prefill_shape(length):
    """TinyLlama prefill shape: Hq 32, Hkv 4, D 64, fp16 inputs, causal."""
    q, k, v = (randn(30 + i, length, 32 if i == 0 else 4, 64, dtype=torch.float16) for i in range(3))
    check(q, k, v)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lq,lk,causal", [(600, 600, False), (520, 520, True), (500, 700, True), (480, 900, False)])
def test_key_split_work_groups(dtype, lq, lk, causal, d):
    """Grids of at most one work-group per CU with rows of 8+ key tiles run two
    key groups per work-group and merge them in LDS."""
    q = randn(70, lq, 8, d, dtype=dtype)
    k = randn(71, lk, 2, d, dtype=dtype)
    v = randn(72, lk, 2, d, dtype=dtype)
    check(q, k, v, causal)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lq,lk,causal", [(600, 600, False), (700, 900, True)])
def test_key_split_short_tiles(dtype, lq, lk, causal, d):
    """Between one and four work-groups per CU (Hq 32) with long rows: two key
    groups of 32-key tiles per work-group."""
    q = randn(73, lq, 32, d, dtype=dtype)
    k = randn(74, lk, 4, d, dtype=dtype)
    v = randn(75, lk, 4, d, dtype=dtype)
    check(q, k, v, causal)


@pytest.mark.parametrize("length", [512, 2048])
def test_llama3_8b_head_prefill(length):
    """Llama-3-8B head shape (Hq 32, Hkv 8, head_dim 128), fp16, causal."""
    q, k, v = (randn(80 + i, length, 32 if i == 0 else 8, 128, dtype=torch.float16) for i in range(3))
    check(q, k, v)


def test_unequal_lengths_top_left_causal():
    q = randn(40, 40, 8, 64, dtype=torch.float16)
    k = randn(41, 100, 2, 64, dtype=torch.float16)
    v = randn(42, 100, 2, 64, dtype=torch.float16)
    check(q, k, v, True)
    q32 = randn(43, 10, 4, 32)
    check(q32, randn(44, 30, 4, 32), randn(45, 30, 4, 32), True)


def test_strided_inputs_from_fused_qkv():
    """q/k/v as views into one [L, (Hq+2Hkv)*D] projection output."""
    L, hq, hkv, d = 96, 8, 2, 64
    qkv = randn(46, L, (hq + 2 * hkv) * d, dtype=torch.float16).cuda()
    q = qkv[:, :hq * d].view(L, hq, d)
    k = qkv[:, hq * d:(hq + hkv) * d].view(L, hkv, d)
    v = qkv[:, (hq + hkv) * d:].view(L, hkv, d)
    out = _op()(q.unsqueeze(0), k.unsqueeze(0), v.unsqueeze(0), True)[0]
    want = flash_prefill_ref(q.float().cpu().numpy()[None], k.float().cpu().numpy()[None],
                             v.float().cpu().numpy()[None], True)[0]
    assert np.abs(out.float().cpu().numpy() - want).max() <= 2e-2


def test_rejects_batch_above_one():
    q = randn(47, 2, 8, 4, 32).cuda()
    with pytest.raises(ValueError, match="batch 1"):
        _op()(q, q[:, :, :4], q[:, :, :4], True)


@pytest.mark.parametrize("chunk_tiles", [1, 2, 3, 5])
@pytest.mark.parametrize("lq,causal", [(130, True), (500, True), (200, False)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_mfma_split_rows_merge(chunk_tiles, lq, causal, dtype):
    """Long rows split into key chunks on separate work-groups, merged by a second kernel."""
    q, k, v = (randn(60 + i, lq, 8 if i == 0 else 2, 64, dtype=dtype) for i in range(3))
    out = _op()(q.unsqueeze(0).cuda(), k.unsqueeze(0).cuda(), v.unsqueeze(0).cuda(), causal,
                chunk_tiles=chunk_tiles)[0]
    want = flash_prefill_ref(q.float().numpy()[None], k.float().numpy()[None], v.float().numpy()[None], causal)[0]
    assert np.abs(out.float().cpu().numpy() - want).max() <= 2e-2


# ---- seeded random shapes -------------------------------------------------------------

def _random_prefill_cases(n=None, seed=71):
    n = case_count(24) if n is None else n
    rng = np.random.Generator(np.random.PCG64(case_seed(seed)))
    cases = []
    for i in range(n):
        hkv = int(rng.choice([1, 2, 4, 8]))
        hq = hkv * int(rng.choice([1, 2, 4, 8]))
        d = int(rng.choice([64, 128, 64, 128, 32, 80]))
        lq = int(rng.integers(1, 700))
        lk = lq if rng.random() < 0.7 else int(rng.integers(1, 700))
        causal = bool(rng.random() < 0.7)
        dtype = [torch.float16, torch.bfloat16, torch.float32][int(rng.integers(0, 3))]
        chunk = int(rng.choice([0, 0, 0, 1, 2, 4]))
        cases.append((i, hq, hkv, d, lq, lk, causal, dtype, chunk))
    return cases


@pytest.mark.parametrize("i,hq,hkv,d,lq,lk,causal,dtype,chunk", _random_prefill_cases())
def test_random_shapes(i, hq, hkv, d, lq, lk, causal, dtype, chunk):
    """Seeded random head counts, head dims (MFMA and generic), lengths
    (Lq != Lk included), masks, dtypes and key-chunk splits against the oracle."""
    q = randn(300 + i, lq, hq, d, dtype=dtype)
    k = randn(400 + i, lk, hkv, d, dtype=dtype)
    v = randn(500 + i, lk, hkv, d, dtype=dtype)
    out = _op()(q.unsqueeze(0).cuda(), k.unsqueeze(0).cuda(), v.unsqueeze(0).cuda(), causal,
                chunk_tiles=chunk)[0]
    torch.cuda.synchronize()
    want = flash_prefill_ref(q.float().numpy()[None], k.float().numpy()[None], v.float().numpy()[None], causal)[0]
    assert np.abs(out.float().cpu().numpy() - want).max() <= TOL[dtype]


def _random_split_cases(n=None, seed=83):
    n = case_count(6) if n is None else n
    rng = np.random.Generator(np.random.PCG64(case_seed(seed)))
    cases = []
    for i in range(n):
        hkv = int(rng.choice([1, 2, 4]))
        hq = hkv * int(rng.choice([2, 4, 8]))
        hq = min(hq, 16)
        lq = int(rng.integers(2048, 3300 if hq <= 8 else 2560))   # grids that leave resident slots free
        lk = lq if rng.random() < 0.6 else lq + int(rng.integers(1, 500))
        dtype = [torch.float16, torch.bfloat16][int(rng.integers(0, 2))]
        out_f32 = bool(rng.random() < 0.3)
        scale = 3.0 if rng.random() < 0.3 else 1.0
        cases.append((i, hq, hkv, lq, lk, dtype, out_f32, scale))
    return cases


@pytest.mark.parametrize("i,hq,hkv,lq,lk,dtype,out_f32,scale", _random_split_cases())
def test_random_split_key_halves(i, hq, hkv, lq, lk, dtype, out_f32, scale):
    """Seeded random causal prompts of 2048+ rows at head_dim 128 with few heads
    (1-16 query heads over 1-4 KV heads), so the 128-row kernel runs the longer
    query tiles as two key halves and merges them: Lk >= Lq, fp16 / bf16,
    outputs in the input type or fp32, and peaked scores; rows of the first and
    last KV groups' query heads against the oracle."""
    from tinyvllm_amd import _lib
    lib = _lib.load()
    assert lib.tv_flash_prefill_workspace_bytes(lq, lk, hq, 128, 128, 1, _lib.dtype_code(dtype), 0) > 0
    q = (randn(600 + i, lq, hq, 128) * scale).to(dtype)
    k = (randn(700 + i, lk, hkv, 128) * scale).to(dtype)
    v = randn(800 + i, lk, hkv, 128).to(dtype)
    out = _op()(q.unsqueeze(0).cuda(), k.unsqueeze(0).cuda(), v.unsqueeze(0).cuda(), True,
                out_dtype=torch.float32 if out_f32 else None)[0]
    torch.cuda.synchronize()
    _check_heads(out, q, k, v, True, sorted({0, hkv - 1}), dtype)


# ---- several prompts per launch (no reference counterpart) ------------------------------

@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lens,hq,hkv,d,causal", [
    ([512, 1024], 32, 4, 64, True),            # the TinyLlama prompts of the benchmark in one launch
    ([1, 17, 64, 300, 65], 8, 2, 64, True),    # ragged, single-token and tile-boundary prompts
    ([129, 7, 1000], 16, 8, 128, True),
    ([33, 200, 64], 8, 8, 64, False),
    ([300, 41, 512], 8, 2, 64, True),          # <= 256 work-groups with long rows: two key groups + LDS merge
    ([300, 41, 512], 8, 2, 128, True),
    ([2048, 300, 2200], 8, 2, 128, True),      # longest prompt >= 2048 at head_dim 128: the 128-row kernel
])
def test_varlen_matches_per_prompt(lens, hq, hkv, d, causal, dtype):
    """Every prompt of a packed batch equals the oracle on that prompt alone and
    the single-prompt launch (each within the fp16/bf16 bar)."""
    from tinyvllm_amd.attention import flash_prefill_varlen
    tot = sum(lens)
    q, k, v = randn(60, tot, hq, d, dtype=dtype), randn(61, tot, hkv, d, dtype=dtype), randn(62, tot, hkv, d, dtype=dtype)
    out = flash_prefill_varlen(q.cuda(), k.cuda(), v.cuda(), lens, causal)
    torch.cuda.synchronize()
    assert out.shape == (tot, hq, d) and out.dtype == dtype
    got = out.float().cpu().numpy()
    s = 0
    for n in lens:
        sl = slice(s, s + n)
        want = flash_prefill_ref(q[sl].float().numpy()[None], k[sl].float().numpy()[None],
                                 v[sl].float().numpy()[None], causal)[0]
        assert np.abs(got[sl] - want).max() <= TOL[dtype], (n, s)
        single = flash(q[sl], k[sl], v[sl], causal).float().cpu().numpy()
        assert np.abs(got[sl] - single).max() <= TOL[dtype], (n, s)
        s += n


def _random_varlen_cases(n=None, seed=73):
    n = case_count(8) if n is None else n
    rng = np.random.Generator(np.random.PCG64(case_seed(seed)))
    cases = []
    for i in range(n):
        hkv = int(rng.choice([1, 2, 4, 8]))
        hq = hkv * int(rng.choice([1, 2, 4, 8]))
        d = int(rng.choice([64, 128]))
        lens = [int(x) for x in rng.integers(1, 700, int(rng.integers(1, 6)))]
        causal = bool(rng.random() < 0.7)
        dtype = [torch.float16, torch.bfloat16][int(rng.integers(0, 2))]
        cases.append((i, lens, hq, hkv, d, causal, dtype))
    return cases


@pytest.mark.parametrize("i,lens,hq,hkv,d,causal,dtype", _random_varlen_cases())
def test_random_varlen(i, lens, hq, hkv, d, causal, dtype):
    """Seeded random packs of 1-5 prompts (lengths 1-699), GQA shapes, head
    dims, masks and dtypes: every prompt equals the oracle and its own launch."""
    test_varlen_matches_per_prompt(lens, hq, hkv, d, causal, dtype)


def test_varlen_fp32_output_and_strided_inputs():
    """fp32 output, and q/k/v as views into one fused [T, (Hq + 2 Hkv) * D] buffer."""
    from tinyvllm_amd.attention import flash_prefill_varlen
    lens = [70, 3, 130]
    tot, hq, hkv, d = sum(lens), 8, 2, 64
    fused = randn(70, tot, (hq + 2 * hkv) * d, dtype=torch.bfloat16).cuda()
    q = fused[:, :hq * d].view(tot, hq, d)
    k = fused[:, hq * d:(hq + hkv) * d].view(tot, hkv, d)
    v = fused[:, (hq + hkv) * d:].view(tot, hkv, d)
    out = flash_prefill_varlen(q, k, v, lens, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert out.dtype == torch.float32
    s = 0
    for n in lens:
        sl = slice(s, s + n)
        want = flash_prefill_ref(q[sl].float().cpu().numpy()[None], k[sl].float().cpu().numpy()[None],
                                 v[sl].float().cpu().numpy()[None], True)[0]
        assert np.abs(out[sl].cpu().numpy() - want).max() <= TOL[torch.bfloat16], n
        s += n


def test_varlen_plan_replays_in_graph():
    """The plan captured in a HIP graph: replays (with eager work between them)
    equal the eager launch."""
    from tinyvllm_amd.attention import VarlenPrefillPlan
    lens = [300, 41, 512]
    tot = sum(lens)
    q, k, v = (randn(63 + i, tot, h, 64, dtype=torch.float16).cuda() for i, h in enumerate((8, 2, 2)))
    plan = VarlenPrefillPlan(q, k, v, lens)
    eager = plan.run().clone()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            plan.run()
    torch.cuda.synchronize()
    for _ in range(3):
        plan.out.zero_()
        junk = torch.randn(1 << 20, device="cuda").sum()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(plan.out, eager)
        del junk


def test_varlen_rejects_bad_arguments():
    from tinyvllm_amd.attention import flash_prefill_varlen
    q = torch.zeros((10, 4, 64), dtype=torch.float16, device="cuda")
    k = torch.zeros((10, 2, 64), dtype=torch.float16, device="cuda")
    with pytest.raises(ValueError):
        flash_prefill_varlen(q, k, k, [4, 5])                  # lengths do not sum to T
    with pytest.raises(ValueError):
        flash_prefill_varlen(q, k, k, [10, 0])                 # empty prompt
    with pytest.raises(RuntimeError, match="head_dim 64 or 128"):
        flash_prefill_varlen(q.float(), k.float(), k.float(), [10])   # fp32: MFMA path only


# ---- a chunk attending through the paged cache (no reference counterpart) -----------------

def _paged_case(seed, total, hkv, d, bs, dtype, spare=5):
    """A sequence of `total` tokens' K/V scattered over a shuffled block pool."""
    rng = np.random.Generator(np.random.PCG64(seed))
    nblk = -(-total // bs)
    pool = nblk + spare
    table = rng.permutation(pool)[:nblk].astype(np.int32)
    k = randn(seed + 1, total, hkv, d, dtype=dtype)
    v = randn(seed + 2, total, hkv, d, dtype=dtype)
    kc = torch.zeros((pool, bs, hkv, d), dtype=dtype)
    vc = torch.zeros_like(kc)
    pos = np.arange(total)
    kc.view(pool * bs, hkv, d)[torch.from_numpy(table[pos // bs] * bs + pos % bs).long()] = k
    vc.view(pool * bs, hkv, d)[torch.from_numpy(table[pos // bs] * bs + pos % bs).long()] = v
    return k, v, kc, vc, table


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d,hq,hkv", [(64, 32, 4), (128, 8, 2)])
@pytest.mark.parametrize("start,n,bs,causal", [(0, 100, 16, True), (300, 77, 16, True), (1000, 256, 16, True),
                                               (64, 64, 4, True), (200, 50, 32, False), (3584, 512, 16, True)])
def test_paged_prefill_equals_last_rows_of_whole_prompt(dtype, d, hq, hkv, start, n, bs, causal):
    """flash_prefill_paged: a chunk at start_pos reading K/V through a shuffled
    block table equals the last n rows of prefill attention over the whole
    sequence (the oracle on the contiguous rows; causal bottom-right aligned,
    key j <= start + i), for block sizes 4, 16 and 32."""
    from tinyvllm_amd.attention import flash_prefill_paged
    total = start + n
    k, v, kc, vc, table = _paged_case(200 + start + n, total, hkv, d, bs, dtype)
    q = randn(97, total, hq, d, dtype=dtype)
    out = flash_prefill_paged(q[start:].cuda(), kc.cuda(), vc.cuda(), torch.from_numpy(table).cuda(), start, causal)
    torch.cuda.synchronize()
    want = flash_prefill_ref(q[start:].float().numpy()[None], k.float().numpy()[None], v.float().numpy()[None],
                             causal, q_offset=start)[0]
    assert np.abs(out[0].float().cpu().numpy() - want).max() <= TOL[dtype]


def _random_paged_prefill_cases(n=None, seed=77):
    n = case_count(8) if n is None else n
    rng = np.random.Generator(np.random.PCG64(case_seed(seed)))
    cases = []
    for i in range(n):
        hkv = int(rng.choice([1, 2, 4, 8]))
        hq = hkv * int(rng.choice([1, 2, 4, 8]))
        d = int(rng.choice([64, 128]))
        bs = int(rng.choice([4, 8, 16, 16, 32]))
        start = int(rng.integers(0, 1500))
        n_rows = int(rng.integers(1, 400))
        causal = bool(rng.random() < 0.8)
        dtype = [torch.float16, torch.bfloat16][int(rng.integers(0, 2))]
        cases.append((i, dtype, d, hq, hkv, start, n_rows, bs, causal))
    return cases


@pytest.mark.parametrize("i,dtype,d,hq,hkv,start,n,bs,causal", _random_paged_prefill_cases())
def test_random_paged_prefill(i, dtype, d, hq, hkv, start, n, bs, causal):
    """Seeded random chunks (start 0-1499, 1-399 rows) over shuffled block pools
    of block size 4-32: the chunk equals the last rows of the whole prompt."""
    test_paged_prefill_equals_last_rows_of_whole_prompt(dtype, d, hq, hkv, start, n, bs, causal)


@pytest.mark.parametrize("dtype,out_dtype", [(torch.float16, None), (torch.bfloat16, None),
                                             (torch.float16, torch.float32), (torch.bfloat16, torch.float32)])
def test_paged_prefill_invalid_block_id_gives_nan(dtype, out_dtype):
    # the NaNs are written as bit patterns (the kernel has no NaN arithmetic):
    # every element of the head's rows is a quiet NaN of the output type
    from tinyvllm_amd.attention import flash_prefill_paged
    k, v, kc, vc, table = _paged_case(5, 80, 2, 64, 16, dtype)
    table[2] = kc.shape[0] + 7
    q = randn(98, 16, 8, 64, dtype=dtype)
    out = flash_prefill_paged(q.cuda(), kc.cuda(), vc.cuda(), torch.from_numpy(table).cuda(), 64, True,
                              out_dtype=out_dtype)
    torch.cuda.synchronize()
    assert out.dtype == (dtype if out_dtype is None else out_dtype)
    assert torch.isnan(out.float()).all()


def test_paged_prefill_rejects_bad_arguments():
    from tinyvllm_amd.attention import flash_prefill_paged
    kc = torch.zeros((4, 16, 2, 64), dtype=torch.float16, device="cuda")
    q = torch.zeros((8, 4, 64), dtype=torch.float16, device="cuda")
    table = torch.zeros(2, dtype=torch.int32, device="cuda")
    with pytest.raises(ValueError):
        flash_prefill_paged(q, kc, kc, table, 30)                      # table covers 32 positions, needs 38
    kc3 = torch.zeros((4, 12, 2, 64), dtype=torch.float16, device="cuda")
    with pytest.raises(RuntimeError, match="power of two"):
        flash_prefill_paged(q, kc3, kc3, table, 0)


# ---- fp32 on split bf16 products (flash_prefill_f32.hip) -------------------------------

def attend_visible(q, k, v, causal, scale=None):
    """Float64 attention in which a key touches only the rows that see it."""
    hq, hkv = q.shape[1], k.shape[1]
    scale = q.shape[2] ** -0.5 if scale is None else scale
    q, k, v = (t.double().cpu().numpy() for t in (q, k, v))
    out = np.zeros(q.shape[:2] + v.shape[2:])
    with np.errstate(invalid="ignore", over="ignore"):
        for i in range(q.shape[0]):
            n = min(i + 1, k.shape[0]) if causal else k.shape[0]
            for h in range(hq):
                s = k[:n, h // (hq // hkv)] @ q[i, h] * scale
                e = np.exp(s - s.max())
                out[i, h] = (e @ v[:n, h // (hq // hkv)]) / e.sum()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("hq,hkv,lq,lk,causal", [(2, 1, 1, 1, True), (8, 2, 33, 33, True), (3, 3, 64, 64, True),
                                                 (4, 1, 97, 65, True), (2, 2, 130, 31, False), (1, 1, 70, 290, True),
                                                 (8, 1, 1100, 1100, True), (40, 8, 800, 800, True)])   # one / two key groups
def test_prefill_f32_split_products(d, hq, hkv, lq, lk, causal):
    """Tile edges, rows and keys past the last tile, both key groupings.  A score's error is
    a few roundings of the sum of its products' magnitudes; it moves a weight by as much, and
    the output by twice that of the largest value."""
    from tinyvllm_amd.attention import flash_prefill_attention
    q, k, v = (randn(300 + i, n, h, d).cuda() for i, (n, h) in enumerate([(lq, hq), (lk, hkv), (lk, hkv)]))
    out = flash_prefill_attention(q[None], k[None], v[None], causal)[0].double().cpu().numpy()
    rows = np.unique(np.concatenate([np.arange(min(lq, 70)), np.arange(max(0, lq - 70), lq)]))
    want = attend_visible(q, k, v, causal) if lq <= 200 else None
    if want is None:
        s = torch.einsum("qhd,khd->hqk", q[rows].double().cpu(), k.double().cpu().repeat_interleave(hq // hkv, 1))
        s = s * d ** -0.5
        if causal:
            s.masked_fill_(torch.arange(lk)[None, None] > torch.from_numpy(rows)[None, :, None], -np.inf)
        vv = v.double().cpu().repeat_interleave(hq // hkv, 1)
        want, out = torch.einsum("hqk,khd->qhd", torch.softmax(s, -1), vv).numpy(), out[rows]
    mag = float((q.abs().amax(1).amax(0) * k.abs().amax(1).amax(0)).sum()) * d ** -0.5
    tol = (2 * 4 * mag + 8) * 2.0 ** -24 * float(v.abs().max())
    assert np.abs(out - want).max() <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("hq,lq,lk,causal", [(8, 12, 12, True), (8, 13, 13, True), (2, 20, 20, True), (2, 21, 21, True),
                                             (32, 32, 32, True), (32, 33, 33, True), (16, 44, 44, True), (16, 45, 45, True), (4, 64, 64, True),
                                             (4, 300, 20, True), (4, 20, 300, True), (4, 3, 21, False), (4, 300, 12, False)])
def test_prefill_f32_few_keys(d, hq, lq, lk, causal):
    """Both sides of the line between the generic kernel and the one on split products."""
    from tinyvllm_amd.attention import flash_prefill_attention
    q, k, v = (randn(380 + i, n, h, d).cuda() for i, (n, h) in enumerate([(lq, hq), (lk, hq // 2), (lk, hq // 2)]))
    out = flash_prefill_attention(q[None], k[None], v[None], causal)[0].double().cpu().numpy()
    want = attend_visible(q, k, v, causal)
    # a score errs by a few 2^-24 of sum |q k|, about 2 sqrt(d) here, a weight and the output by as much
    assert np.linalg.norm(out - want) < 4 * d ** 0.5 * 2.0 ** -24 * np.linalg.norm(want)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n", [60, 150, 500])               # one, two, four key groups
def test_prefill_f32_parts_of_weights_and_values(d, n):
    """Equal values come out as they went in, whatever the weights: every part of a weight counts
    against the row sum, which holds it whole, and every part of the value.  Six products,
    their sum, the row sum's adds, the division and at most 2^-24 left out: 8 * 2^-24.  A part
    product that is lost is 2^-17 of the value, over the root of the keys that matter."""
    from tinyvllm_amd.attention import flash_prefill_attention
    hq, hkv = 16, 8
    q, k = randn(390, n, hq, d).cuda(), randn(391, n, hkv, d).cuda()
    bits = np.random.default_rng(392).integers(0, 1 << 23, (hkv, d)) | 0x3f800000
    bits[0], bits[1], bits[2] = 0x3f80ffff, 0x3f807fc0, 0x3f8080ff      # all low bits, the largest remainders
    v = torch.from_numpy(bits.astype(np.int32)).view(torch.float32).expand(n, hkv, d).contiguous().cuda()
    out = flash_prefill_attention(q[None], k[None], v[None])[0].double()
    want = v[0].double().repeat_interleave(hq // hkv, 0)
    assert ((out - want).abs() <= 8 * 2.0 ** -24 * want).all()


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
def test_prefill_f32_parts_of_scores(d):
    """Scores of one product each, x y / sqrt(d) = s against zero, with values 1 and -1: the output
    is tanh(s / 2).  s errs by at most 2.5 * 2^-24 of it (one part product lost: 2^-17), an
    exponential by 2^-22, and neither moves the output by more than half as much."""
    from tinyvllm_amd.attention import flash_prefill_attention
    n, m, hq, hkv = 64, 32, 32, 32
    rng = np.random.default_rng(393)

    def draw(*shape):
        bits = rng.integers(0, 1 << 23, shape) | 0x3f800000
        bits[::2] |= 0xffff
        return torch.from_numpy(bits.astype(np.int32)).view(torch.float32)

    x, y = draw(n, hq), draw(hkv)
    dim = torch.from_numpy(rng.permutation(np.arange(hkv) * (d // hkv)))       # every 32-element step has some
    q, k, v = torch.zeros(n, hq, d), torch.zeros(m, hkv, d), torch.zeros(m, hkv, d)
    q[:, torch.arange(hq), dim] = x
    k[0, torch.arange(hkv), dim] = y * d ** 0.5 / 2
    k[2:, torch.arange(hkv), dim] = -1e4
    v[0], v[1] = 1, -1
    out = flash_prefill_attention(q.cuda()[None], k.cuda()[None], v.cuda()[None], False)[0].double().cpu()
    s = x.double() * k[0, torch.arange(hkv), dim].double() * d ** -0.5
    assert ((out - torch.tanh(s / 2)[:, :, None]).abs() <= (2.5 * s[:, :, None] + 8) * 2.0 ** -24 / 2).all()


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
def test_prefill_f32_positive_sums(d):
    """Equal weights over 32768 positive values: the sum of a key group's 512 (or 256) tiles
    walks by at most 2^-24 of it per tile, about sqrt(512) 2^-24 = 1.3e-6 in the end; the row sum
    is exact.  (Low parts added to the whole sum one by one: 1e-5 and above.)"""
    from tinyvllm_amd.attention import flash_prefill_attention
    q = torch.zeros((1, 64, 2, d), device="cuda")
    k = randn(340, 1, 32768, 1, d).cuda()
    v = torch.rand((1, 32768, 1, d), generator=torch.Generator().manual_seed(341)).cuda()
    out = flash_prefill_attention(q, k, v, False)
    want = v[0, :, 0].double().mean(0)
    assert ((out.double() - want).norm() / want.norm() / (64 * 2) ** 0.5).item() < 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("eq,ek,ev", [(0, 0, -118), (0, 0, -130), (-118, 119, 0), (119, -118, 0), (0, 0, 100)])
def test_prefill_f32_range(d, eq, ek, ev):
    """Queries, keys and values scaled by powers of two lose no low bits.  A score's error is a
    few 2^-24 of sum |q k|, about 2 sqrt(d) here, and moves the output by as much; values
    near 2^-130 are rounded to 2^-149 once more on the way out, 2^-19 of the smallest outputs
    (0.1 of a value's size)."""
    from tinyvllm_amd.attention import flash_prefill_attention
    n, hq, hkv = 200, 4, 2
    q, k, v = (randn(350 + i, n, h, d).cuda() * 2.0 ** e for i, (h, e) in enumerate([(hq, eq), (hkv, ek), (hkv, ev)]))
    out = flash_prefill_attention(q[None], k[None], v[None])[0].double().cpu().numpy()
    want = attend_visible(q, k, v, True)
    err = np.linalg.norm(out - want) / np.linalg.norm(want)
    assert err < 4 * d ** 0.5 * 2.0 ** -24 + (2.0 ** -18 if ev == -130 else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n", [50, 300])         # one, two key groups
def test_prefill_f32_scores_that_overflow_on_the_way(d, n):
    """The products of a score pass -2^80 before they come back to +2^80: the last key takes all
    the weight, whatever the partial sums did."""
    from tinyvllm_amd.attention import flash_prefill_attention
    q, k = torch.zeros(n, 2, d), torch.zeros(n, 1, d)
    q[:] = 2.0 ** 40
    k[n - 1, 0, :d // 4] = -1.3 * 2.0 ** 35 * 128 / d
    k[n - 1, 0, d // 4:] = 0.9 * 2.0 ** 35 * 128 / d
    v = randn(360, n, 1, d)
    out = flash_prefill_attention(q.cuda()[None], k.cuda()[None], v.cuda()[None], False)[0].cpu()
    assert torch.equal(out, v[n - 1].expand(n, 2, d))


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
def test_prefill_f32_non_finite_values(d):
    """Infinities, NaN and values near the fp32 limit reach the rows that see them and no other."""
    from tinyvllm_amd.attention import flash_prefill_attention
    n, hq, hkv = 150, 4, 2
    q, k, v = (randn(310 + i, n, h, d).cuda() for i, h in enumerate([hq, hkv, hkv]))
    v[40, 0, 3] = float("inf")
    v[90, 0, 5] = float("nan")
    v[20, 1, 7] = 3.4e38
    k[120, 1, 2] = float("nan")
    out = flash_prefill_attention(q[None], k[None], v[None])[0].double().cpu().numpy()
    want = attend_visible(q, k, v, True)
    assert np.array_equal(np.isnan(out), np.isnan(want)) and np.array_equal(np.isposinf(out), np.isposinf(want))
    ok = np.isfinite(want)
    assert (np.abs(out - want)[ok] <= 2e-5 * np.maximum(1.0, np.abs(want[ok]))).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,start,bs", [(1000, 77, 16), (1024, 0, 4), (901, 640, 32)])
def test_prefill_paged_128_row_kernel(dtype, n, start, bs):
    """Grids of two 128-row work-groups per CU: prefixes and chunks that end inside a tile
    and inside a block, small blocks, and an invalid block id, which makes NaN of the query
    tiles that see it and of no other."""
    from tinyvllm_amd.attention import flash_prefill_paged
    hq, hkv, d = 64, 8, 128
    total = start + n
    nb = -(-total // bs) + 3
    q, kc, vc = (randn(320 + i, *s, dtype=dtype).cuda()
                 for i, s in enumerate([(n, hq, d), (nb, bs, hkv, d), (nb, bs, hkv, d)]))
    table = torch.from_numpy(np.random.default_rng(5).permutation(nb)[:-(-total // bs)].astype(np.int32)).cuda()
    out = flash_prefill_paged(q, kc, vc, table, start)[0].double().cpu()
    k, v = (c[table.long()].reshape(-1, hkv, d)[:total].double().cpu() for c in (kc, vc))
    rows = np.unique([0, 1, 31, 32, 127, 128, 500, n - 2, n - 1])
    for h in (0, 7, 8, 63):
        s = q[rows, h].double().cpu() @ k[:, h // 8].T.contiguous() / d ** 0.5
        s.masked_fill_(torch.arange(total)[None] > torch.from_numpy(rows)[:, None] + start, -np.inf)
        want = torch.softmax(s, -1) @ v[:, h // 8].contiguous()
        assert (out[rows, h] - want).abs().max() < TOL[dtype]
    bad = table.clone()
    at = (start + 300) // bs                      # seen by the query tiles from row 300 - bs on
    bad[at] = nb
    out = flash_prefill_paged(q, kc, vc, bad, start)[0]
    first = (at * bs - start) // 128 * 128        # first row of the first tile that sees the block
    assert torch.isnan(out[first:]).all() and torch.isfinite(out[:first]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_prefill_paged_128_row_kernel_divides_by_the_rounded_weights(dtype):
    """A weight is rounded to the input type on its way into P V; the row sum has to hold the
    rounded ones, so that the rounding cancels where one key dominates.  Here a weight w = 2^t,
    t in 6.5 .. 7.6 above a key of weight one and value zero, meets one value: the output is
    v w / (w + 1), and a relative error e of w (its rounding of 2^-9 at most, at fp16 the
    2^-11 t of the scaled queries) moves it by e / (w + 1), 7e-5 at most.  A sum of unrounded
    weights is off by the rounding itself, up to 2e-3 (bf16) and 4e-4 (fp16)."""
    from tinyvllm_amd.attention import flash_prefill_paged
    hq, hkv, d, n, start, bs = 64, 8, 128, 1000, 77, 16
    total = start + n
    nb = -(-total // bs)
    t = torch.linspace(6.5, 7.6, n * hq, dtype=torch.float64).reshape(n, hq)
    q = torch.zeros((n, hq, d), dtype=torch.float64)
    q[:, :, 0] = t / math.log2(math.e) * d ** 0.5 / 16
    k = torch.zeros((nb * bs, hkv, d), dtype=torch.float64)
    k[1:, :, 0], k[70, :, 0] = -64, 16
    v = torch.zeros((nb * bs, hkv, d), dtype=torch.float64)
    v[70] = randn(330, hkv, d).double()
    q, k, v = (x.to(dtype) for x in (q, k, v))
    table = torch.from_numpy(np.random.default_rng(6).permutation(nb).astype(np.int32))
    kc, vc = (torch.empty((nb, bs, hkv, d), dtype=dtype) for _ in range(2))
    kc[table.long()], vc[table.long()] = k.view(nb, bs, hkv, d), v.view(nb, bs, hkv, d)
    out = flash_prefill_paged(q.cuda(), kc.cuda(), vc.cuda(), table.cuda(), start, out_dtype=torch.float32)[0]
    out = out.double().cpu()
    w = torch.exp(q[:, :, 0].double() * 16 / d ** 0.5)
    want = v[70].double().repeat_interleave(hq // hkv, 0) * (w / (w + 1))[:, :, None]
    assert ((out - want).abs() <= 1e-4 * want.abs()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,out_dtype", [(torch.float16, None), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("row", [63, 64, 191, 340, 999])       # first row that sees the invalid block
def test_prefill_paged_128_row_kernel_invalid_block_in_half_a_tile(dtype, out_dtype, row):
    """The 64-row query tiles whose keys include an invalid block are NaN; the rows before them
    are those of a valid table, in the same 128-row tile too, whatever block 0 holds."""
    from tinyvllm_amd.attention import flash_prefill_paged
    hq, hkv, d, n, start, bs = 64, 8, 128, 1000, 64, 8
    nb = (start + n) // bs + 1
    q, kc, vc = (randn(370 + i, *s, dtype=dtype).cuda()
                 for i, s in enumerate([(n, hq, d), (nb, bs, hkv, d), (nb, bs, hkv, d)]))
    table = torch.arange(1, nb, dtype=torch.int32).cuda()       # block 0 is not the sequence's
    good = flash_prefill_paged(q, kc, vc, table, start, out_dtype=out_dtype)[0]
    kc[0], vc[0] = float("nan"), float("nan")
    for bad_id in (nb, -1):
        table[(start + row) // bs] = bad_id
        out = flash_prefill_paged(q, kc, vc, table, start, out_dtype=out_dtype)[0]
        first = row // bs * bs // 64 * 64
        assert torch.isnan(out[first:]).all() and torch.equal(out[:first], good[:first])


@pytest.mark.gpu
@pytest.mark.parametrize("blocks", [2048, 2049])              # the longest table of the 128-row kernel, and one more
def test_prefill_paged_128_row_kernel_longest_table(blocks):
    from tinyvllm_amd.attention import flash_prefill_paged
    hq, hkv, d, n, bs = 64, 8, 128, 1000, 4
    start = blocks * bs - n
    q, kc, vc = (randn(400 + i, *s, dtype=torch.bfloat16).cuda()
                 for i, s in enumerate([(n, hq, d), (blocks + 1, bs, hkv, d), (blocks + 1, bs, hkv, d)]))
    table = torch.from_numpy(np.random.default_rng(7).permutation(blocks + 1)[:blocks].astype(np.int32)).cuda()
    out = flash_prefill_paged(q, kc, vc, table, start)[0].double()
    k, v = (c[table.long()].reshape(-1, hkv, d).double() for c in (kc, vc))
    rows = torch.tensor([0, 1, 31, 32, 127, 128, 500, n - 2, n - 1]).cuda()
    for h in (0, 7, 8, 63):
        s = q[rows, h].double() @ k[:, h // 8].T.contiguous() / d ** 0.5
        s.masked_fill_(torch.arange(blocks * bs, device="cuda")[None] > rows[:, None] + start, -np.inf)
        want = torch.softmax(s, -1) @ v[:, h // 8].contiguous()
        assert (out[rows, h] - want).abs().max() < TOL[torch.bfloat16]
