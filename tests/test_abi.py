"""The C ABI: libtvattn.so loads on the host and exports exactly what include/*.h declares.

Only host-side entry points run here (no kernel launch): argument validation
paths return before any HIP call.
"""

import ctypes
import re
from pathlib import Path

import pytest

from tinyvllm_amd import _lib

HEADERS = sorted((Path(__file__).resolve().parents[1] / "include").glob("*.h"))


def header_text():
    return re.sub(r"/\*.*?\*/", "", "\n".join(h.read_text() for h in HEADERS), flags=re.S)


def declared_functions():
    return set(re.findall(r"^\s*(?:const\s+)?[a-z_0-9]+\s*\*?\s*(tv_[a-z_0-9]+)\s*\(", header_text(), flags=re.M))


def test_header_parses():
    names = declared_functions()
    assert {"tv_paged_decode", "tv_flash_prefill", "tv_reshape_and_cache", "tv_write_kv",
            "tv_read_kv_blocks", "tv_last_error", "tv_abi_version",
            "tv_paged_decode_workspace_bytes", "tv_linear", "tv_rms_norm_residual", "tv_qkv_rope_cache",
            "tv_argmax_advance", "tv_llama_decode_step", "tv_llama_prefill", "tv_llama_graph_create"} <= names


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    for name in declared_functions():
        assert hasattr(lib, name), f"{name} declared in include/ but not exported"
    assert set(_lib.SIGNATURES) == declared_functions()
    assert lib.tv_abi_version() == _lib.ABI_VERSION


def test_argument_counts_match_header():
    text = header_text()
    for name, (_, args) in _lib.SIGNATURES.items():
        m = re.search(name + r"\s*\(([^)]*)\)", text)
        params = [p for p in m.group(1).split(",") if p.strip() and p.strip() != "void"]
        assert len(params) == len(args), name


def test_workspace_size_is_host_arithmetic():
    lib = _lib.load()
    # prefill: L=1024 causal, 32 heads, D=64, split into chunks of one key tile:
    # 16 query tiles x max_chunks x 64 rows x (64 + 2) floats
    ws = lib.tv_flash_prefill_workspace_bytes(1024, 1024, 32, 64, 64, 1, 1, 1)
    unit = 32 * 16 * 64 * 66 * 4
    assert ws > 0 and ws % unit == 0 and ws // unit in (8, 16)      # 128- or 64-key tiles
    assert lib.tv_flash_prefill_workspace_bytes(1024, 1024, 32, 64, 64, 1, 1, 0) == 0      # default: no split
    assert lib.tv_flash_prefill_workspace_bytes(1024, 1024, 32, 64, 64, 1, 0, 4) == 0      # fp32: generic kernel
    assert lib.tv_paged_decode_workspace_bytes(4, 32, 64, 16, 16, 512) == 0      # one partition
    # one partition: the schedule (KV heads per row + order) only, in 256-byte units
    assert lib.tv_paged_decode_workspace_bytes(256, 32, 128, 256, 16, 4096) == 1280
    assert lib.tv_paged_decode_workspace_bytes(255, 32, 128, 256, 16, 4096) == 1024
    assert lib.tv_paged_decode_workspace_bytes(300, 32, 128, 256, 16, 4096) == 1280
    # 256 seqs x 32 heads x 8 partitions x (128 + 2) floats
    assert lib.tv_paged_decode_workspace_bytes(256, 32, 128, 256, 16, 512) == 256 * 32 * 8 * 130 * 4


def test_validation_errors_are_reported_without_launch():
    lib = _lib.load()
    rc = lib.tv_paged_decode(None, None, None, None, None, None, 1, 32, 8, 128, 16, 10, 4, 4,
                             0.1, 1, 1, 512, None, 0, None)
    assert rc == _lib.TV_EINVAL
    assert b"null pointer" in lib.tv_last_error()
    with pytest.raises(ValueError, match="null pointer"):
        _lib.check(rc, "tv_paged_decode")
    fake = ctypes.c_void_p(16)      # never dereferenced: rejected before any launch
    rc = lib.tv_paged_decode(fake, fake, fake, fake, fake, fake, 1, 32, 8, 96, 16, 10, 4, 4,
                             0.1, 1, 1, 512, None, 0, None)
    assert rc == _lib.TV_EUNSUPPORTED and b"head_dim 96" in lib.tv_last_error()
    rc = lib.tv_paged_decode(fake, fake, fake, fake, fake, fake, 1, 32, 8, 128, 16, 10, 4, 4,
                             0.1, 1, 1, 500, None, 0, None)
    assert rc == _lib.TV_EINVAL and b"partition_size" in lib.tv_last_error()
    rc = lib.tv_paged_decode(fake, fake, fake, fake, fake, fake, 1, 32, 8, 128, 16, 10, 64, 64,
                             0.1, 1, 1, 512, None, 0, None)
    assert rc == _lib.TV_EINVAL and b"workspace" in lib.tv_last_error()
    rc = lib.tv_write_kv(fake, fake, fake, fake, 10, 0, 1, 4, 64, 16, 10, 256, 256, 1, None)
    assert rc == _lib.TV_EINVAL and b"block_id" in lib.tv_last_error()
    rc = lib.tv_write_kv(fake, fake, fake, fake, 0, 10, 7, 4, 64, 16, 10, 256, 256, 1, None)
    assert rc == _lib.TV_EINVAL and b"do not fit" in lib.tv_last_error()
    rc = lib.tv_flash_prefill(fake, fake, fake, fake, 0, 4, 8, 8, 64, 64, 512, 512, 512, 512,
                              1, 0.1, 1, 1, 0, None, 0, None)
    assert rc == _lib.TV_EINVAL and b"empty" in lib.tv_last_error()
    rc = lib.tv_flash_prefill(fake, fake, fake, fake, 2048, 2048, 8, 2, 128, 128, 1024, 256, 256, 1024,
                              1, 0.1, 1, 1, 0, ctypes.c_void_p(24), 1 << 20, None)
    assert rc == _lib.TV_EINVAL and b"16-byte aligned" in lib.tv_last_error()
    rc = lib.tv_read_kv_blocks(fake, fake, fake, fake, fake, 1, 17, 4, 64, 16, 10, 1, None)
    assert rc == _lib.TV_EINVAL and b"exceeds" in lib.tv_last_error()


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", tmp_path / "absent.so")
    with pytest.raises(ImportError, match="no fallback"):
        _lib.load()


def test_no_bit_cast_of_vector_element_lvalues():
    """hipcc (ROCm 7.2) reads element 0 when __builtin_bit_cast is applied to an
    element of an ext_vector_type lvalue (v[i]); sources must go through a
    by-value helper such as u32_as_f32 instead."""
    csrc = Path(__file__).resolve().parents[1] / "tinyvllm_amd" / "csrc"
    bad = []
    for f in sorted(csrc.glob("*")):
        for n, line in enumerate(f.read_text().splitlines(), 1):
            if re.search(r"__builtin_bit_cast\(\s*\w+\s*,\s*\w+(\[[^\]]*\])+\s*\)", line):
                bad.append(f"{f.name}:{n}: {line.strip()}")
    assert not bad, "\n".join(bad)


def test_linear_split_choice():
    """K splits the decode step uses: about 192 work-groups, whole 256-wide K
    chunks, and one split once the output tiles alone fill half of that."""
    lib = _lib.load()
    assert lib.tv_linear_k_split(64, 2560, 2048) == 512        # q|k|v: 40 tiles x 4 splits
    assert lib.tv_linear_k_split(64, 2048, 2048) == 256        # output projection: 32 tiles x 8 splits
    assert lib.tv_linear_k_split(64, 2048, 5632) == 1024       # down projection: 32 tiles x 6 splits
    assert lib.tv_linear_k_split(64, 11264, 2048) == 2048      # w1|w3: 176 tiles, one split
    assert lib.tv_linear_k_split(1024, 2560, 2048) == 2048     # prefill rows fill the GPU
    assert lib.tv_linear_k_split(4, 96, 64) % 32 == 0


@pytest.mark.parametrize("dtype,M,N,K,splits,epilogue,tiled", [
    # measured faster on 64 x 64 tiles: little work for many rows
    ("F32", 65, 512, 512, 8, 0, False), ("F32", 128, 1024, 1024, 6, 0, False), ("F32", 65, 512, 4096, 16, 0, False),
    ("F32", 65, 1024, 4096, 1, 1, False), ("F32", 256, 1000, 2048, 1, 2, False), ("F32", 128, 5632, 1024, 1, 1, False),
    ("F32", 320, 512, 512, 4, 0, False), ("F16", 65, 1024, 1024, 6, 0, False), ("F16", 128, 512, 4096, 16, 0, False),
    ("BF16", 256, 4096, 256, 1, 0, False), ("BF16", 65, 2816, 1024, 1, 1, False), ("F16", 320, 1024, 4096, 1, 1, False),
    ("F16", 128, 1000, 2048, 1, 2, False),
    # and on the tiled kernels
    ("F32", 300, 11264, 2048, 1, 1, True), ("F32", 512, 32000, 2048, 1, 2, True), ("F32", 300, 2048, 5632, 8, 0, True),
    ("F16", 1000, 2560, 2048, 1, 0, True), ("BF16", 2048, 32768, 4096, 1, 1, True), ("F16", 300, 2048, 5632, 4, 0, True),
    ("F16", 128, 11264, 2048, 1, 1, True), ("BF16", 128, 32000, 2048, 1, 2, True)])
def test_kernel_of_a_many_row_product(dtype, M, N, K, splits, epilogue, tiled):
    """More than 64 rows go to the tiled kernels only where those are the faster ones."""
    ks = -(-K // splits // 32) * 32
    kernel = _lib.load().tv_linear_kernel(M, N, K, ks, epilogue, getattr(_lib, "TV_" + dtype))
    assert kernel >= 2 if tiled else kernel == 0


def test_a_planned_split_takes_the_kernel_it_was_planned_for():
    """300 rows of 2048 x 2048 at fp32 are split eight ways for the tiled kernel (26 us); at that
    split alone the estimates differ by 5%, and 64 x 64 tiles take 34."""
    lib = _lib.load()
    assert lib.tv_linear_kernel(300, 2048, 2048, 256, 0, _lib.TV_F32) >= 2
    for M, N, K in ((1000, 2560, 2048), (300, 2048, 5632), (16, 2048, 2048), (65, 2048, 2048), (16, 4096, 1024)):
        ks = lib.tv_linear_k_split(M, N, K)
        want = {(16, 4096, 1024): 0}.get((M, N, K), 1 if M <= 16 else 2)
        kernel = lib.tv_linear_kernel(M, N, K, ks, 0, _lib.TV_F16)
        assert kernel >= 2 if want == 2 else kernel == want


@pytest.mark.parametrize("dtype,M,N,K,epilogue,few", [
    # measured faster on 64 x 64 tiles: one or two chunks of K under many features
    ("F16", 4, 32768, 256, 1, False), ("F16", 16, 32768, 512, 1, False), ("BF16", 4, 8192, 256, 1, False),
    ("F16", 16, 16384, 384, 1, False), ("F16", 4, 16384, 256, 0, False), ("F32", 4, 32768, 128, 1, False),
    ("F32", 16, 16384, 128, 0, False), ("F16", 16, 32000, 256, 2, False),
    # and on the kernel that streams W past few rows
    ("F16", 4, 11264, 2048, 1, True), ("BF16", 16, 5632, 512, 1, True), ("F16", 16, 32768, 768, 1, True),
    ("F16", 1, 32000, 2048, 2, True), ("F32", 16, 11264, 2048, 1, True), ("F32", 4, 8192, 256, 1, True),
    ("F32", 16, 32000, 128, 2, True), ("F16", 16, 6144, 2048, 0, True)])
def test_kernel_of_a_few_row_product(dtype, M, N, K, epilogue, few):
    kernel = _lib.load().tv_linear_kernel(M, N, K, K, epilogue, getattr(_lib, "TV_" + dtype))
    assert kernel == (1 if few else 0)


@pytest.mark.parametrize("dtype,es", [("F32", 4), ("F16", 2), ("BF16", 2)])
def test_products_of_rows_beyond_32_bit_offsets_are_refused(dtype, es):
    """16 rows of W and 64 of A have to lie within 4 GiB, or 16 of both within 2 GiB for at most 16
    rows (nothing is launched)."""
    lib, p = _lib.load(), 0x1000
    code = getattr(_lib, "TV_" + dtype)

    def refused(M, K, lda):
        rc = lib.tv_linear(p, p, p, M, 64, K, lda, 0, K, 0, None, code, None)
        return rc == _lib.TV_EUNSUPPORTED and b"32-bit" in lib.tv_last_error()

    assert refused(4, (1 << 32) // (16 * es) + 32, (1 << 32) // (16 * es) + 32)
    for M in (2, 4, 16):
        assert refused(M, 64, (1 << 31) // (16 * es))
    for M in (17, 64, 65, 1000):
        assert refused(M, 64, (1 << 32) // (64 * es) + 8)


@pytest.mark.parametrize("dtype", ["F32", "F16", "BF16"])
@pytest.mark.parametrize("dim,heads,kv_heads,hidden", [(2048, 32, 4, 5632), (4096, 32, 8, 16384), (1024, 16, 4, 2816),
                                                       (512, 8, 2, 1376), (64, 4, 2, 256), (768, 12, 12, 3072)])
def test_a_prefill_workspace_serves_every_smaller_count(dtype, dim, heads, kv_heads, hidden):
    """A caller sizes one buffer for its longest prompt.  Shorter ones are split further along K,
    so they can hold more partials than a long one."""
    from tinyvllm_amd.llama import _Model
    lib = _lib.load()
    m = _Model(n_layers=1, dim=dim, n_heads=heads, n_kv_heads=kv_heads, head_dim=dim // heads, hidden_dim=hidden,
               vocab_size=32000, dtype=getattr(_lib, "TV_" + dtype))
    need = [lib.tv_llama_prefill_workspace_bytes(ctypes.byref(m), n) for n in range(1, 2200)]
    assert all(a <= b for a, b in zip(need, need[1:]))
    if dtype != "F32":
        qd, nqkv = dim, dim + 2 * kv_heads * (dim // heads)
        for n in list(range(1, 70)) + list(range(96, 2200, 37)):
            for N, K in ((nqkv, dim), (dim, qd), (dim, hidden)):
                assert -(-K // lib.tv_linear_k_split(n, N, K)) * n * N * 4 <= need[n - 1]


def test_dense_entry_points_validate_on_host():
    lib = _lib.load()
    p = ctypes.c_void_p(256)
    # K not a multiple of 32, N not a multiple of 4, bad dtype, multi-split logits
    assert lib.tv_linear(p, p, p, 4, 64, 48, 48, 0, 48, 0, None, _lib.TV_F16, None) == _lib.TV_EUNSUPPORTED
    assert lib.tv_linear(p, p, p, 4, 66, 64, 64, 0, 64, 0, None, _lib.TV_F16, None) == _lib.TV_EUNSUPPORTED
    assert lib.tv_linear(p, p, p, 4, 64, 64, 64, 0, 64, 0, None, 7, None) == _lib.TV_EUNSUPPORTED   # no such dtype
    assert lib.tv_linear(p, p, p, 4, 64, 64, 64, 64, 32, 2, None, _lib.TV_F16, None) == _lib.TV_EINVAL
    assert b"one split" in lib.tv_last_error()
    assert lib.tv_qkv_rope_cache(p, None, None, p, None, p, 1, None, 0, p, 8, p, 0, 1, 16, 4, 1, 4, 2, 16,
                                 _lib.TV_F16, None, None, None) == _lib.TV_EINVAL
    assert lib.tv_llama_decode_step(None, None, None, None) == _lib.TV_EINVAL
    assert lib.tv_llama_graph_create(None, None, None, None, None) == _lib.TV_EINVAL


def test_decode_step_workspace_tinyllama():
    """Workspace of the TinyLlama-1.1B step at batch 64 (the end-to-end decode workload)."""
    from tinyvllm_amd.llama import LlamaConfig, _Model
    c = LlamaConfig.tinyllama_1b()
    m = _Model(c.n_layers, c.dim, c.n_heads, c.n_kv_heads, c.head_dim, c.hidden_dim, c.vocab_size, _lib.TV_F16,
               c.norm_eps)
    lib = _lib.load()
    ws = lib.tv_llama_decode_workspace_bytes(ctypes.byref(m), 64, 72, 16, 2048)
    # 8 split partials of the widest product + activations + 500 x 64 argmax keys
    assert 64 * 2560 * 8 * 4 < ws < 16 << 20
    assert lib.tv_llama_decode_workspace_bytes(ctypes.byref(m), 0, 72, 16, 2048) == 0


def test_noalloc_rejects_oversize_launch_on_the_host():
    """tv_paged_decode_noalloc checks the launch against its 16 MiB per-device
    scratch before any HIP call: a launch needing more fails with TV_EINVAL."""
    lib = _lib.load()
    assert lib.tv_paged_decode_workspace_bytes(64, 32, 128, 2048, 16, 256) > (16 << 20)
    rc = lib.tv_paged_decode_noalloc(None, None, None, None, None, None, 64, 32, 8, 128, 16, 100, 2048, 2048,
                                     0.1, _lib.TV_F16, _lib.TV_F16, 256, None)
    assert rc == _lib.TV_EINVAL and b"scratch" in lib.tv_last_error()
