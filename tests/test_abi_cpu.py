"""CPU-side checks of the boundary: the shared library loads without a GPU and exports exactly the symbols that
include/mtj_abi.h declares; the Python binding covers every one of them; argument validation that needs no
device works.  No kernel is launched here."""
import ctypes
import os
import re

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "mtj_abi.h")


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mtj_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_entry_points():
    syms = declared_symbols()
    for s in ("mtj_version", "mtj_last_error", "mtj_pack_weight", "mtj_embed", "mtj_layernorm", "mtj_gemm", "mtj_gemv",
              "mtj_attn_prefill", "mtj_attn_decode", "mtj_attn_decode_work_bytes", "mtj_sample_greedy",
              "mtj_sample_nucleus", "mtj_sample_work_bytes", "mtj_gemv_greedy"):
        assert s in syms


def test_library_exports_every_declared_symbol_and_binding_covers_them():
    from mesh_transformer import _abi
    lib = _abi.lib()                      # raises if the library is missing: there is no fallback path
    syms = declared_symbols()
    for s in syms:
        assert hasattr(lib, s), f"{s} is declared in mtj_abi.h but not exported by libmtj_hip.so"
    assert sorted(_abi.SIGNATURES) == syms
    assert lib.mtj_version() == _abi.ABI_VERSION


def test_struct_layouts_match_the_header():
    from mesh_transformer import _abi
    # field order of mtj_inproj / mtj_next_embed as written in the header
    text = open(HEADER).read()
    body = text[text.index("typedef struct {"):text.index("} mtj_inproj;")]
    names = re.findall(r"\b([a-zA-Z_0-9]+)\s*(?:,|;)", re.sub(r"/\*.*?\*/", "", body, flags=re.S))
    assert names == [f[0] for f in _abi.InProj._fields_]
    assert ctypes.sizeof(_abi.InProj) % 8 == 0
    body = text[text.index("typedef struct {", text.index("mtj_inproj;")):text.index("} mtj_attn_merge;")]
    names = re.findall(r"\b([a-zA-Z_0-9]+)\s*(?:,|;)", re.sub(r"/\*.*?\*/", "", body, flags=re.S))
    assert names == [f[0] for f in _abi.AttnMerge._fields_]
    body = text[text.index("typedef struct {", text.index("mtj_attn_merge;")):text.index("} mtj_next_embed;")]
    names = re.findall(r"\b([a-zA-Z_0-9]+)\s*(?:,|;)", re.sub(r"/\*.*?\*/", "", body, flags=re.S))
    assert names == [f[0] for f in _abi.NextEmbed._fields_]


def test_argument_validation_needs_no_device():
    from mesh_transformer import _abi
    lib = _abi.lib()
    # shape errors are reported before anything touches the GPU
    assert lib.mtj_layernorm(None, None, None, 1, 8, None, 0, None) == -1
    assert b"null pointer" in lib.mtj_last_error()
    with pytest.raises(ValueError):
        _abi.check(lib.mtj_gemv(None, None, None, None, None, 8, 8, 0, 0, None, 0, None, None, None))
    # one sequence of 16 heads: 8 key ranges per head (128 workgroups); 32 sequences fill the chip with one range each
    assert lib.mtj_attn_decode_splits(1, 16, 2047) == 8 and lib.mtj_attn_decode_splits(32, 16, 2047) == 1
    assert lib.mtj_attn_decode_splits(1, 16, 20) == 2          # never fewer than 16 slots per range at a full window
    assert lib.mtj_attn_decode_work_bytes(1, 16, 256, 2047) == 16 * 8 * 260 * 4
    # in one launch: a line for the counter and up to 16 (8 from 65 pairs on) partials of whole lines per (sequence, head)
    assert lib.mtj_attn_decode_joined_work_bytes(3, 16, 256, 2047) == 48 * (128 + 16 * 288 * 4)
    assert lib.mtj_attn_decode_joined_work_bytes(64, 16, 64, 2047) == 1024 * (128 + 8 * 96 * 4)
    for B, H, Tcap in ((65, 16, 100), (64, 4096, 10000), (1, 0, 5), (0, 16, 5), (2, 16, 0)):
        assert lib.mtj_attn_decode_joined_work_bytes(B, H, 256, Tcap) == 0
    assert lib.mtj_attn_decode_joined(*[None] * 4, 65, 16, 100, 256, None, 4096, 0, 2, None, None) == -5
    assert lib.mtj_attn_decode_joined(*[None] * 4, 2, 16, 100, 256, None, 4096, 0, 2, None, None) == -1
    assert lib.mtj_sample_work_bytes(32, 50400) == 256         # kept in the ABI; the sampler sorts nothing


def test_host_tensors_are_refused():
    import torch
    from mesh_transformer import _abi
    with pytest.raises(ValueError):
        _abi.ptr(torch.zeros(4))
    assert _abi.ptr(None) is None


def test_product_fails_loudly_without_a_gpu():
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is visible")
    from mesh_transformer.transformer_shard import CausalTransformer
    cfg = dict(layers=1, d_model=64, n_heads=1, n_vocab=64, pe="rotary", cores_per_replica=1)
    with pytest.raises(RuntimeError):
        CausalTransformer(cfg)
    from mesh_transformer import sampling
    with pytest.raises(RuntimeError):
        sampling.nucleaus_filter(np.zeros((1, 8), np.float32))


def test_util_casts():
    import torch
    from mesh_transformer.util import to_bf16, to_f32
    t = {"a": {"w": torch.ones(2, 2), "i": torch.ones(2, dtype=torch.int32)}}
    b = to_bf16(t)
    assert b["a"]["w"].dtype == torch.bfloat16 and b["a"]["i"].dtype == torch.int32
    assert to_f32(b)["a"]["w"].dtype == torch.float32


def test_session_workspace_covers_every_prompt_length():
    """The out projection of a prefill is cut into MORE K ranges the FEWER rows it has, so the workspace of a session
    sized for its longest prompt must also hold the partials of every shorter one (host-side sizes only)."""
    from mesh_transformer import _abi
    from mesh_transformer.engine import splitk_work_bound
    lib = _abi.lib()
    for dtype in (_abi.F32, _abi.F16, _abi.BF16):
        for M_max, N, K in ((8 * 599, 4096, 20480), (700, 512, 2560), (2047, 4096, 20480), (100, 4096, 20480)):
            bound = splitk_work_bound(M_max, N, K, dtype)
            need = max(lib.mtj_gemm_splitk_work_bytes(m, N, K, dtype) for m in range(1, M_max + 1))
            assert bound == need, (dtype, M_max, N, K)
    # the case that used to fail: a session first sized for 8 x 599 rows, later used with 8 x 99
    assert lib.mtj_gemm_splitk_work_bytes(8 * 99, 4096, 20480, _abi.F16) > lib.mtj_gemm_splitk_work_bytes(8 * 599, 4096, 20480, _abi.F16)


def test_splitk_takes_the_workspace_of_more_rows():
    """float32: the faster cuts are taken where the workspace holds them, and nothing is refused for want of them - neither the
    workspace that the query asks for nor that of 199 rows with fewer rows; a session holds the fastest cut of every prompt."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("the pointers of this test must never reach a GPU")
    from mesh_transformer import _abi
    from mesh_transformer.engine import splitk_work_bound
    lib, P, N, K = _abi.lib(), 1 << 20, 4096, 20480
    need = lambda m: lib.mtj_gemm_splitk_work_bytes(m, N, K, 0)
    best = lambda m: lib.mtj_gemm_splitk_best_work_bytes(m, N, K, 0)
    for m in (65, 100, 128, 150, 199, 256, 300, 511, 700):
        assert need(m) == (4 if m <= 512 else 2) * m * N * 4 and best(m) in (need(m), 2 * need(m), 4 * need(m)), m
        for have in (need(m), max(need(m), need(199)), best(m) - 4, best(m)):
            for rc in (lib.mtj_gemm_splitk(P, K, P, P, m, N, K, 0, _abi.EPI_RESID, P, N, 0, P, have, 1.0, None),
                       lib.mtj_gemm_splitk_ln(P, K, P, P, m, N, K, 0, P, N, P, have, P, P, P, N, 0, 1.0, None)):
                assert rc == -4 if have >= need(m) else rc == -1, (m, have, rc)
    assert best(128) == 16 * 128 * N * 4 and need(199) >= need(128)
    for M_max in (100, 700, 2047):
        assert splitk_work_bound(M_max, N, K, 0, best=True) == max(best(m) for m in range(1, M_max + 1))
    for dtype in (1, 2):
        for M, n, k in _splitk_sizes():
            assert lib.mtj_gemm_splitk_best_work_bytes(M, n, k, dtype) == lib.mtj_gemm_splitk_work_bytes(M, n, k, dtype)


def _needs_ranges(lib, M, N, K, dtype):
    """The products that mtj_gemm_splitk has always cut into K ranges, and for which it asks for rows that its reduce can
    take: ranges are doubled while they are no more than the CUs (128-column tiles, 256 x 256 tiles) or two per CU
    (128 x 128 tiles) and keep 4 or 16 k-tiles each."""
    from mesh_transformer import _abi
    up = lambda a, b: -(-a // b)
    kt = K // (32 if dtype == _abi.F32 else 64)
    if N % 4:
        return False

    def doubled(tiles, limit, most, least):
        s = 1
        while s < most and tiles * s * 2 <= limit and kt % (s * 2) == 0 and kt // (s * 2) >= least:
            s *= 2
        return s
    if M <= 64:
        return doubled(up(N, 128), 256, 16, 4) > 1
    if dtype != _abi.F32:
        big = up(M, 256) * up(N, 256)
        s = doubled(big, 256, 16, 16)
        if big * s >= 200:
            return s > 1
    return doubled(up(M, 128) * up(N, 128), 512, 4, 16) > 1


def _splitk_sizes():
    for M in (1, 33, 64, 65, 100, 128, 129, 200, 256, 257, 384, 700, 1025, 1808, 2048, 3195, 4097, 9000):
        for N in (64, 408, 512, 1024, 2048, 4096, 4098, 8192, 16384, 25600, 32768):
            for K in (64, 256, 512, 704, 1024, 1984, 2048, 2560, 4096, 20480):
                yield M, N, K


@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_splitk_takes_rows_of_any_alignment_where_it_need_not_cut(dtype):
    """An `out` whose rows are no whole number of quads, an unaligned out and an unaligned bias are refused only where the
    product is always cut into K ranges; elsewhere the call passes the checks (and then finds no device here)."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("the pointers of this test must never reach a GPU")
    from mesh_transformer import _abi
    lib, P = _abi.lib(), 1 << 20
    for M, N, K in _splitk_sizes():
        nb = lib.mtj_gemm_splitk_work_bytes(M, N, K, dtype)
        for out, bias, ldo in ((P, P, N + 2), (P + 4, P, N), (P, P + 4, N)):
            rc = lib.mtj_gemm_splitk(P, K, P, bias, M, N, K, dtype, _abi.EPI_RESID, out, ldo, 0, P, nb, 1.0, None)
            refused = rc == -1
            assert rc in (-1, -4) and refused == _needs_ranges(lib, M, N, K, dtype), (M, N, K, out, bias, ldo, rc)


@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_splitk_ln_takes_padded_rows_where_it_always_cuts(dtype):
    """x and h with padded rows: taken exactly where the product is always cut into K ranges, and then every row goes
    through the reduce (the workspace holds whole copies of the output), since the separate LayerNorm wants dense rows."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("the pointers of this test must never reach a GPU")
    from mesh_transformer import _abi
    lib, P = _abi.lib(), 1 << 20
    for M, N, K in _splitk_sizes():
        if N % 4 or N > 16384:
            continue
        nb = lib.mtj_gemm_splitk_work_bytes(M, N, K, dtype)
        need = _needs_ranges(lib, M, N, K, dtype)
        if need:
            assert nb >= 2 * M * N * 4 and nb % (M * N * 4) == 0, (M, N, K, nb)
        for ldx, ldh in ((N + 8, N), (N, N + 8), (N, N)):
            rc = lib.mtj_gemm_splitk_ln(P, K, P, P, M, N, K, dtype, P, ldx, P, nb, P, P, P, ldh, dtype, 1.0, None)
            assert (rc == -1) == (not need and (ldx, ldh) != (N, N)), (M, N, K, ldx, ldh, rc)


@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_splitk_without_a_workspace_where_it_need_not_cut(dtype):
    """No workspace, or one that is too small: refused where the product is always cut into K ranges, one range elsewhere -
    also where a cut would be faster."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("the pointers of this test must never reach a GPU")
    from mesh_transformer import _abi
    lib, P = _abi.lib(), 1 << 20
    for M, N, K in _splitk_sizes():
        nb = lib.mtj_gemm_splitk_work_bytes(M, N, K, dtype)
        refused = _needs_ranges(lib, M, N, K, dtype) and nb > 0
        for work, have in ((None, nb), (P, nb - 4), (P + 4, nb)):
            if nb == 0 and have < 0:
                continue
            rc = lib.mtj_gemm_splitk(P, K, P, P, M, N, K, dtype, _abi.EPI_RESID, P, N, 0, work, have, 1.0, None)
            assert rc in (-1, -4) and (rc == -1) == refused, (M, N, K, work, have, rc)
            if N % 4 == 0 and N <= 4096:                      # (the separate LayerNorm takes no longer rows)
                rc = lib.mtj_gemm_splitk_ln(P, K, P, P, M, N, K, dtype, P, N, work, have, P, P, P, N, dtype, 1.0, None)
                assert rc in (-1, -4) and (rc == -1) == refused, (M, N, K, work, have, rc)


def test_torch_ops_are_registered_for_the_gpu_only():
    """Every kernel entry point is a dispatcher-visible operator torch.ops.mtj.*; there is no CPU implementation, so
    host tensors are refused by the dispatcher instead of taking another path."""
    import torch
    from mesh_transformer import ops
    for name in ops.OPS:
        assert hasattr(torch.ops.mtj, name), name
    assert "Tensor(a!)" in str(torch.ops.mtj.gemm_resid_.default._schema)
    with pytest.raises((NotImplementedError, RuntimeError)):
        torch.ops.mtj.layernorm(torch.zeros(2, 8), torch.ones(8), torch.zeros(8), 0)
