"""C-ABI checks that need no GPU: the library loads and exports every symbol
that ``include/kch.h`` declares, with the declared version."""

from __future__ import annotations

import ctypes
import os
import re

import pytest
from conftest import REPO

HEADER = os.path.join(REPO, "include", "kch.h")


def _declared():
    src = open(HEADER).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"\b(kch_[a-z0-9_]+)\s*\(", src)))


def test_header_declares_entry_points():
    names = _declared()
    assert "kch_abi_version" in names and "kch_last_error" in names
    assert "kch_kda_chunk_fwd" in names


def test_library_exports_every_declared_symbol():
    from kch import _lib
    lib = _lib.load()
    for name in _declared():
        assert hasattr(lib, name), f"libkch.so does not export {name}"
    version = int(re.search(r"#define KCH_ABI_VERSION (\d+)", open(HEADER).read()).group(1))
    assert lib.kch_abi_version() == version


def test_python_binding_covers_header():
    from kch import _lib
    assert set(_declared()) == set(_lib.EXPORTED)


def test_invalid_arguments_report_errors_without_gpu():
    # argument validation happens before any HIP call
    from kch import _lib
    lib = _lib.load()
    rc = lib.kch_kda_chunk_fwd(None, None, None, None, None, None, None, None,
                               1, 8, 3, 4, 128, 128, ctypes.c_float(1.0),
                               ctypes.c_float(-10.0), 1, None)
    assert rc == 1
    assert b"divisible" in lib.kch_last_error()
    rc = lib.kch_kda_chunk_fwd(None, None, None, None, None, None, None, None,
                               1, 8, 2, 2, 96, 128, ctypes.c_float(1.0),
                               ctypes.c_float(-10.0), 1, None)
    assert rc == 2
    # kch_linear_rows: row count and K checked before any pointer or HIP call
    rc = lib.kch_linear_rows(None, 64, None, 64, None, 8, 17, 8, 64, 1, None)
    assert rc == 2 and b"M=17" in lib.kch_last_error()
    rc = lib.kch_linear_rows(None, 64, None, 64, None, 8, 2, 8, 48, 1, None)
    assert rc == 2 and b"multiple of 32" in lib.kch_last_error()
    # the prefill projections: sizes checked before any pointer or HIP call
    rc = lib.kch_linear_up(None, 48, None, 48, None, 8, 4, 8, 48, 1, None)
    assert rc == 2 and b"K=48" in lib.kch_last_error()
    rc = lib.kch_linear_up(None, 64, None, 64, None, 8, 4, 8, 64, 0, None)
    assert rc == 2 and b"bf16 or fp16" in lib.kch_last_error()
    rc = lib.kch_linear_up(None, 64, None, 64, None, 8, 4, 8, 64, 1, None)
    assert rc == 1 and b"null pointer" in lib.kch_last_error()
    assert lib.kch_linear_up(None, 64, None, 64, None, 8, 0, 8, 64, 1, None) == 0


def test_kda_backward_validation_and_workspace():
    """kch_kda_recurrent_bwd: sizes checked before any pointer or HIP call; the
    workspace is the checkpoints (one state slice per segment) plus one
    partial record (3K + 1 values) per (b, t, hv, 16-column slice)."""
    from kch import _lib
    lib = _lib.load()
    P = [None] * 14
    rc = lib.kch_kda_recurrent_bwd(*P, 1, 8, 2, 2, 48, 16, 0.25, -10.0, 0, None, 0, None)
    assert rc == 2 and b"K=48" in lib.kch_last_error()
    rc = lib.kch_kda_recurrent_bwd(*P, 1, 0, 2, 2, 64, 16, 0.25, -10.0, 0, None, 0, None)
    assert rc == 1 and b"T >= 1" in lib.kch_last_error()
    rc = lib.kch_kda_recurrent_bwd(*P, 1, 8, 2, 2, 64, 16, 0.25, -10.0, 7, None, 0, None)
    assert rc == 1 and b"dtype" in lib.kch_last_error()
    rc = lib.kch_kda_recurrent_bwd(*P, 1, 8, 2, 2, 64, 16, 0.25, -10.0, 3, None, 0, None)
    assert rc == 1 and b"null" in lib.kch_last_error()
    assert lib.kch_kda_recurrent_bwd_ws_bytes(1, 8, 2, 48, 16, 0) == 0
    pad = lambda x: (x + 255) // 256 * 256  # noqa: E731
    # 16-column slices; K = 128: 8-token segments (fp32), 4 (fp64: LDS)
    B, T, HV, K, V = 2, 100, 3, 128, 40
    nvs = (V + 15) // 16
    for code, acc, seg in ((0, 4, 8), (1, 4, 8), (3, 8, 4)):
        ck = B * HV * nvs * (-(-T // seg)) * K * 16 * acc
        part = B * T * HV * nvs * (3 * K + 1) * acc
        assert lib.kch_kda_recurrent_bwd_ws_bytes(B, T, HV, K, V, code) == pad(ck) + pad(part)


def _csa_bwd_status(lib, B, T, nh, c, m, topk, win, normalize, slots=True, dsel=False, dsel_add=0):
    """kch_csa_attn_bwd without a workspace: the call ends before any tensor is read."""
    x = ctypes.c_void_p(4096)
    return lib.kch_csa_attn_bwd(x, x, x, x, x, x, c, x, c, x, c, x, c, x, x, None, x, x, x, x, x, x, x,
                                None, x if slots else None, x if dsel else None, dsel_add, None, B, T,
                                nh, c, m, topk, win, 1.0, normalize, 0, 0, 0, None, 0, None)


def _csa_bwd_needs(lib, *sizes, **kw):
    """The workspace that kch_csa_attn_bwd says a call without one requires."""
    assert _csa_bwd_status(lib, *sizes, **kw) == 1
    return int(re.search(rb"workspace of (\d+) bytes", lib.kch_last_error()).group(1))


def test_csa_backward_workspace_holds_every_head_group():
    """Head groups share one workspace, sized for the first: a last group of 16
    or fewer heads needs no more than the whole ones before it (32 heads of 64
    on raw rows, 16 on normalised ones)."""
    from kch import _lib
    lib = _lib.load()
    for B, T, c, m, topk, win in ((1, 64, 64, 4, 4, 8), (2, 4096, 64, 4, 64, 128), (1, 1024, 128, 1, 8, 0)):
        for normalize, most in ((0, 256 // (c // 8)), (1, 16)):
            held = lib.kch_csa_attn_bwd_ws_bytes(B, T, most, c, m, win, topk)
            for nh in range(1, most + 1):
                assert _csa_bwd_needs(lib, B, T, nh, c, m, topk, win, normalize) <= held, (nh, normalize)


def test_csa_backward_refuses_slots_beside_an_added_dsel():
    """The slots would be read from a dsel that holds earlier calls' values too."""
    from kch import _lib
    lib = _lib.load()
    assert _csa_bwd_status(lib, 1, 64, 16, 64, 4, 8, 8, 1, dsel=True, dsel_add=1) == 2
    assert b"slot_grad" in lib.kch_last_error()
    for kw in (dict(dsel=True), dict(slots=False, dsel=True, dsel_add=1), dict(dsel_add=1)):
        assert _csa_bwd_needs(lib, 1, 64, 16, 64, 4, 8, 8, 1, **kw) > 0


def test_attention_backward_of_many_heads_takes_contiguous_rows_only():
    """More than 16 heads a call run on kernels that read contiguous rows: a row
    stride of its own is refused for each tensor, the window rows among them."""
    from kch import _lib
    lib = _lib.load()
    x, c = ctypes.c_void_p(4096), 64
    hca = lambda nh, win, ll, lc, lz: lib.kch_hca_attn_bwd(  # noqa: E731
        x, x, x, x, x, ll, x, lc, x, lz, x, None, x, x, x, x, x, None, 1, 64, nh, c, 16, win, 1.0, 0, 0, 0,
        None, 0, None)
    for lds, name in (((c + 4, c, c), b"window"), ((c, c + 4, c), b"C"), ((c, c, 2 * c), b"Z")):
        assert hca(17, 8, *lds) == 2 and name + b" rows must be contiguous" in lib.kch_last_error()
        assert hca(16, 8, *lds) == 1 and b"workspace" in lib.kch_last_error()
    assert hca(17, 0, c + 4, c, c) == 1 and b"workspace" in lib.kch_last_error()  # no window: not read
    csa = lambda nh, norm, la, lb: lib.kch_csa_attn_bwd(  # noqa: E731
        x, x, x, x, x, x, la, x, c, x, c, x, lb, x, x, None, x, x, x, x, x, x, x, None, None, None, 0, None,
        1, 64, nh, c, 4, 8, 8, 1.0, norm, 0, 0, 0, None, 0, None)
    for la, lb in ((c + 4, c), (c, c + 4)):
        for nh, norm in ((17, 1), (4, 0)):
            assert csa(nh, norm, la, lb) == 2 and b"contiguous" in lib.kch_last_error()
        assert csa(16, 1, la, lb) == 1 and b"workspace" in lib.kch_last_error()


def test_csa_backward_workspace_of_long_sequences():
    """Where a query selects few of its blocks, the selection costs the workspace
    one bit a (query, block) and no value: 0.5 GiB at T 131072, m 4 (a dense
    fp32 array would be 16). In tiles, at most three values a slot more."""
    from kch import _lib
    lib = _lib.load()
    ws = lib.kch_csa_attn_bwd_ws_bytes
    for T, topk in ((131072, 512), (32768, 64)):
        assert ws(1, T, 16, 128, 4, 128, topk) - ws(1, T, 16, 128, 4, 128, 0) == T * (T // 4) // 8
    for T, topk in ((4096, 512), (6144, 512)):
        assert ws(1, T, 16, 128, 4, 128, topk) - ws(1, T, 16, 128, 4, 128, 0) <= T * (T // 32 + 3 * topk * 4)
        # ... and none where dsel takes the values, or nobody
        for dsel in (True, False):
            need = _csa_bwd_needs(lib, 1, T, 16, 128, 4, topk, 128, 1, slots=False, dsel=dsel)
            assert need - ws(1, T, 16, 128, 4, 128, 0) == T * (T // 4) // 8
            assert need == lib.kch_csa_attn_bwd_ws_bytes_for(1, T, 16, 128, 4, 128, topk, 1, 0)


@pytest.mark.parametrize("H,HV,K,V,code,chunk", [
    (131071, 131071, 128, 64, 0, True), (131072, 131072, 128, 64, 0, False),   # rows, fp32
    (262143, 262143, 64, 128, 1, True), (262144, 262144, 64, 128, 1, False),   # bf16
    (1, 43577, 128, 128, 1, True), (1, 43578, 128, 128, 1, False),             # partials, HV > H
])
def test_kda_chunk_backward_takes_rows_within_32_bit_offsets(monkeypatch, H, HV, K, V, code, chunk):
    """A chunk's 64 rows of all heads (of the per-value-head partials, HV > H) are
    addressed with 32-bit byte offsets; from 4 GiB on the entry refuses and the
    gradient runs on the recurrence's kernel."""
    import torch
    from kch import _lib, ops_kda
    lib = _lib.load()
    x = ctypes.c_void_p(4096)
    rc = lib.kch_kda_chunk_bwd(*[x] * 14, 1, 1, H, HV, K, V, 1.0, -10.0, code, None, 0, None)
    assert (rc, b"4 GiB" in lib.kch_last_error()) == ((1, False) if chunk else (2, True))
    seen = []
    monkeypatch.setattr(_lib, "call", lambda name, *a: seen.append(name))
    monkeypatch.setattr(_lib, "stream_of", lambda t: None)
    monkeypatch.setattr(torch, "empty", lambda *a, **k: torch.zeros(1))  # the workspace
    dt = torch.float32 if code == 0 else torch.bfloat16
    z = lambda *s: torch.zeros(1, dtype=dt).expand(1, 1, *s)  # noqa: E731
    ops_kda.kda_recurrent_grad(z(H, K), z(H, K), z(HV, V), z(HV, K), z(HV), z(HV, V), chunked=True)
    assert seen == ["kch_kda_chunk_bwd" if chunk else "kch_kda_recurrent_bwd"]


def test_chunk_workspace_size_query():
    """kch_kda_chunk_ws_bytes: 0 where no workspace is used, else the sum of
    the six per-chunk records, each region padded to 256 bytes."""
    from kch import _lib
    lib = _lib.load()
    assert lib.kch_kda_chunk_ws_bytes(2, 100, 2, 2, 128, 128, 0) == 0    # fp32
    assert lib.kch_kda_chunk_ws_bytes(2, 100, 2, 2, 128, 192, 1) == 0    # V outside {64,128}
    assert lib.kch_kda_chunk_ws_bytes(2, 0, 2, 2, 128, 128, 1) == 0
    B, T, HV, K, V = 2, 100, 4, 128, 64
    R = B * HV * ((T + 63) // 64)
    pad = lambda x: (x + 255) // 256 * 256  # noqa: E731
    expect = (3 * pad(R * 64 * K * 2) + pad(R * 64 * 64 * 2) + pad(R * 64 * V * 2)
              + pad(R * K * 4))
    assert lib.kch_kda_chunk_ws_bytes(B, T, 2, HV, K, V, 1) == expect


def test_decode_plan_takes_keys_or_candidates():
    """What the planned CSA step merges past 8192 blocks, by its workspace: all
    logit keys (4 bytes a block) up to 40960 blocks, for a small selection of a
    small batch up to 32768, and only where its estimate of the boundary leaves
    room; else the ranges' top-k candidates (8 bytes each)."""
    from kch import _lib
    ws = _lib.load().kch_decode_ws_bytes
    pad = lambda x: (x + 255) // 256 * 256  # noqa: E731
    for B, nb, topk, keys in ((1, 8193, 64, True), (16, 8200, 2048, True), (1, 32768, 64, True),
                              (1, 32769, 255, False), (7, 40000, 128, False), (8, 40000, 128, True),
                              (1, 40960, 256, True), (16, 40960, 512, True), (16, 40961, 512, False),
                              (16, 32768, 1024, True), (16, 39000, 1024, False), (4, 131073, 512, False)):
        region = ws(B, nb, 16, 128, topk, 128, 1) - ws(B, 1024, 16, 128, topk, 128, 1)
        per = max(1024, 2 * topk)
        r = max(-(-nb // 8192), min(-(-1024 // B), -(-nb // per)))
        rb = (-(-nb // r) + 15) // 16 * 16
        want = pad(B * ((nb + 3) // 4 * 4) * 4) if keys else pad(B * -(-nb // rb) * topk * 8)
        assert region == want, (B, nb, topk, region, want)


def test_hybrid_decoding_default_geometry_is_the_references():
    """``HybridDecoding()`` builds the reference's decode model
    (``run_decoding.py:642-656``)."""
    import kch
    cfg = kch.HybridDecoding().cfg
    expect = dict(d_model=64, n_heads_qk=2, n_heads_v=2, head_dim_k=16, head_dim_v=16,
                  kda_chunk_size=0, csa_m=4, csa_topk=2, csa_nh=2, csa_c=8, csa_dc=8,
                  csa_nIh=1, csa_cI=4, csa_sliding_window=4, hca_m2=4, hca_nh=2, hca_c=8,
                  hca_dc=8, hca_sliding_window=4, n_kda=3, n_csa=1, n_hca=1)
    assert {k: getattr(cfg, k) for k in expect} == expect
