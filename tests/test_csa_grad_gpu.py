"""Gradients of the HIP CSA operators (needs a ROCm GPU).

The reference differentiates ``naive_csa`` with autograd, its top-k selection
held fixed, and adds a straight-through surrogate for the indexer
(``ops_csa.py:1033-1099``; tests ``run_correctness.py:1312-1473``,
``2710-2830``). Checked here:

* ``kch_csa_attn_bwd`` (attention, overlapped compression, window, sink,
  with and without ``normalize_qk``) against ``oracle.csa.csa_attn_grad``
  (pinned by central finite differences on the CPU), including the per-slot
  quantity the surrogate consumes: fp32 within 1e-4 of each tensor's largest
  gradient;
* the whole ``csa_core`` with ``use_ste=True`` against a float64 torch
  statement of the reference's forward with the surrogate identity
  ``kv + (soft_kv - soft_kv.detach())``, differentiated by autograd on the
  CPU on the selection the kernel made: every gradient, indexer inputs
  included, within 1e-4 of its largest entry;
* the reference's contract: ``use_ste`` does not change the forward value, and
  every indexer weight of ``naive_csa`` gets a finite, non-zero gradient;
* ``naive_csa`` in fp32 with ``use_ste=True`` against the reference's own
  gradients (``tests/golden/csa_ste_fp32.npz``, both ``ste_mode`` values,
  with and without ``normalize_qk``): the selection the reference made, and
  every gradient (H, each weight, the sink) within 1e-4 of its largest entry;
* ``full_softmax`` against ``oracle.csa.csa_ste_grad`` (itself pinned by that
  fixture) at a shape with padded channels, and the reference's distinctness
  contract (``run_correctness.py:1588-1731``): the same forward as
  ``topk_columns``, a different and larger indexer gradient.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch
import torch.nn.functional as F

import ste_fixture as SF
from oracle.csa import csa_attn_grad as o_grad
from oracle.csa import csa_ste_grad as o_ste_grad

pytestmark = pytest.mark.gpu


def _check(name, got, ref, tol_max=1e-4):
    got = np.asarray(got, np.float64)
    ref = np.asarray(ref, np.float64)
    assert got.shape == ref.shape, (name, got.shape, ref.shape)
    assert np.isfinite(got).all(), f"{name}: non-finite"
    scale = np.abs(ref).max() + 1e-30
    err = np.abs(got - ref).max()
    assert err <= tol_max * scale, f"{name}: max err {err:.3e} of max {scale:.3e}"


def _selection(rng, B, T, m, topk, hole=None):
    idx = np.full((B, T, topk), -1, np.int32)
    for b in range(B):
        for t in range(T):
            vis = (t + 1) // m
            if vis and t != hole:
                pick = rng.choice(vis, size=min(vis, topk), replace=False)
                idx[b, t, :len(pick)] = pick
    return idx


CASES = [
    # B, T, nh, c, m, topk, win, sink, norm
    (2, 64, 4, 64, 4, 8, 8, True, True),
    (1, 128, 16, 128, 8, 4, 0, False, False),
    (1, 48, 2, 16, 4, 3, 5, True, False),      # c padded to 64
    (1, 64, 18, 128, 4, 6, 4, True, True),     # two head groups
    (2, 1040, 3, 64, 8, 16, 24, True, False),  # several query chunks per key tile
    (1, 64, 37, 64, 4, 4, 8, True, False),     # raw rows: a group of 32 heads, then one of 5
]


@pytest.mark.parametrize("B,T,nh,c,m,topk,win,sink,norm", CASES)
def test_attn_grad_matches_oracle(dev, B, T, nh, c, m, topk, win, sink, norm):
    import kch
    rng = np.random.default_rng(T + nh + c + topk)
    X = {k: rng.standard_normal((B, T, c)) for k in ("Ca", "Cb", "Za", "Zb")}
    q = rng.standard_normal((B, T, nh, c))
    Ba, Bb = rng.standard_normal((m, c)) * 0.3, rng.standard_normal((m, c)) * 0.3
    sk = rng.standard_normal(nh) if sink else None
    W = rng.standard_normal((B, T, nh, c))
    idx = _selection(rng, B, T, m, topk, hole=T // 2)
    ref = o_grad(X["Ca"], X["Cb"], X["Za"], X["Zb"], q, Ba, Bb, idx, W, m=m, sliding_window=win,
                 sink_logits=sk, normalize_qk=norm)
    t = lambda x: torch.tensor(x, dtype=torch.float32, device=dev)  # noqa: E731
    g = kch.ops_csa.csa_attn_grad(t(X["Ca"]), t(X["Cb"]), t(X["Za"]), t(X["Zb"]), t(q), t(Ba),
                                  t(Bb), torch.tensor(idx, device=dev), t(W), m=m,
                                  sliding_window=win, sink_logits=None if sk is None else t(sk),
                                  normalize_qk=norm)
    torch.cuda.synchronize()
    for name in ("Ca", "Cb", "Za", "Zb", "q", "Ba", "Bb", "slot") + (("sink_logits",) if sink else ()):
        _check(name, g[name].cpu().numpy(), ref[name])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,nh,c,m,topk,win,sink,norm", [CASES[0], CASES[2], CASES[3]])
def test_attn_grad_half_storage_is_exact(dev, dtype, B, T, nh, c, m, topk, win, sink, norm):
    """bf16 / fp16 q and d_out move in their own dtype where the queries are
    normalised (read and written by the MFMA kernels; fp32 copies otherwise):
    the same bits as the fp32-storage path on the same values, dq rounded to
    nearest even."""
    import kch
    rng = np.random.default_rng(T + nh + c + topk + 7)
    X = {k: rng.standard_normal((B, T, c)) for k in ("Ca", "Cb", "Za", "Zb")}
    q = rng.standard_normal((B, T, nh, c))
    Ba, Bb = rng.standard_normal((m, c)) * 0.3, rng.standard_normal((m, c)) * 0.3
    sk = rng.standard_normal(nh) if sink else None
    W = rng.standard_normal((B, T, nh, c))
    idx = torch.tensor(_selection(rng, B, T, m, topk, hole=T // 2), device=dev)
    t = lambda x: torch.tensor(x, dtype=torch.float32, device=dev)  # noqa: E731
    qh, Wh = t(q).to(dtype), t(W).to(dtype)
    args = [t(X[k]) for k in ("Ca", "Cb", "Za", "Zb")]
    kw = dict(m=m, sliding_window=win, sink_logits=None if sk is None else t(sk),
              normalize_qk=norm, want_gsum=True)
    got = kch.ops_csa.csa_attn_grad(*args, qh, t(Ba), t(Bb), idx, Wh, **kw)
    ref = kch.ops_csa.csa_attn_grad(*args, qh.float(), t(Ba), t(Bb), idx, Wh.float(), **kw)
    torch.cuda.synchronize()
    assert got["q"].dtype == dtype
    assert torch.equal(got["q"], ref["q"].to(dtype)), "dq"
    for name in ref:
        if name != "q":
            assert torch.equal(got[name], ref[name]), name


def _torch_reference(X, idx, *, m, topk, win, sink, norm):
    """The reference's CSA forward (compression ``ops_csa.py:237-305``,
    indexer ``:330-573``, the STE gather ``:1033-1099``, attention with window
    and sink ``:1100-1155``) in float64 torch on the CPU, the selection given."""
    Ca, Cb, Za, Zb, Kx, Zx, q, qi, wi, Ba, Bb, Bi = (X[k] for k in (
        "Ca", "Cb", "Za", "Zb", "K_idx", "Z_idx", "q", "q_idx", "w_idx", "Ba", "Bb", "B_idx"))
    B_, T, c = Ca.shape
    nb = T // m
    nh = q.shape[2]

    def blocks(x):
        return x.reshape(B_, nb, m, x.shape[-1])

    zb_prev = torch.cat([torch.full_like(blocks(Zb)[:, :1], float('-inf')), blocks(Zb)[:, :-1]], 1)
    cb_prev = torch.cat([torch.zeros_like(blocks(Cb)[:, :1]), blocks(Cb)[:, :-1]], 1)
    wts = torch.softmax(torch.cat([blocks(Za) + Ba, zb_prev + Bb], dim=2), dim=2)
    Ccomp = (wts * torch.cat([blocks(Ca), cb_prev], dim=2)).sum(2)
    Kcomp = (torch.softmax(blocks(Zx) + Bi, dim=2) * blocks(Kx)).sum(2)
    cI = Kx.shape[-1]
    qn, Cn = (F.normalize(q, dim=-1), F.normalize(Ccomp, dim=-1)) if norm else (q, Ccomp)
    qin, Kn = (F.normalize(qi, dim=-1), F.normalize(Kcomp, dim=-1)) if norm else (qi, Kcomp)
    scale = 1.0 if norm else c ** -0.5
    iscale = 1.0 if norm else cI ** -0.5
    logits = torch.einsum('bhtn,bth->btn', torch.relu(torch.einsum('bthd,bnd->bhtn', qin, Kn) * iscale), wi)
    tt, nn = torch.arange(T), torch.arange(nb)
    logits = logits.masked_fill(~((tt[:, None] + 1) // m > nn[None, :]), float('-inf'))
    allm = logits.isinf().all(-1, keepdim=True)
    soft = torch.softmax(logits.masked_fill(allm, 0.0), -1).masked_fill(allm, 0.0)
    idx = torch.as_tensor(idx, dtype=torch.long)
    valid = idx >= 0
    isafe = idx.clamp(min=0)
    kv = Cn[torch.arange(B_)[:, None, None], isafe]                             # [B,T,k,c]
    ssel = torch.gather(soft, -1, isafe) * valid.to(soft.dtype)
    soft_kv = ssel.unsqueeze(-1) * kv.detach()
    kv = kv + (soft_kv - soft_kv.detach())
    s = torch.einsum('bthd,btkd->bthk', qn, kv) * scale
    s = s.masked_fill(~valid[:, :, None, :], float('-inf'))
    vals = [kv]
    scores = [s]
    if win:
        Cl = F.normalize(Ca, dim=-1) if norm else Ca
        pad = torch.cat([torch.zeros(B_, win - 1, c, dtype=Ca.dtype), Cl], 1)
        wi_ = torch.arange(T)[:, None] + torch.arange(win)[None, :]
        Cw = pad[:, wi_]                                                          # [B,T,w,c]
        wv = torch.arange(win)[None, :] >= (win - 1 - torch.arange(T)[:, None])
        sw = (torch.einsum('bthd,btwd->bthw', qn, Cw) * scale).masked_fill(~wv[None, :, None, :],
                                                                            float('-inf'))
        vals.append(Cw)
        scores.append(sw)
    cat = torch.cat(scores, -1)
    catv = ~torch.isinf(cat)
    rm = torch.clamp(cat.masked_fill(~catv, float('-inf')).amax(-1, keepdim=True), min=0.0)
    e = torch.exp(cat - rm).masked_fill(~catv, 0.0)
    den = e.sum(-1, keepdim=True)
    if sink is not None:
        den = den + torch.exp(sink.view(1, 1, nh, 1) - rm)
    p = torch.where(den > 0, e / den.clamp_min(1e-300), torch.zeros_like(e))
    out = torch.einsum('bthk,btkd->bthd', p[..., :topk], vals[0])
    if win:
        out = out + torch.einsum('bthw,btwd->bthd', p[..., topk:], vals[1])
    return out


@pytest.mark.parametrize("norm", [False, True])
def test_csa_core_ste_grads_match_torch_reference(dev, norm):
    import kch
    rng = np.random.default_rng(21 + norm)
    B, T, nh, c, m, topk, win, cI, nIh = 1, 64, 2, 64, 4, 4, 6, 32, 2
    shapes = dict(Ca=(B, T, c), Cb=(B, T, c), Za=(B, T, c), Zb=(B, T, c), K_idx=(B, T, cI),
                  Z_idx=(B, T, cI), q=(B, T, nh, c), q_idx=(B, T, nIh, cI), w_idx=(B, T, nIh),
                  Ba=(m, c), Bb=(m, c), B_idx=(m, cI))
    X = {k: rng.standard_normal(s) * (0.3 if k.startswith("B") else 1.0) for k, s in shapes.items()}
    sk = rng.standard_normal(nh)
    W = rng.standard_normal((B, T, nh, c))
    xt = {k: torch.tensor(v, dtype=torch.float32, device=dev, requires_grad=True) for k, v in X.items()}
    st = torch.tensor(sk, dtype=torch.float32, device=dev, requires_grad=True)
    args = [xt[k] for k in ("Ca", "Cb", "Za", "Zb", "K_idx", "Z_idx", "q", "q_idx", "w_idx", "Ba",
                            "Bb", "B_idx")]
    out, idx = kch.csa_core(*args, m=m, topk=topk, sliding_window=win, sink_logits=st,
                            normalize_qk=norm, return_indices=True, use_ste=True)
    (out.double() * torch.tensor(W, device=dev)).sum().backward()
    torch.cuda.synchronize()
    # the same loss through the float64 torch statement, on the kernel's selection
    xr = {k: torch.tensor(v, dtype=torch.float64, requires_grad=True) for k, v in X.items()}
    sr = torch.tensor(sk, dtype=torch.float64, requires_grad=True)
    ref_out = _torch_reference(xr, idx.cpu().numpy(), m=m, topk=topk, win=win, sink=sr, norm=norm)
    # the forward holds its compressed rows in bf16 (2^-9 relative); without
    # normalisation the scores reach |q||k| / sqrt(c) ~ 8, so the outputs move
    # by a few 1e-3 of their largest value
    _check("out", out.detach().cpu().numpy(), ref_out.detach().numpy(), 1e-2)
    (ref_out * torch.tensor(W)).sum().backward()
    for k in X:
        _check(k, xt[k].grad.cpu().numpy(), xr[k].grad.numpy())
    _check("sink", st.grad.cpu().numpy(), sr.grad.numpy())


def test_naive_csa_ste_contract(dev):
    """``run_correctness.py:1312-1473``: ``use_ste`` leaves the forward value
    unchanged, and every indexer weight gets a finite, non-zero gradient."""
    import kch
    torch.manual_seed(42)
    B, T, d = 1, 32, 16
    m, topk, nh, nIh, c, cI, dc = 4, 2, 2, 2, 8, 4, 8
    H = torch.randn(B, T, d, device=dev)
    P = dict(W_aKV=(c, d), W_bKV=(c, d), W_aZ=(c, d), W_bZ=(c, d), Ba=(m, c), Bb=(m, c),
             W_DQ=(dc, d), W_UQ=(c * nh, dc), W_IUQ=(cI * nIh, dc), W_w=(nIh, d),
             W_KV_idx=(cI, d), W_Z_idx=(cI, d), B_idx=(m, cI))
    base = {k: torch.randn(*s) * (0.02 if k.startswith("B") else 0.1) for k, s in P.items()}
    outs = []
    for ste in (False, True):
        ps = {k: v.clone().to(dev).requires_grad_(True) for k, v in base.items()}
        o = kch.naive_csa(H, *[ps[k] for k in P], m=m, topk=topk, nh=nh, nIh=nIh, c=c, c_I=cI,
                          dc=dc, use_ste=ste)
        o.square().sum().backward()
        outs.append((o.detach(), ps))
    assert torch.allclose(outs[0][0], outs[1][0], rtol=0, atol=1e-6)
    for k in ("W_IUQ", "W_w", "W_KV_idx", "W_Z_idx", "B_idx"):
        g = outs[1][1][k].grad
        assert g is not None and torch.isfinite(g).all() and g.abs().sum() > 0, k
        g0 = outs[0][1][k].grad
        assert g0 is None or g0.abs().sum() == 0, k
    for k in ("W_aKV", "W_bKV", "W_aZ", "W_bZ", "W_DQ", "W_UQ", "Ba", "Bb"):
        g = outs[1][1][k].grad
        assert g is not None and torch.isfinite(g).all() and g.abs().sum() > 0, k


@pytest.mark.parametrize("topk,win", [(6, 0), (0, 5)])
def test_attn_grad_sparse_edges(dev, topk, win):
    """A selection wider than the visible blocks (mostly -1 slots), and no
    selection at all (window only)."""
    import kch
    rng = np.random.default_rng(31 + topk)
    B, T, nh, c, m = 1, 16, 2, 64, 4
    X = {k: rng.standard_normal((B, T, c)) for k in ("Ca", "Cb", "Za", "Zb")}
    q = rng.standard_normal((B, T, nh, c))
    Ba, Bb = rng.standard_normal((m, c)) * 0.3, rng.standard_normal((m, c)) * 0.3
    sk = rng.standard_normal(nh)
    W = rng.standard_normal((B, T, nh, c))
    idx = _selection(rng, B, T, m, topk) if topk else np.zeros((B, T, 0), np.int32)
    ref = o_grad(X["Ca"], X["Cb"], X["Za"], X["Zb"], q, Ba, Bb, idx, W, m=m, sliding_window=win,
                 sink_logits=sk, normalize_qk=True)
    t = lambda x: torch.tensor(x, dtype=torch.float32, device=dev)  # noqa: E731
    g = kch.ops_csa.csa_attn_grad(t(X["Ca"]), t(X["Cb"]), t(X["Za"]), t(X["Zb"]), t(q), t(Ba),
                                  t(Bb), torch.tensor(idx, device=dev) if topk else None, t(W),
                                  m=m, sliding_window=win, sink_logits=t(sk), normalize_qk=True)
    torch.cuda.synchronize()
    for name in ("Ca", "Cb", "Za", "Zb", "q", "Ba", "Bb", "sink_logits"):
        _check(name, g[name].cpu().numpy(), ref[name])


@pytest.mark.parametrize("T,m,nh", [(16, 4, 2), (15, 1, 18)])  # rows of whole float4s or not; two head groups
def test_attn_grad_dense_values_without_selection(dev, T, m, nh):
    """With no selection the dense slot values are zeros, whatever their memory held."""
    import kch
    torch.manual_seed(T)
    B, c = 2, 64
    x = [torch.randn(B, T, c, device=dev) for _ in range(4)]
    q, W = (torch.randn(B, T, nh, c, device=dev) for _ in range(2))
    pos = [torch.randn(m, c, device=dev) for _ in range(2)]
    empty, held = torch.empty, []

    def poisoned(*a, **k):
        t = empty(*a, **k)
        if t.shape == (B, T, T // m):
            held.append(t.fill_(float("nan")))
        return t

    torch.empty = poisoned
    try:
        g = kch.ops_csa.csa_attn_grad(*x, q, *pos, None, W, m=m, sliding_window=5, _dense=True)
    finally:
        torch.empty = empty
    assert held and g["dsel"] is held[0] and not bool(g["dsel"].ne(0).any())


@pytest.mark.parametrize("nIh,cI,norm", [(4, 64, True), (4, 64, False), (2, 32, True),
                                         (1, 128, False), (8, 64, True), (3, 48, False)])
def test_ste_kernel_matches_dense_statement(dev, nIh, cI, norm):
    """``kch_csa_ste_bwd`` against the dense torch statement of the same
    surrogate (softmax over every causal block, autograd through the logits
    and the key compression), on a selection with -1 slots; fp32, 1e-4 of each
    tensor's largest gradient. Covers padded heads (3 -> 4) and channels
    (32 -> 64, 48 -> 64)."""
    from kch.ops_csa import _ste_indexer_grads, _ste_indexer_grads_dense
    rng = np.random.default_rng(nIh * cI + norm)
    B, T, m, topk = 2, 256, 4, 16
    t = lambda x: torch.tensor(x, dtype=torch.float32, device=dev)  # noqa: E731
    K = t(rng.standard_normal((B, T, cI)))
    Z = t(rng.standard_normal((B, T, cI)))
    q = t(rng.standard_normal((B, T, nIh, cI)))
    w = t(rng.standard_normal((B, T, nIh)))
    Bi = t(rng.standard_normal((m, cI)) * 0.3)
    idx = torch.tensor(_selection(rng, B, T, m, topk, hole=100), device=dev)
    slot = t(rng.standard_normal((B, T, topk))) * (idx >= 0)
    got = _ste_indexer_grads(K, Z, q, w, Bi, idx, slot, m=m, normalize_qk=norm)
    ref = _ste_indexer_grads_dense(K, Z, q, w, Bi, idx, slot, m=m, normalize_qk=norm)
    torch.cuda.synchronize()
    for name, a, r in zip(("K_idx", "Z_idx", "q_idx", "w_idx", "B_idx"), got, ref):
        _check(name, a.cpu().numpy(), r.cpu().numpy())


@pytest.mark.parametrize("norm,mode", SF.CASES)
def test_naive_csa_ste_grads_match_reference_fixture(dev, norm, mode):
    import kch
    z, meta, W = SF.load()
    t = SF.tag(norm, mode)
    Wt = {k: torch.tensor(v, device=dev, requires_grad=True) for k, v in W.items()}
    H = torch.tensor(z["H"], device=dev, requires_grad=True)
    sk = torch.tensor(z["sink"], device=dev, requires_grad=True)
    with kch.record_selections() as sel:
        out = kch.naive_csa(H, *[Wt[n] for n in SF.NAMES], m=meta["m"], topk=meta["topk"],
                            nh=meta["nh"], nIh=meta["nIh"], c=meta["c"], c_I=meta["cI"],
                            dc=meta["dc"], sliding_window=meta["win"], sink_logits=sk,
                            use_ste=True, ste_mode=mode, normalize_qk=norm)
    (out * torch.tensor(z["G"], device=dev)).sum().backward()
    torch.cuda.synchronize()
    got_idx = sel[0].cpu().numpy().astype(np.int64)
    ref_idx = z[f"{t}.idx"]
    assert got_idx.shape == ref_idx.shape
    for r, (a, b) in enumerate(zip(got_idx.reshape(-1, got_idx.shape[-1]),
                                   ref_idx.reshape(-1, ref_idx.shape[-1]))):
        assert set(a.tolist()) == set(b.tolist()), f"row {r}: {a} vs the reference's {b}"
    _check("out", out.detach().cpu().numpy(), z[f"{t}.out"], 1e-2)
    got = {f"d{n}": Wt[n].grad.cpu().numpy() for n in SF.NAMES}
    got["dH"] = H.grad.cpu().numpy()
    got["dsink"] = sk.grad.cpu().numpy()
    err = SF.worst_rel(got, z, t)
    bad = {k: v for k, v in err.items() if v > 1e-4}
    assert not bad, bad


@pytest.mark.parametrize("norm", [True, False])
def test_csa_core_full_softmax_matches_oracle(dev, norm):
    import kch
    rng = np.random.default_rng(61 + norm)
    B, T, nh, c, m, topk, win, cI, nIh = 2, 64, 3, 40, 4, 5, 6, 24, 3
    shapes = dict(Ca=(B, T, c), Cb=(B, T, c), Za=(B, T, c), Zb=(B, T, c), K_idx=(B, T, cI),
                  Z_idx=(B, T, cI), q=(B, T, nh, c), q_idx=(B, T, nIh, cI), w_idx=(B, T, nIh),
                  Ba=(m, c), Bb=(m, c), B_idx=(m, cI))
    X = {k: rng.standard_normal(s) * (0.3 if k.startswith("B") else 1.0) for k, s in shapes.items()}
    sk = rng.standard_normal(nh)
    Gw = rng.standard_normal((B, T, nh, c))
    names = ("Ca", "Cb", "Za", "Zb", "K_idx", "Z_idx", "q", "q_idx", "w_idx", "Ba", "Bb", "B_idx")
    grads, outs = {}, {}
    for mode in ("topk_columns", "full_softmax"):
        xt = {k: torch.tensor(v, dtype=torch.float32, device=dev, requires_grad=True)
              for k, v in X.items()}
        st = torch.tensor(sk, dtype=torch.float32, device=dev, requires_grad=True)
        out, idx = kch.csa_core(*[xt[k] for k in names], m=m, topk=topk, sliding_window=win,
                                sink_logits=st, normalize_qk=norm, return_indices=True,
                                use_ste=True, ste_mode=mode)
        (out.double() * torch.tensor(Gw, device=dev)).sum().backward()
        torch.cuda.synchronize()
        grads[mode] = {k: xt[k].grad.cpu().numpy() for k in X}
        grads[mode]["sink_logits"] = st.grad.cpu().numpy()
        outs[mode] = out.detach().cpu().numpy()
        if mode == "full_softmax":
            ref = o_ste_grad(*[X[k] for k in names], idx.cpu().numpy(), Gw, m=m,
                             sliding_window=win, sink_logits=sk, normalize_qk=norm,
                             ste_mode=mode)
            for k in list(X) + ["sink_logits"]:
                _check(k, grads[mode][k], ref[k])
    # run_correctness.py:1588-1731: same forward, distinct and larger indexer gradient
    np.testing.assert_array_equal(outs["topk_columns"], outs["full_softmax"])
    for k in ("K_idx", "q_idx", "w_idx"):
        a, b = grads["topk_columns"][k], grads["full_softmax"][k]
        assert np.abs(a - b).max() > 1e-6 * np.abs(b).max(), k
    assert np.abs(grads["full_softmax"]["K_idx"]).sum() > np.abs(grads["topk_columns"]["K_idx"]).sum()


def test_naive_csa_aux_contrastive_raises(dev):
    import kch
    B, T, d, c, nh, dc, nIh, cI, m = 1, 8, 16, 8, 2, 8, 2, 4, 4
    H = torch.randn(B, T, d, device=dev)
    P = dict(W_aKV=(c, d), W_bKV=(c, d), W_aZ=(c, d), W_bZ=(c, d), Ba=(m, c), Bb=(m, c),
             W_DQ=(dc, d), W_UQ=(c * nh, dc), W_IUQ=(cI * nIh, dc), W_w=(nIh, d),
             W_KV_idx=(cI, d), W_Z_idx=(cI, d), B_idx=(m, cI))
    ps = [torch.randn(*s, device=dev) for s in P.values()]
    with pytest.raises(NotImplementedError):
        kch.naive_csa(H, *ps, m=m, topk=2, nh=nh, nIh=nIh, c=c, c_I=cI, dc=dc,
                      ste_mode='aux_contrastive')


STE_EDGES = [
    # B, T, m, topk, nIh, cI, norm: heads per tile, channels, blocks off whole tiles
    (1, 1, 1, 1, 1, 64, True),         # one query, one block
    (2, 63, 3, 5, 2, 64, False),       # 21 blocks (no 4-element rows), raw queries and keys
    (1, 129, 1, 16, 4, 64, True),      # a 129-block row: two key tiles, one block in the last
    (2, 132, 4, 8, 8, 64, True),       # eight heads: two queries a tile
    (1, 260, 4, 64, 1, 128, True),     # 16 queries a tile, 65 blocks
    (1, 576, 2, 24, 4, 128, False),    # several query chunks per key tile
    (3, 100, 4, 3, 2, 48, True),       # channels padded to 64
]


@pytest.mark.parametrize("B,T,m,topk,nIh,cI,norm", STE_EDGES)
def test_ste_indexer_kernels_at_tile_edges(dev, B, T, m, topk, nIh, cI, norm):
    """``kch_csa_ste_scatter`` + ``kch_csa_ste_bwd`` against float64 autograd of the
    same surrogate: every gradient within 1e-4 of its largest entry (fp32 sums of
    up to T * nIh <= 2304 terms: at most 2304 * 2^-24 = 1.4e-4 of the terms'
    absolute sum, and random signs leave its square root)."""
    import kch
    rng = np.random.default_rng(B * T + nIh + cI)
    nb = T // m
    r = lambda *s: torch.tensor(rng.standard_normal(s))  # noqa: E731
    K, Z, q, w, Bp = r(B, T, cI), r(B, T, cI), r(B, T, nIh, cI), r(B, T, nIh), 0.3 * r(m, cI)
    idx = torch.tensor(_selection(rng, B, T, m, topk, hole=T // 2))
    slot = r(B, T, topk)
    leaves = [x.clone().requires_grad_(True) for x in (K, Z, q, w, Bp)]
    Kl, Zl, ql, wl, Bl = leaves
    kn = (torch.softmax(Zl.view(B, nb, m, cI) + Bl, 2) * Kl.view(B, nb, m, cI)).sum(2)
    qn = ql
    if norm:
        kn, qn = F.normalize(kn, dim=-1), F.normalize(ql, dim=-1)
    a = torch.einsum('bthd,bnd->bthn', qn, kn) * (1.0 if norm else cI ** -0.5)
    lg = (torch.relu(a) * wl[..., None]).sum(2)
    seen = (torch.arange(T)[:, None] + 1) // m > torch.arange(nb)
    none = ~seen.any(-1, keepdim=True)
    soft = torch.softmax(lg.masked_fill(~seen, -np.inf).masked_fill(none, 0.0), -1)
    sel = soft.gather(-1, idx.long().clamp(min=0))
    ref = torch.autograd.grad((sel * slot * (idx >= 0)).sum(), leaves)
    f = lambda x: x.to(dev, torch.float32)  # noqa: E731
    got = kch.ops_csa._ste_indexer_grads(f(K), f(Z), f(q), f(w), f(Bp), idx.to(dev), f(slot),
                                         m=m, normalize_qk=norm)
    torch.cuda.synchronize()
    for name, g, x in zip(("K_idx", "Z_idx", "q_idx", "w_idx", "B_idx"), got, ref):
        _check(name, g.cpu().numpy(), x.numpy())


TILE_EDGES = [
    # B, T, nh, c, m, topk, win, dtype: blocks in tiles (nb <= 3 topk) or gathered
    (2, 9, 16, 128, 1, 3, 5, torch.bfloat16),      # 9 queries: a workgroup of one; in tiles
    (1, 132, 5, 64, 2, 66, 37, torch.bfloat16),    # 66 blocks: a second group of 64 keys, 3-row step
    (1, 301, 16, 128, 7, 20, 128, torch.float16),  # 43 blocks, window of whole steps
    (2, 264, 18, 128, 4, 23, 33, torch.float32),   # 66 blocks in tiles, two head groups
    (1, 264, 16, 128, 4, 21, 33, torch.bfloat16),  # 66 blocks > 3 topk: gathered
    (1, 260, 17, 64, 4, 6, 40, torch.float32),     # gathered, two head groups
]


@pytest.mark.parametrize("B,T,nh,c,m,topk,win,dtype", TILE_EDGES)
def test_attn_grad_at_tile_edges(dev, B, T, nh, c, m, topk, win, dtype):
    """The tiled and the gathering query pass and both key passes at remainders of
    their tiles, against the fp64 oracle on the same (dtype-representable) q and
    d_out: within 1e-4 of each tensor's largest entry (two-part products, 2^-16);
    dq one rounding of dtype more. ``_dense`` gives the slots' values at their
    blocks."""
    import kch
    rng = np.random.default_rng(T + nh + topk)
    t = lambda x: torch.tensor(x, dtype=torch.float32, device=dev)  # noqa: E731
    X = {k: rng.standard_normal((B, T, c)).astype(np.float32) for k in ("Ca", "Cb", "Za", "Zb")}
    q, W = (t(rng.standard_normal((B, T, nh, c))).to(dtype) for _ in range(2))
    Ba, Bb = ((rng.standard_normal((m, c)) * 0.3).astype(np.float32) for _ in range(2))
    sk = rng.standard_normal(nh).astype(np.float32)
    idx = _selection(rng, B, T, m, topk, hole=T // 2)
    ref = o_grad(X["Ca"], X["Cb"], X["Za"], X["Zb"], q.float().cpu().numpy(), Ba, Bb, idx,
                 W.float().cpu().numpy(), m=m, sliding_window=win, sink_logits=sk, normalize_qk=True)
    args = [t(X[k]) for k in ("Ca", "Cb", "Za", "Zb")] + [q, t(Ba), t(Bb)]
    kw = dict(m=m, sliding_window=win, sink_logits=t(sk))
    ix = torch.tensor(idx, device=dev)
    g = kch.ops_csa.csa_attn_grad(*args, ix, W, **kw)
    dsel = kch.ops_csa.csa_attn_grad(*args, ix, W, _dense=True, **kw)["dsel"].cpu().numpy()
    torch.cuda.synchronize()
    ulp = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    for name in ("Ca", "Cb", "Za", "Zb", "q", "Ba", "Bb", "slot", "sink_logits"):
        _check(name, g[name].float().cpu().numpy(), ref[name], 1e-4 + (ulp if name == "q" else 0.0))
    want = np.zeros((B, T, T // m))
    np.put_along_axis(want, np.maximum(idx, 0), 0.0, -1)
    for b, i, j in zip(*np.nonzero(idx >= 0)):
        want[b, i, idx[b, i, j]] = ref["slot"][b, i, j]
    _check("dsel", dsel, want)


def test_grads_move_inputs_to_the_first_ones_device(dev):
    """The compression's other inputs, their biases and the indexer's weights may
    lie on the host: they are copied to the first input's device, and the
    gradients are those of device inputs, bit for bit."""
    import kch
    from kch.ops_csa import _bwd_rows, _ste_indexer_grads
    torch.manual_seed(3)
    B, T, nh, c, m, topk, nIh = 1, 24, 2, 64, 4, 3, 2
    assert [x.device.type for x in _bwd_rows("meta", torch.float32, c, torch.zeros(B, T, c))[::2]] == ["meta"]
    X = [torch.randn(B, T, c) for _ in range(4)]
    q, W = torch.randn(B, T, nh, c), torch.randn(B, T, nh, c)
    pos = [torch.randn(m, c) for _ in range(2)]
    idx = torch.tensor(_selection(np.random.default_rng(3), B, T, m, topk))
    on = lambda xs: [x.to(dev) for x in xs]  # noqa: E731
    ref = kch.ops_csa.csa_attn_grad(*on(X), q.to(dev), *on(pos), idx.to(dev), W.to(dev), m=m)
    got = kch.ops_csa.csa_attn_grad(X[0].to(dev), *X[1:], q, *pos, idx, W, m=m)
    for k in ref:
        assert got[k].is_cuda and torch.equal(got[k], ref[k]), k
    K, Z, Bi = X[0], X[1], pos[0]
    qi, w, slot = torch.randn(B, T, nIh, c), torch.randn(B, T, nIh), ref["slot"]
    a = _ste_indexer_grads(*on((K, Z, qi, w, Bi)), idx.to(dev), slot, m=m, normalize_qk=True)
    b = _ste_indexer_grads(K.to(dev), Z, qi.to(dev), w, Bi, idx.to(dev), slot, m=m, normalize_qk=True)
    for x, y in zip(a, b):
        assert y.is_cuda and torch.equal(x, y)


@pytest.mark.parametrize("norm,m,topk", [(True, 4, 4), (True, 1, 4), (False, 4, 4)])  # in tiles, gathered, raw
def test_core_backward_without_surrogate_computes_no_slots(dev, monkeypatch, norm, m, topk):
    """``use_ste=False``: nothing reads the slots' values, so the kernel is given
    no place for them; the gradients are those of a call that takes them."""
    from kch import _lib
    import kch
    torch.manual_seed(topk + m)
    B, T, nh, c, cI, nIh = 1, 48, 3, 64, 32, 2
    x = [torch.randn(B, T, w, device=dev, requires_grad=True) for w in (c, c, c, c, cI, cI)]
    q = torch.randn(B, T, nh, c, device=dev, requires_grad=True)
    qi, w = torch.randn(B, T, nIh, cI, device=dev), torch.randn(B, T, nIh, device=dev)
    pos = [torch.randn(m, n, device=dev) for n in (c, c, cI)]
    kw = dict(m=m, topk=topk, sliding_window=5, normalize_qk=norm)
    out, idx = kch.csa_core(*x, q, qi, w, *pos, return_indices=True, use_ste=False, **kw)
    W = torch.randn_like(out)
    seen, call = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (seen.append((name, a)), call(name, *a))[1])
    got = torch.autograd.grad(out, [*x[:4], q], W)
    args, = [a for name, a in seen if name == "kch_csa_attn_bwd"]
    assert args[24] is None and args[25] is None  # slot_grad, dsel
    ref = kch.ops_csa.csa_attn_grad(*x[:4], q, *pos[:2], idx, W, m=m, sliding_window=5,
                                    normalize_qk=norm)
    for g, name in zip(got, ("Ca", "Cb", "Za", "Zb", "q")):
        assert torch.equal(g, ref[name]), name


@pytest.mark.parametrize("norm,cI,nIh", [(True, 64, 1), (False, 64, 1), (False, 128, 1), (False, 64, 4)])
def test_ste_kernels_gate_a_score_alike(dev, norm, cI, nIh):
    """A score that is 0 but for its rounding (the second half of the channels
    repeats the first's products, shuffled, with the other sign) opens the ReLU
    gate of the query's gradient and of the key's, or of neither: per sequence,
    query 1 sees block 0 with such scores and block 1 with negative ones, so its
    gradient and block 0's are zero together, head for head of one."""
    from kch.ops_csa import _ste_indexer_grads
    g = torch.Generator().manual_seed(cI + nIh)
    B, h = 2048, cI // 2
    perm = torch.randperm(h, generator=g)
    u, v = (torch.randn(B, h, generator=g) for _ in range(2))
    q = torch.cat([u, u[:, perm]], 1)
    K = torch.stack([torch.cat([v, -v[:, perm]], 1), -q], 1)
    qi = torch.zeros(B, 2, nIh, cI)
    qi[:, 1, 0] = q
    w = torch.zeros(B, 2, nIh)
    w[..., 0] = 1.0
    idx = torch.tensor([[0, -1], [0, 1]], dtype=torch.int32).expand(B, 2, 2).contiguous()
    slot = torch.tensor([[0.0, 0.0], [1.0, 0.0]]).expand(B, 2, 2).contiguous()
    dK, _, dq, _, _ = _ste_indexer_grads(*(x.to(dev) for x in (K, torch.zeros_like(K), qi, w, torch.zeros(1, cI),
                                                               idx, slot)), m=1, normalize_qk=norm)
    in_q, in_k = dq[:, 1, 0].ne(0).any(-1), dK[:, 0].ne(0).any(-1)
    assert 0 < int(in_q.sum()) < B and torch.equal(in_q, in_k)


@pytest.mark.parametrize("zero", ["queries", "keys", "both"])
def test_ste_zero_rows(dev, zero):
    """Zero rows (a padded sequence): finite gradients against the dense statement,
    and no time of their own (each of their pairs was once summed again, five
    times the time of random rows)."""
    from kch.ops_csa import _ste_indexer_grads, _ste_indexer_grads_dense
    torch.manual_seed(7)

    def inputs(B, T, m, topk, nIh, cI):
        r = lambda *s: torch.randn(*s, device=dev)  # noqa: E731
        K, Z, q, w, Bi = r(B, T, cI), r(B, T, cI), r(B, T, nIh, cI), r(B, T, nIh), 0.1 * r(m, cI)
        score = torch.rand(B, T, T // m, device=dev)
        t, n = torch.arange(T, device=dev), torch.arange(T // m, device=dev)
        val, idx = score.masked_fill((t[:, None] + 1) // m <= n, -1.0).topk(topk, -1)
        return [K, Z, q, w, Bi, torch.where(val >= 0, idx, -1).int(), r(B, T, topk) * (val >= 0)]

    def pad(x):
        K, q = x[0].clone(), x[2].clone()
        if zero != "queries":
            K[:, :K.shape[1] // 2] = 0
        if zero != "keys":
            q[:, q.shape[1] // 2:] = 0
        return [K, x[1], q, *x[3:]]

    x = pad(inputs(2, 128, 4, 8, 2, 64))
    got = _ste_indexer_grads(*x, m=4, normalize_qk=True)
    ref = _ste_indexer_grads_dense(*x, m=4, normalize_qk=True)
    for i, name in ((1, "Z_idx"), (3, "w_idx"), (4, "B_idx")):
        _check(name, got[i].cpu().numpy(), ref[i].cpu().numpy())
    # (a zero row's own gradient is 1e12 times what reaches it: its scale)
    for i, name in ((0, "K_idx"), (2, "q_idx")):
        live = x[i].ne(0).any(-1)
        if zero != "queries" and i == 0:
            live[:, :64] = False
        _check(name, got[i][live].cpu().numpy(), ref[i][live].cpu().numpy())
        assert torch.isfinite(got[i]).all()

    def time(x):
        best = float("inf")
        for _ in range(6):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(3):
                _ste_indexer_grads(*x, m=4, normalize_qk=True)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    x = inputs(2, 4096, 4, 64, 4, 64)
    plain, padded = time(x), time(pad(x))
    assert padded < 1.8 * plain, (plain, padded)


@pytest.mark.parametrize("kind,norm", [("csa", True), ("csa", False), ("hca", True)])
def test_empty_batch_gives_zero_bias_and_sink_gradients(dev, monkeypatch, kind, norm):
    """The gradients that sum over the batch (position biases, sink) of a batch of
    no sequences are zeros, whatever the memory that they are given held."""
    import kch
    c, cI, nh, nIh, m, T = 64, 32, 2, 2, 4, 16
    r = lambda *s: torch.randn(*s, device=dev, requires_grad=True)  # noqa: E731
    sk = r(nh)
    if kind == "csa":
        pos = [r(m, n) for n in (c, c, cI)]
        o = kch.csa_core(*[r(0, T, n) for n in (c, c, c, c, cI, cI)], r(0, T, nh, c), r(0, T, nIh, cI),
                         r(0, T, nIh), *pos, m=m, topk=3, sliding_window=4, sink_logits=sk, use_ste=True,
                         normalize_qk=norm)
    else:
        pos = [r(m, c)]
        o = kch.hca_core(r(0, T, c), r(0, T, c), r(0, T, nh, c), *pos, m2=m, sliding_window=4, sink_logits=sk)
    W, empty = torch.empty_like(o), torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: (lambda t: t.fill_(float("nan"))
                                                         if t.is_floating_point() else t)(empty(*a, **k)))
    for g in torch.autograd.grad(o, [*pos, sk], W):
        assert not bool(g.ne(0).any())
