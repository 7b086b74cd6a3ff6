"""The work that programs have this package do, as cases to time and to compare.

Every case is one pass through public entry points of ``kch``: the KDA chunk
operator, CSA and HCA attention (prefill, forward and backward, decode through
their caches) and the 3:1:1 hybrid stack (prefill, decode step). Sizes are
those of ``bench.py`` and of the default ``HybridConfig``; ``draw`` spreads
further cases over the ranges that they stand for.

``exact`` restates each operator in float64 with plain torch. The whole stack
has none: in 16 bits its selections depend on every earlier rounding.
"""

import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.abspath("kda-csa-hca-fusion_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import kch  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_D64 = torch.float64

# d_model, attention heads, head dim, query latent, indexer heads and key dim
# of the benchmark's CSA / HCA configurations
_D, _NH, _C, _DC, _NI, _CI = 2048, 16, 128, 128, 4, 64


def _kda(name, kind, B, T, H, HV, K, V, dtype, decay, state):
    return {"name": name, "kind": kind, "B": B, "T": T, "H": H, "HV": HV, "K": K, "V": V,
            "dtype": dtype, "decay": decay, "state": state}


def _csa(name, kind, B, T, topk, win, dtype):
    return {"name": name, "kind": kind, "B": B, "T": T, "m": 4, "topk": topk, "win": win,
            "dtype": dtype}


def _hca(name, kind, B, T, m2, win, dtype):
    return {"name": name, "kind": kind, "B": B, "T": T, "m2": m2, "win": win, "dtype": dtype}


def listed():
    return [
        # a first call at the default HybridConfig's head shapes (4 heads of 64), fp32,
        # on a short ragged prompt: launches and latency
        _kda("kda_prefill_short", "kda", 2, 77, 4, 4, 64, 64, "fp32", 0.1, False),
        # the benchmark's headline prefill: a batch of prompts, state carried in and out
        _kda("kda_prefill", "kda", 8, 4096, 16, 16, 128, 128, "bf16", 1.0, True),
        # one long document at the layers' decay scale, a length that is no multiple of 64
        _kda("kda_prefill_long", "kda", 1, 20011, 16, 16, 128, 128, "bf16", 0.1, False),
        # training: output, final state and every gradient of a batch of sequences
        _kda("kda_train", "kda_train", 4, 4096, 16, 16, 128, 128, "bf16", 0.1, True),
        # CSA prefill: compression, indexer with top-512, sparse + window attention
        _csa("csa_prefill", "csa", 4, 8192, 512, 128, "bf16"),
        # CSA training with the straight-through indexer, as CSAHybridLayer trains
        _csa("csa_train", "csa_train", 2, 4096, 512, 128, "bf16"),
        # HCA prefill of long documents, projections included
        _hca("hca_prefill", "hca", 4, 32768, 128, 128, "bf16"),
        # HCA training: output and every gradient of the attention block
        _hca("hca_train", "hca_train", 2, 8192, 128, 128, "bf16"),
        # one token of a batch of long conversations through the CSA cache
        _csa("csa_decode", "csa_decode", 16, 131072, 512, 128, "bf16"),
        # one token of a larger batch through the HCA cache
        _hca("hca_decode", "hca_decode", 64, 131072, 128, 128, "bf16"),
        # the 5-layer stack: prefill of prompts, caches populated
        {"name": "stack_prefill", "kind": "stack", "B": 2, "T": 8192, "decode": False},
        # the 5-layer stack: one decode step after a prefill
        {"name": "stack_decode", "kind": "stack", "B": 2, "T": 8192, "decode": True},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    case = _draw(rng)
    case.pop("name", None)
    return case


def _draw(rng):
    kind = rng.choice(["kda", "kda", "kda_train", "csa", "csa_train", "hca", "hca_train",
                       "csa_decode", "hca_decode", "stack"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    if kind in ("kda", "kda_train"):
        H = rng.choice([4, 8, 16])
        HV = H * rng.choice([1, 1, 2])
        K, V = rng.choice([(64, 64), (128, 128), (128, 128)])
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        T = _log_int(rng, 65, 20000 if kind == "kda" else 4096)
        most = (1 << 19 if kind == "kda" else 1 << 18) // (4 if dtype == "fp32" else 1)
        B = _log_int(rng, 1, max(1, min(16, most // (T * HV))))
        return _kda("", kind, B, T, H, HV, K, V, dtype, rng.choice([0.1, 1.0]),
                    rng.random() < 0.5)
    if kind in ("csa", "csa_train"):
        T = 4 * _log_int(rng, 33, 4096 if kind == "csa" else 1024)
        B = _log_int(rng, 1, max(1, min(8, (32768 if kind == "csa" else 8192) // T)))
        return _csa("", kind, B, T, rng.choice([64, 128, 256, 512]), rng.choice([16, 64, 128]),
                    dtype)
    if kind in ("hca", "hca_train"):
        m2 = rng.choice([64, 128])
        T = (_log_int(rng, 200, 32768) if kind == "hca"
             else m2 * _log_int(rng, 2, 8192 // m2))
        B = _log_int(rng, 1, max(1, min(8, (131072 if kind == "hca" else 16384) // T)))
        return _hca("", kind, B, T, m2, rng.choice([16, 64, 128]), dtype)
    if kind in ("csa_decode", "hca_decode"):
        T = _log_int(rng, 515, 131072)
        most = 16 if kind == "csa_decode" else 64
        B = _log_int(rng, 1, max(1, min(most, most * 131072 // T)))
        if kind == "csa_decode":
            return _csa("", kind, B, T, rng.choice([128, 512]), 128, "bf16")
        return _hca("", kind, B, T, 128, 128, "bf16")
    B = rng.choice([1, 2])
    return {"kind": "stack", "B": B, "T": _log_int(rng, 200, 16384 // B),
            "decode": rng.random() < 0.5}


# --------------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


def _kda_inputs(case, seed):
    g, dt = _gen(seed), _DTYPES[case["dtype"]]
    B, T, H, HV, K, V = (case[n] for n in ("B", "T", "H", "HV", "K", "V"))
    q = F.normalize(_randn(g, B, T, H, K), dim=-1).to(dt)
    k = F.normalize(_randn(g, B, T, H, K), dim=-1).to(dt)
    v = _randn(g, B, T, HV, V).to(dt)
    gate = (case["decay"] * F.logsigmoid(_randn(g, B, T, HV, K))).to(dt)
    beta = torch.sigmoid(_randn(g, B, T, HV)).to(dt)
    s0 = 0.02 * _randn(g, B, HV, K, V) if case["state"] else None
    return {"x": [q, k, v, gate, beta], "s0": s0, "do": _randn(g, B, T, HV, V).to(dt),
            "ds": 0.02 * _randn(g, B, HV, K, V)}


def _csa_inputs(case, seed):
    """The projections of one layer input, as views of one fused projection."""
    g, dt = _gen(seed), _DTYPES[case["dtype"]]
    B, T, m = case["B"], case["T"], case["m"]
    fused = _randn(g, B, T, 4 * _C + 2 * _CI + 8).to(dt)
    Ca, Cb, Za, Zb, Ki, Zi, w = fused[..., :4 * _C + 2 * _CI + _NI].split(
        [_C, _C, _C, _C, _CI, _CI, _NI], -1)
    q = _randn(g, B, T, _NH, _C).to(dt)
    qi = _randn(g, B, T, _NI, _CI).to(dt)
    pos = [(0.02 * _randn(g, m, n)).to(dt) for n in (_C, _C, _CI)]
    return {"x": [Ca, Cb, Za, Zb, Ki, Zi, q, qi, w, *pos], "sink": _randn(g, _NH),
            "do": _randn(g, B, T, _NH, _C).to(dt)}


def _hca_inputs(case, seed):
    g, dt = _gen(seed), _DTYPES[case["dtype"]]
    B, T, m2 = case["B"], case["T"], case["m2"]
    pos = (0.02 * _randn(g, m2, _C)).to(dt)
    sink = _randn(g, _NH)
    if case["kind"] == "hca":
        W = [(_randn(g, n, _D) * _D ** -0.5).to(dt) for n in (_C, _C, _DC)]
        W.append((_randn(g, _C * _NH, _DC) * _DC ** -0.5).to(dt))
        return {"H": _randn(g, B, T, _D).to(dt), "W": W, "pos": pos, "sink": sink}
    fused = _randn(g, B, T, 2 * _C).to(dt)
    q = _randn(g, B, T, _NH, _C).to(dt)
    return {"x": [fused[..., :_C], fused[..., _C:], q, pos], "sink": sink,
            "do": _randn(g, B, T, _NH, _C).to(dt)}


def _decode_inputs(case, seed):
    """The projections of the cached tokens and of the next one."""
    g, B, T = _gen(seed), case["B"], case["T"]
    dt = _DTYPES[case["dtype"]]
    csa = case["kind"] == "csa_decode"
    widths = [_C, _C, _C, _C, _CI, _CI] if csa else [_C, _C]
    past = [_randn(g, B, T, w).to(dt) for w in widths]
    new = list(_randn(g, B, 1, sum(widths)).to(dt).split(widths, -1))
    rows = case["m"] if csa else case["m2"]
    pos = [0.02 * _randn(g, rows, w) for w in ([_C, _C, _CI] if csa else [_C])]
    s = {"past": past, "new": new, "pos": pos, "sink": _randn(g, _NH),
         "q": F.normalize(_randn(g, B, 1, _NH, _C), dim=-1)}
    if csa:
        s["qi"], s["w"] = _randn(g, B, 1, _NI, _CI), _randn(g, B, 1, _NI)
    return s


def _stack_config():
    return kch.HybridConfig(
        d_model=_D, n_heads_qk=16, n_heads_v=16, head_dim_k=128, head_dim_v=128,
        kda_chunk_size=64, csa_m=4, csa_topk=512, csa_nh=_NH, csa_c=_C, csa_dc=_DC,
        csa_nIh=_NI, csa_cI=_CI, csa_sliding_window=128, hca_m2=128, hca_nh=_NH, hca_c=_C,
        hca_dc=_DC, hca_sliding_window=128)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("kda", "kda_train"):
        s = _kda_inputs(case, seed)
        if kind == "kda_train":
            s["leaves"] = [t.requires_grad_(True) for t in s["x"] + [s["s0"]] if t is not None]
    elif kind in ("csa", "csa_train"):
        s = _csa_inputs(case, seed)
        if kind == "csa_train":
            s["x"] = [t.detach().requires_grad_(True) for t in s["x"]]
            s["leaves"] = s["x"] + [s["sink"].requires_grad_(True)]
    elif kind in ("hca", "hca_train"):
        s = _hca_inputs(case, seed)
        if kind == "hca_train":
            s["x"] = [t.detach().requires_grad_(True) for t in s["x"]]
            s["leaves"] = s["x"] + [s["sink"].requires_grad_(True)]
    elif kind == "csa_decode":
        s = _decode_inputs(case, seed)
        s["cache"] = kch.CSADecodingCache(case["B"], _C, _CI, case["m"], case["win"], "cuda",
                                          _DTYPES[case["dtype"]])
        s["cache"].append_step(*s.pop("past"), *s["pos"])
    elif kind == "hca_decode":
        s = _decode_inputs(case, seed)
        s["cache"] = kch.HCADecodingCache(case["B"], _C, case["m2"], case["win"], "cuda",
                                          _DTYPES[case["dtype"]])
        s["cache"].append_step(*s.pop("past"), *s["pos"])
    else:
        torch.manual_seed(seed)
        with torch.device("cuda"):
            dec = kch.HybridDecoding(cfg=_stack_config(), total_layers=5)
        dec = dec.to("cuda", torch.bfloat16).eval()
        g = _gen(seed)
        s = {"dec": dec, "x": _randn(g, case["B"], case["T"], _D).to(torch.bfloat16),
             "new": _randn(g, case["B"], 1, _D).to(torch.bfloat16)}
        if case["decode"]:
            dec(s["x"])
    return dict(s, case=case)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "kda":
        return kch.naive_chunk_kda(*s["x"], initial_state=s["s0"], output_final_state=True)
    if kind == "kda_train":
        o, st = kch.naive_chunk_kda(*s["x"], initial_state=s["s0"], output_final_state=True)
        return [o.detach(), st.detach(),
                *torch.autograd.grad([o, st], s["leaves"], [s["do"], s["ds"]])]
    if kind == "csa":
        return kch.csa_core(*s["x"], m=case["m"], topk=case["topk"],
                            sliding_window=case["win"], sink_logits=s["sink"])
    if kind == "csa_train":
        o = kch.csa_core(*s["x"], m=case["m"], topk=case["topk"], sliding_window=case["win"],
                         sink_logits=s["sink"], use_ste=True)
        return [o.detach(), *torch.autograd.grad(o, s["leaves"], s["do"])]
    if kind == "hca":
        W_KV, W_Z, W_DQ, W_UQ = s["W"]
        return kch.naive_hca(s["H"], W_KV, W_Z, s["pos"], W_DQ, W_UQ, m2=case["m2"], nh=_NH,
                             c=_C, dc=_DC, sliding_window=case["win"], sink_logits=s["sink"])
    if kind == "hca_train":
        o = kch.hca_core(*s["x"], m2=case["m2"], sliding_window=case["win"],
                         sink_logits=s["sink"])
        return [o.detach(), *torch.autograd.grad(o, s["leaves"], s["do"])]
    if kind == "csa_decode":
        s["cache"].append_step(*s["new"], *s["pos"])
        o = s["cache"].forward_step(s["q"], s["qi"], s["w"], topk=case["topk"], nh=_NH, nIh=_NI,
                                    sink_logits=s["sink"])
        return [o, s["cache"].sw_buffer.raw()]
    if kind == "hca_decode":
        s["cache"].append_step(*s["new"], *s["pos"])
        o = s["cache"].forward_step(s["q"], nh=_NH, sink_logits=s["sink"])
        return [o, s["cache"].sw_buffer.raw()]
    # the output stream and the KDA states that the call left behind
    if not case["decode"]:
        s["dec"].reset()
    y = s["dec"](s["new"] if case["decode"] else s["x"])
    return [y, s["dec"].model._kda_state]


# --------------------------------------------------------------------------- work

def _kda_work(c, size):
    B, T, H, HV, K, V = (c[n] for n in ("B", "T", "H", "HV", "K", "V"))
    tok = B * T
    # the chunk form's products at 64 tokens a chunk
    flops = tok * HV * (2.0 * (3 * K * V + 64 * (3 * K + 2 * V)) + 64 * 64 / 3.0)
    state = B * HV * K * V * 4
    io = tok * (2 * H * K + HV * (2 * V + K + 1)) * size
    return flops, io + state * (2 if c["state"] else 1), state, tok * (
        2 * (2 * H * K + HV * (K + 1)) + 3 * HV * V) * size


def work(case):
    kind = case["kind"]
    size = 4 if case.get("dtype") == "fp32" else 2
    B, T = case["B"], case["T"]
    if kind in ("kda", "kda_train"):
        flops, byts, state, grads = _kda_work(case, size)
        if kind == "kda":
            return {"bytes": byts, "flops": flops}
        return {"bytes": byts + grads + 2 * state, "flops": 3 * flops}
    if kind in ("csa", "csa_train"):
        m, topk, win = case["m"], case["topk"], case["win"]
        vis = [(t + 1) // m for t in range(T)]
        idx = B * sum(vis) * 2.0 * _NI * _CI
        attn = B * (sum(min(v, topk) for v in vis) + sum(min(win, t + 1) for t in range(T))) \
            * 4.0 * _NH * _C
        io = B * T * (4 * _C + 2 * _CI + _NH * _C + _NI * _CI + _NI) * size
        out = B * T * _NH * _C * size
        if kind == "csa":
            return {"bytes": io + out, "flops": idx + attn}
        return {"bytes": 2 * (io + out), "flops": 3 * idx + 3.5 * attn}
    if kind in ("hca", "hca_train"):
        m2, win = case["m2"], case["win"]
        attn = B * sum((t + 1) // m2 + min(win, t + 1) for t in range(T)) * 4.0 * _NH * _C
        out = B * T * _NH * _C * size
        if kind == "hca":
            proj = 2.0 * B * T * (_D * (2 * _C + _DC) + _DC * _NH * _C)
            return {"bytes": B * T * _D * size + out, "flops": attn + proj}
        io = B * T * (2 * _C + _NH * _C) * size
        return {"bytes": 2 * (io + out), "flops": 3.5 * attn}
    if kind == "csa_decode":
        nb = T // case["m"]
        rows = min(nb, case["topk"]) + case["win"]
        return {"bytes": B * (nb * (_CI * 2 + 4) + rows * _C * 2 + _NH * _C * 8),
                "flops": B * (nb * 2.0 * _NI * _CI + rows * 4.0 * _NH * _C)}
    if kind == "hca_decode":
        rows = T // case["m2"] + case["win"]
        return {"bytes": B * (rows * _C * 2 + _NH * _C * 8), "flops": B * rows * 4.0 * _NH * _C}
    # weights of 3 KDA layers, one CSA and one HCA layer with their output projections
    kda = _D * (3 * 2048 + 16 + 128) + 128 * 2048 + 2048 * _D
    csa = _D * (4 * _C + 2 * _CI + _DC + _NI) + _DC * (_NH * _C + _NI * _CI) + _NH * _C * _D
    hca = _D * (2 * _C + _DC) + _DC * _NH * _C + _NH * _C * _D
    weights = 3 * kda + csa + hca
    state = 3 * B * 16 * 128 * 128 * 4
    if case["decode"]:
        cache = B * (T // 4 * (_CI * 2 + 4) + (512 + T // 128 + 256) * _C * 2)
        return {"bytes": 2 * weights + 2 * state + cache, "flops": 2.0 * B * weights}
    attn = work(_csa("", "csa", B, T // 4 * 4, 512, 128, "bf16"))["flops"] + \
        work(_hca("", "hca_train", B, T // 128 * 128, 128, 128, "bf16"))["flops"] / 3.5
    chunk = 3 * _kda_work(_kda("", "kda", B, T, 16, 16, 128, 128, "bf16", 1.0, False), 2)[0]
    # each sub-layer reads and writes the residual stream once
    return {"bytes": 2 * weights + 5 * 2 * B * T * _D * 2 + state,
            "flops": 2.0 * B * T * weights + attn + chunk}


def tolerance(case):
    # about four times the measured distance from float64
    kind = case["kind"]
    if case.get("dtype") == "fp32":
        # outputs and states up to 6e-7; gradients through two-part products 1e-5
        return {"rel": 3e-6 if kind == "kda" else 5e-5, "max": 1e-3}
    if kind in ("kda", "kda_train"):
        return {"rel": 1.6e-2, "max": 0.2}   # output 4.4e-3, gradients 1.7e-3
    if kind in ("csa", "csa_train", "hca", "hca_train"):
        return {"rel": 1.1e-2, "max": 0.2}   # 2.8e-3
    if kind in ("csa_decode", "hca_decode"):
        return {"rel": 8e-3, "max": 0.1}     # 2.2e-3
    return {"rel": 1.5e-2, "max": 0.2}


# --------------------------------------------------------------------------- float64

def _l2n(x):
    return x / x.norm(dim=-1, keepdim=True).clamp_min(1e-12)


def _blocks(x, m):
    return x.reshape(x.shape[0], x.shape[1] // m, m, x.shape[2])


def _compress64(C, Z, pos, m):
    return (torch.softmax(_blocks(Z, m) + pos, 2) * _blocks(C, m)).sum(2)


def _compress_two64(Ca, Cb, Za, Zb, Ba, Bb, m):
    """Block i mixes Ca of its own tokens with Cb of block i - 1's."""
    za, zb = _blocks(Za, m) + Ba, _blocks(Zb, m) + Bb
    cb = _blocks(Cb, m)
    zb = torch.cat([torch.full_like(zb[:, :1], -math.inf), zb[:, :-1]], 1)
    cb = torch.cat([torch.zeros_like(cb[:, :1]), cb[:, :-1]], 1)
    w = torch.softmax(torch.cat([za, zb], 2), 2)
    return (w * torch.cat([_blocks(Ca, m), cb], 2)).sum(2)


def _attend64(s, rows, sink):
    """Softmax of scores ``s`` [t, nh, n] (-inf: masked) and the sink logit, times
    ``rows`` [t, n, c]."""
    m = torch.maximum(s.detach().amax(-1, keepdim=True), sink.detach()[None, :, None])
    e = torch.exp(s - m)
    p = e / (e.sum(-1, keepdim=True) + torch.exp(sink[None, :, None] - m))
    return torch.matmul(p, rows)


def _window64(local, t, win):
    """The rows of the last ``win`` positions up to each of ``t``, and which exist."""
    at = t[:, None] - win + 1 + torch.arange(win, device=t.device)
    return local[at.clamp(min=0)], at >= 0


def _csa64(x, sink, case, d_out=None):
    """csa_core of one sequence at a time; with ``d_out`` also the gradients,
    the straight-through surrogate of the selection included."""
    leaves = [t.detach().to(_D64).requires_grad_(d_out is not None) for t in [*x, sink]]
    Ca, Cb, Za, Zb, Ki, Zi, q, qi, w, Ba, Bb, Bi, snk = leaves
    m, topk, win = case["m"], case["topk"], case["win"]
    B, T = Ca.shape[:2]
    nb = T // m
    out = torch.empty(q.shape, dtype=_D64, device=q.device)
    grads = [torch.zeros_like(t) for t in leaves]
    n = torch.arange(nb, device=q.device)
    for b in range(B):
        Cn = _l2n(_compress_two64(*(t[b:b + 1] for t in (Ca, Cb, Za, Zb)), Ba, Bb, m))[0]
        Kn = _l2n(_compress64(Ki[b:b + 1], Zi[b:b + 1], Bi, m))[0]
        local = _l2n(Ca[b])
        shared = [Cn, Kn, local]
        cut = [t.detach().requires_grad_(d_out is not None) for t in shared]
        acc = [torch.zeros_like(t) for t in cut]
        for t0 in range(0, T, 512):
            t = torch.arange(t0, min(T, t0 + 512), device=q.device)
            qs, qis, ws = (z[b, t0:t0 + 512].detach().requires_grad_(d_out is not None)
                           for z in (q, qi, w))
            lg = torch.matmul(_l2n(qis), cut[1].t()).relu()
            lg = (lg * ws[..., None]).sum(1)
            seen = (t[:, None] + 1) // m > n
            lg = lg.masked_fill(~seen, -math.inf)
            k = min(topk, nb)
            val, idx = lg.detach().topk(k, dim=-1)
            ok = val > -math.inf
            rows = cut[0][idx]
            if d_out is not None:
                # rows * (1 + soft - soft): the forward value is the hard selection's
                none = ~seen.any(-1, keepdim=True)
                soft = torch.softmax(lg.masked_fill(none, 0.0), -1).gather(-1, idx) * ok
                rows = rows * (1 + soft - soft.detach())[..., None]
            wrows, wok = _window64(cut[2], t, win)
            rows = torch.cat([rows, wrows], 1)
            s = torch.matmul(_l2n(qs), rows.transpose(1, 2))
            s = s.masked_fill(~torch.cat([ok, wok], 1)[:, None], -math.inf)
            o = _attend64(s, rows, snk)
            out[b, t0:t0 + 512] = o.detach()
            if d_out is not None:
                g = torch.autograd.grad(o, [*cut, qs, qis, ws, snk],
                                        d_out[b, t0:t0 + 512].to(_D64))
                for a, v in zip(acc, g):
                    a += v
                for i, v in zip((6, 7, 8), g[3:6]):
                    grads[i][b, t0:t0 + 512] = v
                grads[12] += g[6]
        if d_out is not None:
            at = [0, 1, 2, 3, 4, 5, 9, 10, 11]
            for i, v in zip(at, torch.autograd.grad(shared, [leaves[i] for i in at], acc)):
                grads[i] += v
    return out if d_out is None else [out, *grads]


def _hca64(C, Z, q, pos, sink, case, d_out=None):
    leaves = [t.detach().to(_D64).requires_grad_(d_out is not None)
              for t in (C, Z, q, pos, sink)]
    C, Z, q, pos, snk = leaves
    m2, win = case["m2"], case["win"]
    B, T = C.shape[:2]
    n = torch.arange(T // m2, device=q.device)
    out = torch.empty(q.shape, dtype=_D64, device=q.device)
    grads = [torch.zeros_like(t) for t in leaves]
    for b in range(B):
        shared = [_l2n(_compress64(C[b:b + 1], Z[b:b + 1], pos, m2))[0], _l2n(C[b])]
        cut = [t.detach().requires_grad_(d_out is not None) for t in shared]
        acc = [torch.zeros_like(t) for t in cut]
        for t0 in range(0, T, 1024):
            t = torch.arange(t0, min(T, t0 + 1024), device=q.device)
            qs = q[b, t0:t0 + 1024].detach().requires_grad_(d_out is not None)
            wrows, wok = _window64(cut[1], t, win)
            rows = torch.cat([cut[0][None].expand(len(t), -1, -1), wrows], 1)
            ok = torch.cat([(t[:, None] + 1) // m2 > n, wok], 1)
            s = torch.matmul(_l2n(qs), rows.transpose(1, 2))
            o = _attend64(s.masked_fill(~ok[:, None], -math.inf), rows, snk)
            out[b, t0:t0 + 1024] = o.detach()
            if d_out is not None:
                g = torch.autograd.grad(o, [*cut, qs, snk], d_out[b, t0:t0 + 1024].to(_D64))
                for a, v in zip(acc, g):
                    a += v
                grads[2][b, t0:t0 + 1024] = g[2]
                grads[4] += g[3]
        if d_out is not None:
            for i, v in zip((0, 1, 3), torch.autograd.grad(
                    shared, [leaves[i] for i in (0, 1, 3)], acc)):
                grads[i] += v
    return out if d_out is None else [out, *grads]


def _kda_steps(q, k, v, a, beta, S):
    """The recurrence over the tokens of ``q`` [B, n, H, K] (a: the decay factors)."""
    o = []
    for t in range(q.shape[1]):
        S = S * a[:, t, :, :, None]
        kt = k[:, t, :, None]
        u = beta[:, t, :, None, None] * (v[:, t, :, None] - torch.matmul(kt, S))
        S = S + kt.transpose(-1, -2) * u
        o.append(torch.matmul(q[:, t, :, None], S))
    return torch.cat(o, 2).transpose(1, 2), S


def _kda64(case, s, grads):
    q, k, v, g, beta = (t.detach().to(_D64) for t in s["x"])
    G, K = case["HV"] // case["H"], case["K"]
    B, T, HV, V = v.shape
    scale = K ** -0.5
    S = torch.zeros(B, HV, K, V, dtype=_D64, device=v.device)
    if s["s0"] is not None:
        S = S + s["s0"].detach()
    if not grads:
        qe, ke = q.repeat_interleave(G, 2) * scale, k.repeat_interleave(G, 2)
        o, S = _kda_steps(qe, ke, v, torch.exp(g.clamp_min(-10.0)), beta, S)
        return [o, S]
    x = [q, k, v, g, beta]
    res = [torch.zeros_like(t) for t in x]
    out, starts, n = torch.empty_like(v), [], 64

    def part(x, S):
        q, k, v, g, beta = x
        return _kda_steps(q.repeat_interleave(G, 2) * scale, k.repeat_interleave(G, 2), v,
                          torch.exp(g.clamp_min(-10.0)), beta, S)

    for t0 in range(0, T, n):
        starts.append(S)
        out[:, t0:t0 + n], S = part([t[:, t0:t0 + n] for t in x], S)
    dS = s["ds"].to(_D64)
    for t0 in reversed(range(0, T, n)):
        xs = [t[:, t0:t0 + n].detach().requires_grad_(True) for t in x]
        S0 = starts.pop().requires_grad_(True)
        with torch.enable_grad():
            o, S1 = part(xs, S0)
        got = torch.autograd.grad([o, S1], [*xs, S0], [s["do"][:, t0:t0 + n].to(_D64), dS])
        for r, v_ in zip(res, got):
            r[:, t0:t0 + n] = v_
        dS = got[5]
    return [out, S, *res] + ([dS] if s["s0"] is not None else [])


def _decode64(case, s):
    """One token through a cache that stores compressed rows and window rows in
    its own 16-bit type."""
    csa = case["kind"] == "csa_decode"
    m = case["m"] if csa else case["m2"]
    dt, win = _DTYPES[case["dtype"]], case["win"]
    T = s["past"][0].shape[1] + 1
    nb = T // m
    outs, rings = [], []
    for b in range(case["B"]):
        x = [torch.cat([p[b:b + 1], n[b:b + 1]], 1).to(_D64) for p, n in zip(s["past"], s["new"])]
        full = [t[:, :nb * m] for t in x]
        pos = [p.to(_D64) for p in s["pos"]]
        if csa:
            comp = _compress_two64(*full[:4], *pos[:2], m)[0]
        else:
            comp = _compress64(*full, *pos, m)[0]
        rows = _l2n(comp.to(dt).to(_D64))
        ok = torch.ones(nb, dtype=torch.bool, device=rows.device)
        if csa:
            Kn = _l2n(_compress64(full[4], full[5], pos[2], m)[0].to(dt).to(_D64))
            lg = torch.matmul(_l2n(s["qi"][b, 0].to(_D64)), Kn.t()).relu()
            lg = (lg * s["w"][b, 0].to(_D64)[:, None]).sum(0)
            rows = rows[lg.topk(min(case["topk"], nb))[1]]
            ok = ok[:rows.shape[0]]
        ring = torch.zeros(win, _C, dtype=_D64, device=rows.device)
        at = torch.arange(max(0, T - win), T, device=rows.device)
        ring[at % win] = _l2n(x[0][0, at])
        n = min(win, T)
        rows = torch.cat([rows, ring[:n]])
        qn = s["q"][b].to(_D64)
        o = _attend64(torch.matmul(qn, rows.t()), rows[None], s["sink"].to(_D64))
        outs.append(o)
        rings.append(ring)
    return [torch.stack(outs), torch.stack(rings)]


def exact(case, seed):
    kind = case["kind"]
    if kind == "stack":
        return None
    if kind in ("kda", "kda_train"):
        with torch.no_grad():
            return _kda64(case, _kda_inputs(case, seed), kind == "kda_train")
    if kind in ("csa", "csa_train"):
        s = _csa_inputs(case, seed)
        with torch.set_grad_enabled(kind == "csa_train"):
            return _csa64(s["x"], s["sink"], case, s["do"] if kind == "csa_train" else None)
    if kind == "hca_train":
        s = _hca_inputs(case, seed)
        return _hca64(*s["x"], s["sink"], case, s["do"])
    with torch.no_grad():
        if kind == "hca":
            s = _hca_inputs(case, seed)
            m2, T = case["m2"], case["T"]
            H = F.pad(s["H"], (0, 0, 0, -T % m2))
            W_KV, W_Z, W_DQ, W_UQ = (w.to(_D64) for w in s["W"])
            o = []
            for b in range(case["B"]):
                h = H[b:b + 1].to(_D64)
                q = (h @ W_DQ.t() @ W_UQ.t()).view(1, -1, _NH, _C)
                o.append(_hca64(h @ W_KV.t(), h @ W_Z.t(), q, s["pos"], s["sink"], case))
            return torch.cat(o)[:, :T].reshape(case["B"], T, _NH * _C)
        return _decode64(case, _decode_inputs(case, seed))
