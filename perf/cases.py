"""Workloads on which the framework's speed is measured.

Each case is a plain dict; ``prepare`` makes what a program holds before the
call, ``run`` is one pass through the public entry points (the ``@attention``
decorator, autograd, the prepared decode launch), ``work`` the bytes and
operations such a pass cannot do without, ``exact`` its outputs in 64 bits in
plain torch, and ``tolerance`` how far a correct implementation at the same
precision may lie from another.

Fields of a case: ``kind`` ("decode", "prefill", "cross", "train" or
"sparse_train"), ``dtype``, ``B``, ``Hq``, ``Hkv``, ``N`` (keys; queries too
unless ``Nq`` is given), ``D``, ``mask`` ("full", "causal" or "window" with
``window``), ``rope`` (RoPE base, 0 for none), ``alibi``, ``layout`` ("bhnd",
or "bnhd": the strided views that projections of (B, N, H, D) give), and for
decode ``prepared`` (a fixed-shape serving loop's launcher instead of the
decorated call).
"""
from __future__ import annotations

import math

import torch

import attentionfuse_amd as af
from attentionfuse_amd.rope_utils import build_rope_cache
from attentionfuse_amd.runtime.block_mask import block_mask_from_blocks
from attentionfuse_amd.runtime.dispatch import alibi_slope_values
from attentionfuse_amd.runtime.prepared import prepare_decode

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, kind, dtype, B, Hq, Hkv, N, D, **more):
    c = dict(kind=kind, dtype=dtype, B=B, Hq=Hq, Hkv=Hkv, N=N, D=D, Nq=N, mask="full", window=0,
             rope=0, alibi=False, layout="bhnd", prepared=False)
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # One sequence's token step in a serving loop at a short cache
        # (Llama-3-8B geometry): the smallest call, launches and latency.
        _case("decode_one", "decode", "bf16", 1, 32, 8, 1024, 128, Nq=1, prepared=True),
        # The same model's token step for a batch of eight at a full 32k
        # cache: streaming K and V from HBM.
        _case("decode_32k", "decode", "bf16", 8, 32, 8, 32768, 128, Nq=1),
        # Token step of a batch of a GPT-2-small-sized model with ALiBi, one
        # key/value head per query head, cache of an odd length.
        _case("decode_mha_alibi", "decode", "fp16", 16, 12, 12, 3001, 64, Nq=1, alibi=True),
        # A chat prompt of a few hundred tokens, GQA, in the (B, N, H, D)
        # layout that a transformers model hands over.
        _case("prompt_300", "prefill", "bf16", 1, 32, 8, 300, 128, mask="causal", layout="bnhd"),
        # GPT-2-small causal attention in fp32 (B=1, H=12, N=512, D=64).
        _case("gpt2_fp32", "prefill", "fp32", 1, 12, 12, 512, 64, mask="causal"),
        # Causal + RoPE + ALiBi prefill at 4096 tokens, the benchmark's
        # forward workload.
        _case("prefill_rope_alibi", "prefill", "fp16", 4, 12, 12, 4096, 64, mask="causal", rope=10000, alibi=True),
        # A long prompt of ragged length, GQA, transformers layout.
        _case("prompt_6001", "prefill", "bf16", 1, 32, 8, 6001, 128, mask="causal", layout="bnhd"),
        # Cross-attention of a few decoder rows over a long encoder output.
        _case("cross_100x1500", "cross", "fp16", 2, 12, 12, 1500, 64, Nq=100),
        # Local attention over a long document (two-sided window).
        _case("window_8192", "prefill", "fp16", 1, 12, 12, 8192, 64, mask="window", window=512),
        # Training step of a small causal model at an odd length.
        _case("train_1000", "train", "fp16", 2, 12, 12, 1000, 64, mask="causal"),
        # BigBird block-sparse training step (global row and column, band of
        # one block, three random blocks per row).
        _case("bigbird_train", "sparse_train", "fp16", 4, 12, 12, 4096, 64),
        # Llama-3-8B-geometry causal GQA training step with fused RoPE.
        _case("train_gqa", "train", "bf16", 1, 32, 8, 4096, 128, mask="causal", rope=500000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges, no larger than the largest."""
    heads = [(12, 12, 64), (16, 16, 64), (32, 8, 128), (16, 4, 128), (8, 1, 64), (16, 16, 128)]
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "cross", "train", "sparse_train"])
    Hq, Hkv, D = rng.choice(heads)
    dtype = rng.choice(["fp16", "bf16"])
    if kind == "decode":
        B, N = _log_int(rng, 1, 32), _log_int(rng, 256, 32768)
        while B * Hkv * N * D > 8 * 8 * 32768 * 128:
            N = max(256, N // 2)
        if rng.random() < 0.1 and B * Hkv * N * D <= 1 << 26:
            dtype = "fp32"
        return _case(None, kind, dtype, B, Hq, Hkv, N, D, Nq=1, alibi=rng.random() < 0.25,
                     prepared=rng.random() < 0.5)
    if kind == "cross":
        return _case(None, kind, dtype, _log_int(rng, 1, 8), Hq, Hkv, _log_int(rng, 64, 4096), D,
                     Nq=_log_int(rng, 2, 2048))
    if kind == "sparse_train":
        return _case(None, kind, dtype, rng.randint(1, 4), 12, 12, 64 * _log_int(rng, 8, 64), 64)
    layout = rng.choice(["bhnd", "bnhd"])
    mask = rng.choice(["causal", "causal", "causal", "window", "full"])
    rope = rng.choice([0, 0, 10000, 500000])
    alibi = mask == "causal" and rng.random() < 0.2
    B, N = _log_int(rng, 1, 8), _log_int(rng, 64, 8192)
    most = 2.2e11 if kind == "prefill" else 1.0e11    # 4 B H D N^2 of the forward, before masking
    if kind == "prefill" and rng.random() < 0.15:
        dtype, most = "fp32", 2.0e10
    while 4.0 * B * Hq * D * N * N > most:
        if B > 1:
            B -= 1
        else:
            N = (3 * N) // 4
    window = max(16, _log_int(rng, 32, 1024)) if mask == "window" else 0
    return _case(None, kind, dtype, B, Hq, Hkv, N, D, mask=mask, window=window, rope=rope, alibi=alibi,
                 layout=layout)


def _grid(case):
    """BigBird tile grid (64 x 64 blocks), the same for every seed."""
    n = (case["N"] + 63) // 64
    g = torch.Generator().manual_seed(7)
    a = torch.zeros(n, n, dtype=torch.bool)
    a[0], a[:, 0] = True, True
    i = torch.arange(n)
    for d in (-1, 0, 1):
        j = i + d
        ok = (j >= 0) & (j < n)
        a[i[ok], j[ok]] = True
    for r in range(n):
        a[r, torch.randperm(n, generator=g)[:3]] = True
    return a


def _program(case):
    """The decorated attention function of a case."""
    H = case["Hq"]

    @af.attention
    def fn(Q, K, V):
        s = af.rope(Q, K) if case["rope"] else af.scaled_dot_product(Q, K)
        if case["alibi"]:
            s = af.alibi(s, H)
        if case["kind"] == "sparse_train":
            s = af.block_sparse(s)
        elif case["mask"] == "causal":
            s = af.causal(s)
        elif case["mask"] == "window":
            s = af.sliding_window(s, case["window"])
        return af.softmax(s) @ V
    return fn


def _inputs(case, seed):
    dev, dt = torch.device("cuda:0"), DTYPES[case["dtype"]]
    g = torch.Generator(device=dev).manual_seed(seed)

    def make(H, N):
        if case["layout"] == "bnhd":
            return torch.randn(case["B"], N, H, case["D"], generator=g, device=dev, dtype=dt).transpose(1, 2)
        return torch.randn(case["B"], H, N, case["D"], generator=g, device=dev, dtype=dt)
    q = make(case["Hq"], case["Nq"])
    k, v = make(case["Hkv"], case["N"]), make(case["Hkv"], case["N"])
    do = make(case["Hq"], case["Nq"]) if "train" in case["kind"] else None
    return q, k, v, do


def _tables(case):
    if not case["rope"]:
        return {}
    cos, sin = build_rope_cache(case["N"], case["D"], base=float(case["rope"]), device=torch.device("cuda:0"),
                                dtype=DTYPES[case["dtype"]])
    return {"cos": cos, "sin": sin}


def prepare(case, seed):
    q, k, v, do = _inputs(case, seed)
    fn, kw = _program(case), _tables(case)
    s = dict(kind=case["kind"], fn=fn, kw=kw, qkv=(q, k, v), do=do)
    if case["kind"] == "sparse_train":
        kw["block_mask"] = block_mask_from_blocks(_grid(case), 64, 64, device=q.device)
    if do is not None:
        for t in (q, k, v):
            t.requires_grad_(True)
    if case["prepared"]:
        s["launch"], s["out"] = prepare_decode(fn(q, k, v, return_graph=True), q, k, v)
    elif case["layout"] == "bnhd" and do is None:
        # the model's own (B, N, H, D) buffer, written through a strided view
        s["kw"]["out"] = torch.empty_like(q)
    return s


def run(state):
    if "launch" in state:
        state["launch"]()
        return state["out"]
    q, k, v = state["qkv"]
    out = state["fn"](q, k, v, **state["kw"])
    if state["do"] is None:
        return out
    return (out.detach(),) + torch.autograd.grad(out, (q, k, v), state["do"])


def _pairs(case):
    """Visible (query, key) pairs of one head."""
    N, W = case["N"], case["window"]
    if case["kind"] == "sparse_train":
        n = torch.full(((N + 63) // 64,), 64)
        n[-1] = N - 64 * (len(n) - 1)
        return int((_grid(case).long() * n[:, None] * n[None, :]).sum())
    if case["mask"] == "causal":
        return N * (N + 1) // 2
    if case["mask"] == "window" and W < N:
        return N * N - (N - W) * (N - W + 1)
    return case["Nq"] * N


def work(case):
    """QK^T and PV are 4 D operations a visible pair, a backward 10 D more;
    every input is read and every output written once."""
    train = "train" in case["kind"]
    size = 4 if case["dtype"] == "fp32" else 2
    rows_q, rows_k = case["B"] * case["Hq"] * case["Nq"], case["B"] * case["Hkv"] * case["N"]
    # forward: q, k, v, o; backward: dO, dQ, dK, dV besides
    words = (rows_q * (4 if train else 2) + rows_k * (4 if train else 2)) * case["D"]
    words += 2 * case["N"] * case["D"] if case["rope"] else 0
    flops = (14 if train else 4) * case["D"] * case["B"] * case["Hq"] * _pairs(case)
    return {"bytes": size * words, "flops": flops}


def tolerance(case):
    # About four times the error against exact() measured over the listed and
    # drawn cases: fp16 up to 3.1e-4 (outputs and gradients alike), bf16
    # 2.5e-3; fp32 2.9e-7 at 512 keys, with room for sums of thousands.
    return {"rel": {"fp16": 1.2e-3, "bf16": 1.0e-2, "fp32": 5e-6}[case["dtype"]]}


def _rotate(x, cos, sin):
    """Rotate-half RoPE."""
    h = x.shape[-1] // 2
    half = torch.cat([-x[..., h:], x[..., :h]], dim=-1)
    return x * cos + half * sin


def _rotate_back(g, cos, sin):
    """The transposed rotation, applied to a gradient."""
    h = g.shape[-1] // 2
    y = g * sin
    return g * cos - torch.cat([-y[..., h:], y[..., :h]], dim=-1)


def exact(case, seed):
    q, k, v, do = _inputs(case, seed)
    dt = DTYPES[case["dtype"]]
    tab = {n: t[0, 0].double() for n, t in _tables(case).items()}
    B, Hq, Hkv, N, Nq, D = (case[x] for x in ("B", "Hq", "Hkv", "N", "Nq", "D"))
    G, scale = Hq // Hkv, 1.0 / math.sqrt(D)
    i = torch.arange(Nq, device=q.device)[:, None]
    j = torch.arange(N, device=q.device)[None, :]
    # a single query stands at the end of its cache
    dist = ((i if case["kind"] != "decode" else N - 1) - j).abs().double()
    hide = None
    if case["kind"] == "sparse_train":
        hide = ~_grid(case).to(q.device).repeat_interleave(64, 0).repeat_interleave(64, 1)[:N, :N]
    elif case["mask"] == "causal":
        hide = j > i
    elif case["mask"] == "window":
        hide = (i - j).abs() >= case["window"]
    slopes = torch.tensor(alibi_slope_values(Hq), dtype=dt).double().tolist()
    out = torch.empty(B, Hq, Nq, D, dtype=torch.float64, device=q.device)
    grads = [torch.zeros(t.shape, dtype=torch.float64, device=q.device) for t in (q, k, v)] if do is not None else []
    for b in range(B):
        for hq in range(Hq):
            hk = hq // G
            qd, kd, vd = q[b, hq].double(), k[b, hk].double(), v[b, hk].double()
            if case["rope"]:
                # q~ and k~ are values of the input type by definition
                qd, kd = (_rotate(t, tab["cos"], tab["sin"]).to(dt).double() for t in (qd, kd))
            s = (qd @ kd.t()) * scale
            if case["alibi"]:
                s -= slopes[hq] * dist
            if hide is not None:
                s.masked_fill_(hide, -math.inf)
            p = torch.softmax(s, dim=-1)
            o = p @ vd
            out[b, hq] = o
            if do is None:
                continue
            dod = do[b, hq].double()
            grads[2][b, hk] += p.t() @ dod
            ds = (dod @ vd.t()).sub_((dod * o).sum(-1, keepdim=True)).mul_(p).mul_(scale)
            dq, dk = ds @ kd, ds.t() @ qd
            if case["rope"]:
                dq, dk = (_rotate_back(g, tab["cos"], tab["sin"]) for g in (dq, dk))
            grads[0][b, hq] += dq
            grads[1][b, hk] += dk
    return out if do is None else (out, *grads)
