"""Performance cases of the public APIs: `sigmoid_attention`,
`sigmoid_attention_padded` and `sigmoid_attention_varlen`.

A case is a dict of plain values:
  kind       "dense" | "padded" | "varlen" | "decode"
  B, T, H, D batch, (longest) sequence, heads, head dim
  Tq         queries per sequence (decode only; T is then the key cache)
  dtype      "float16" | "bfloat16" | "float32"
  causal     top-left causal mask
  train      True: forward and backward, returns O, dQ, dK, dV; False: forward
             without a graph, returns O
  score_mod  True: a per-key additive term
  lo         shortest sequence of a ragged batch (0: every sequence is T)
  lens       seed of the ragged batch's lengths (a case's work is fixed, so
             its lengths are; the values of the tensors follow `seed`)
"""

import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "triton-sigmoid_amd"))
import triton_sigmoid as ts  # noqa: E402

_DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
_BASE = dict(kind="dense", B=1, T=128, Tq=0, H=8, D=64, dtype="bfloat16", causal=False, train=True,
             score_mod=False, lo=0, lens=0)


def _case(name, **kw):
    c = dict(_BASE, **kw)
    c["name"] = name
    return c


def listed():
    return [
        # One short prompt scored by a small model: host time and launches.
        _case("infer-short", B=1, T=128, H=8, D=64, dtype="float16", causal=True, train=False),
        # The fp32 plumbing configuration (B=2 L=256 H=4 D=64), a training step.
        _case("train-fp32-small", B=2, T=256, H=4, D=64, dtype="float32"),
        # The small dense training configuration (fp16 B=2 L=1024 H=8 D=64).
        _case("train-small", B=2, T=1024, H=8, D=64, dtype="float16"),
        # The headline training configuration (bf16 B=4 L=4096 H=16 D=128 causal).
        _case("train-headline", B=4, T=4096, H=16, D=128, causal=True),
        # The right-padded causal training configuration (fp16 B=8 Lmax=2048 H=8
        # D=64, lengths 512..2048).
        _case("train-padded", kind="padded", B=8, T=2048, H=8, D=64, dtype="float16", causal=True, lo=512, lens=1),
        # The padded long-context training configuration (bf16 B=4 Lmax=8192 H=12
        # D=64, lengths 1024..8192).
        _case("train-padded-long", kind="padded", B=4, T=8192, H=12, D=64, lo=1024, lens=2),
        # A point of the benchmark grid (B=16384/L, H=2048/D) at D=64: a training
        # step of a bidirectional encoder.
        _case("train-encoder", B=8, T=2048, H=32, D=64),
        # Encoding one long document: the grid's longest point, forward only.
        _case("infer-long", B=1, T=16384, H=16, D=128, train=False),
        # Packed sequences of odd lengths with a per-key term, as a training loop
        # that packs documents has them.
        _case("train-packed", kind="varlen", B=9, T=3001, H=12, D=128, causal=True, score_mod=True, lo=67, lens=3),
        # Decoding: one new query against ragged key caches.
        _case("decode", kind="decode", B=16, T=8192, Tq=1, H=32, D=128, train=False, lo=1024, lens=4),
        # Speculative decoding: a few queries per sequence, D=64, full caches.
        _case("decode-few", kind="decode", B=32, T=4096, Tq=4, H=32, D=64, train=False),
        # fp32 training at an odd length.
        _case("train-fp32", B=2, T=1999, H=8, D=64, dtype="float32", causal=True),
    ]


def _lens(c):
    """Valid lengths of the case's sequences (the longest is T)."""
    if not c["lo"]:
        return [c["T"]] * c["B"]
    r = random.Random(c["lens"])
    n = [r.randint(c["lo"], c["T"]) for _ in range(c["B"])]
    n[r.randrange(c["B"])] = c["T"]
    return n


def _pairs(c):
    """Visible (query, key) pairs of one head, over the batch."""
    if c["kind"] == "decode":
        return sum(c["Tq"] * n for n in _lens(c))
    return sum(n * (n + 1) // 2 if c["causal"] else n * n for n in _lens(c))


def _flops(c):
    return (14 if c["train"] else 4) * c["D"] * c["H"] * _pairs(c)


def _log_int(r, lo, hi):
    return int(round(math.exp(r.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: dense and ragged training and
    inference from 128 to 16384 rows, and decoding from 512 to 65536 cached
    keys; every dtype and head dim; odd sizes."""
    # The largest listed case is 2.2e12 operations; fp32 runs at about a tenth
    # of the 16-bit rate.
    while True:
        kind = rng.choice(("dense", "dense", "padded", "padded", "varlen", "decode"))
        c = dict(_BASE, kind=kind)
        c["D"] = rng.choice((64, 64, 128, 128, 32, 16)) if kind != "decode" else rng.choice((64, 128, 128))
        c["H"] = rng.choice((4, 8, 12, 16, 32))
        c["score_mod"] = rng.random() < 0.25
        if kind == "decode":
            c.update(train=False, Tq=rng.choice((1, 1, 2, 4, 8, 16, 32)), T=_log_int(rng, 512, 65536),
                     B=_log_int(rng, 1, 32), dtype=rng.choice(("bfloat16", "float16")))
            if rng.random() < 0.6:
                c.update(lo=max(1, c["T"] // rng.choice((2, 4, 8))), lens=rng.randrange(1 << 20))
            if c["B"] * c["T"] * c["H"] * c["D"] > 16 * 8192 * 32 * 128:
                continue
            return c
        c["dtype"] = rng.choice(("bfloat16", "bfloat16", "float16", "float32"))
        c["T"] = _log_int(rng, 128, 16384)
        if rng.random() < 0.3:
            c["T"] = max(128, c["T"] // 128 * 128)
        c["B"] = _log_int(rng, 1, 16)
        c["causal"] = rng.random() < 0.5
        c["train"] = rng.random() < 0.7
        if kind != "dense":
            c["B"] = max(2, c["B"])
            c.update(lo=max(1, c["T"] // rng.choice((2, 4, 8, 16))), lens=rng.randrange(1 << 20))
        most = 6e10 if c["dtype"] == "float32" else 1e12
        if _flops(c) > most or c["B"] * c["T"] * c["H"] * c["D"] > 4 * 4096 * 16 * 128:
            continue
        return c


def _inputs(c, seed):
    """Tensors of the case, on the GPU, and its lengths."""
    dev, dt = torch.device("cuda"), _DTYPES[c["dtype"]]
    g = torch.Generator(device=dev).manual_seed(1000003 * (seed % (1 << 40)) + 17)

    def normal(*shape, dtype=dt):
        return torch.randn(shape, generator=g, device=dev, dtype=torch.float32).to(dtype)

    lens = _lens(c)
    B, T, H, D = c["B"], c["T"], c["H"], c["D"]
    if c["kind"] == "varlen":
        n = sum(lens)
        qs = ks = (n, H, D)
        ms = (n,)
    elif c["kind"] == "decode":
        qs, ks, ms = (B, c["Tq"], H, D), (B, T, H, D), (B, T)
    else:
        qs = ks = (B, T, H, D)
        ms = (B, T)
    s = {"q": normal(*qs), "k": normal(*ks), "v": normal(*ks), "do": None, "score_mod": None}
    if c["train"]:
        s["do"] = normal(*qs)
    if c["score_mod"]:
        s["score_mod"] = normal(*ms, dtype=torch.float32)
    return s, lens


def prepare(case, seed):
    s, lens = _inputs(case, seed)
    dev = s["q"].device
    s["case"] = case
    if case["train"]:
        for x in ("q", "k", "v"):
            s[x].requires_grad_(True)
    if case["kind"] in ("padded", "decode"):
        s["lens_k"] = torch.tensor(lens, dtype=torch.int32, device=dev)
        s["lens_q"] = s["lens_k"] if case["kind"] == "padded" else None
    elif case["kind"] == "varlen":
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        s["cu"] = torch.tensor(cu, dtype=torch.int32, device=dev)
        s["longest"] = max(lens)
    return s


def _attention(s):
    c = s["case"]
    q, k, v, mod = s["q"], s["k"], s["v"], s["score_mod"]
    if c["kind"] == "dense":
        return ts.sigmoid_attention(q, k, v, is_causal=c["causal"], score_mod=mod)
    if c["kind"] == "varlen":
        return ts.sigmoid_attention_varlen(q, k, v, s["cu"], s["cu"], s["longest"], s["longest"],
                                           is_causal=c["causal"], score_mod=mod)
    return ts.sigmoid_attention_padded(q, k, v, seq_lens_k=s["lens_k"], seq_lens_q=s["lens_q"],
                                       is_causal=c["causal"], score_mod=mod)


def run(state):
    if not state["case"]["train"]:
        with torch.no_grad():
            return _attention(state)
    o = _attention(state)
    dq, dk, dv = torch.autograd.grad(o, (state["q"], state["k"], state["v"]), state["do"])
    return {"o": o, "dq": dq, "dk": dk, "dv": dv}


def work(case):
    """Bytes: Q, K, V (and dO) read and O (and dQ, dK, dV) written once, valid
    rows only where rows are read; flops: 4·D per visible pair forward and
    10·D backward."""
    c = case
    size = 4 if c["dtype"] == "float32" else 2
    row = c["H"] * c["D"] * size
    lens = _lens(c)
    valid = sum(lens)
    rows_out = valid if c["kind"] == "varlen" else c["B"] * c["T"]
    if c["kind"] == "decode":
        qrows = c["B"] * c["Tq"]
        nbytes = row * (2 * valid + 2 * qrows)
    elif c["train"]:
        nbytes = row * (4 * valid + 4 * rows_out)
    else:
        nbytes = row * (3 * valid + rows_out)
    if c["score_mod"]:
        nbytes += 4 * valid
    return {"bytes": nbytes, "flops": _flops(c)}


def tolerance(case):
    # About four times the 2-norm error against 64 bits that the gradients show.
    return {"float16": {"rel": 2e-3, "max": 5e-2},
            "bfloat16": {"rel": 1.2e-2, "max": 3e-1},
            "float32": {"rel": 5e-6, "max": 2e-4}}[case["dtype"]]


def _exact_rows(q, k, v, do, mod, bias, scale, causal):
    """O (and dQ, dK, dV) of one sequence and head in 64 bits, [rows, D] each,
    by blocks of queries."""
    nq, nk = q.shape[0], k.shape[0]
    kt, vt = k.t().contiguous(), v.t().contiguous()
    o, dq = torch.empty_like(q), torch.empty_like(q)
    dk, dv = torch.zeros_like(k), torch.zeros_like(v)
    add = bias if mod is None else bias + mod.double()
    step = max(64, (1 << 25) // max(nk, 1))
    for i in range(0, nq, step):
        j = min(nq, i + step)
        p = torch.sigmoid(q[i:j] @ kt * scale + add)
        if causal:
            p = torch.tril(p, diagonal=i)
        o[i:j] = p @ v
        if do is not None:
            ds = (do[i:j] @ vt) * p * (1.0 - p)
            dq[i:j] = ds @ k * scale
            dk += ds.t().contiguous() @ q[i:j]
            dv += p.t().contiguous() @ do[i:j]
    return o, dq, dk * scale, dv


def exact(case, seed):
    c = case
    if 14 * c["D"] * c["H"] * c["B"] * max(c["Tq"] or c["T"], 64) * c["T"] > 4e13:
        return None
    s, lens = _inputs(c, seed)
    q, k, v, do, mod = s["q"], s["k"], s["v"], s["do"], s["score_mod"]
    out = {n: torch.zeros(t.shape, dtype=torch.float64, device=t.device)
           for n, t in (("o", q), ("dq", q), ("dk", k), ("dv", v))}
    scale, first = 1.0 / math.sqrt(c["D"]), 0
    for b, n in enumerate(lens):
        bias = -math.log(n)
        if c["kind"] == "varlen":
            at = kat = slice(first, first + n)
            first += n
        else:
            at = (b, slice(0, c["Tq"] if c["kind"] == "decode" else n))
            kat = (b, slice(0, n))
        for h in range(c["H"]):
            one = [None if t is None else t[w][:, h].double().contiguous()
                   for t, w in ((q, at), (k, kat), (v, kat), (do, at))]
            got = _exact_rows(*one, None if mod is None else mod[kat], bias, scale, c["causal"])
            for name, w, x in zip(("o", "dq", "dk", "dv"), (at, at, kat, kat), got):
                out[name][w][:, h] = x
    return out if c["train"] else out["o"]
