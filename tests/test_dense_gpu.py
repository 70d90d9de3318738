"""GPU parity tests for the dense path (sigmoid_attention -> myops::sigmoid_attention_fwd/bwd
-> libsigattn.so).  Mirrors the reference's tests/test_sigmoid_dense.py."""

import ctypes
import math

import numpy as np
import pytest
import torch

import triton_sigmoid as ts
from conftest import get_tolerance
from helpers import (assert_close_to_oracle, assert_reference_criterion, criterion_errors,
                     oracle_fwd_bwd, randn)
from oracle.eager import sigmoid_attention_eager
from triton_sigmoid import _capi

pytestmark = pytest.mark.gpu
DEV = "cuda"
DTYPES = [torch.float16, torch.bfloat16, torch.float32]


def _inputs(B, T, H, D, dtype, seed=0, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return [randn((B, T, H, D), dtype, DEV, g, std) for _ in range(4)]


# --- tight parity against the float64 oracle (odd sizes, every head dim) -------

@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("T", [1, 17, 130, 300])
@pytest.mark.parametrize("causal", [False, True])
def test_dense_matches_oracle(dtype, D, T, causal):
    B, H = 2, 3
    q, k, v, do = _inputs(B, T, H, D, dtype, seed=T * 7 + D)
    for t in (q, k, v):
        t.requires_grad_(True)
    o = ts.sigmoid_attention(q, k, v, is_causal=causal)
    o.backward(do)
    scale = 1.0 / math.sqrt(D)
    bias = np.full(B, -math.log(T), dtype=np.float32).astype(np.float64)
    want_o, (dq, dk, dv) = oracle_fwd_bwd(q, k, v, do, scale=np.float32(scale), bias=bias, causal=causal)
    assert_close_to_oracle(o, want_o, dtype, "O")
    assert_close_to_oracle(q.grad, dq, dtype, "dQ")
    assert_close_to_oracle(k.grad, dk, dtype, "dK")
    assert_close_to_oracle(v.grad, dv, dtype, "dV")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T", [33, 64, 65, 96])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("with_mod", [False, True])
def test_fp32_few_key_tiles_match_oracle(D, T, causal, with_mod):
    """fp32 lengths of two and three 32-row tiles: the D = 128 dQ kernel
    runs tile t's sigmoid arithmetic under tile t+1's MFMA chains over a
    three-stage ring, whose first and last iterations (and, causal, each
    wave's own last tile) these cover; score_mod sits in that ring too."""
    B, H = 2, 3
    dtype = torch.float32
    q, k, v, do = _inputs(B, T, H, D, dtype, seed=T * 5 + D + causal)
    sm = torch.randn((B, T), generator=torch.Generator().manual_seed(T)).to(DEV) if with_mod else None
    for t in (q, k, v):
        t.requires_grad_(True)
    o = ts.sigmoid_attention(q, k, v, is_causal=causal, score_mod=sm)
    o.backward(do)
    bias = np.full(B, -math.log(T), dtype=np.float32).astype(np.float64)
    want_o, (dq, dk, dv) = oracle_fwd_bwd(q, k, v, do, scale=np.float32(1.0 / math.sqrt(D)), bias=bias,
                                          score_mod=sm, causal=causal)
    assert_close_to_oracle(o, want_o, dtype, "O")
    assert_close_to_oracle(q.grad, dq, dtype, "dQ")
    assert_close_to_oracle(k.grad, dk, dtype, "dK")
    assert_close_to_oracle(v.grad, dv, dtype, "dV")


@pytest.mark.parametrize("H", [1, 5, 12])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
def test_various_num_heads_match_oracle(H, D):
    """Head counts that do not divide any tile (the reference's
    tests/test_sigmoid_dense.py:621-637 checks shape and NaN only)."""
    B, T = 2, 200
    dtype = torch.bfloat16
    q, k, v, do = _inputs(B, T, H, D, dtype, seed=H * 31 + D)
    for t in (q, k, v):
        t.requires_grad_(True)
    o = ts.sigmoid_attention(q, k, v, is_causal=True)
    o.backward(do)
    bias = np.full(B, -math.log(T), dtype=np.float32).astype(np.float64)
    want_o, (dq, dk, dv) = oracle_fwd_bwd(q, k, v, do, scale=np.float32(1.0 / math.sqrt(D)), bias=bias,
                                          causal=True)
    assert o.shape == (B, T, H, D)
    assert_close_to_oracle(o, want_o, dtype, "O")
    assert_close_to_oracle(q.grad, dq, dtype, "dQ")
    assert_close_to_oracle(k.grad, dk, dtype, "dK")
    assert_close_to_oracle(v.grad, dv, dtype, "dV")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_dense_score_mod_matches_oracle(dtype, D, causal):
    B, T, H = 2, 200, 2
    q, k, v, do = _inputs(B, T, H, D, dtype, seed=11)
    g = torch.Generator().manual_seed(5)
    sm = torch.randn((B, T), generator=g).to(dtype).to(DEV)
    for t in (q, k, v):
        t.requires_grad_(True)
    o = ts.sigmoid_attention(q, k, v, is_causal=causal, score_mod=sm, sigmoid_bias=-2.0, scale=0.1)
    o.backward(do)
    want_o, (dq, dk, dv) = oracle_fwd_bwd(q, k, v, do, scale=np.float32(0.1), bias=np.full(B, -2.0),
                                          score_mod=sm, causal=causal)
    assert_close_to_oracle(o, want_o, dtype, "O")
    assert_close_to_oracle(q.grad, dq, dtype, "dQ")
    assert_close_to_oracle(k.grad, dk, dtype, "dK")
    assert_close_to_oracle(v.grad, dv, dtype, "dV")


# --- the reference's own criterion (tests/test_sigmoid_dense.py:35-166) -------
# Same grid as the reference's test_dense_op: B, H in {(1, 2), (4, 8)},
# T in {128 ... 4096}, D in {64, 128}, causal, fp16 / bf16 / fp32.

@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,H", [(1, 2), (4, 8)])
@pytest.mark.parametrize("T", [128, 256, 512, 1024, 2048, 4096])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_dense_reference_criterion(dtype, B, H, T, D, causal):
    tol = get_tolerance(dtype)
    q, k, v, do = _inputs(B, T, H, D, dtype, seed=B + T + D, std=0.5)
    do = (do.float() * 2.0).to(dtype)  # N(0, 1) like torch.randn_like(out) in the reference test
    errs = criterion_errors(q, k, v, do, lambda a, b, c: ts.sigmoid_attention(a, b, c, is_causal=causal),
                            dict(causal=causal))
    assert_reference_criterion(errs, tol)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [16, 32])
@pytest.mark.parametrize("T", [128, 1024, 4096])
@pytest.mark.parametrize("causal", [False, True])
def test_dense_reference_criterion_small_head(dtype, D, T, causal):
    """head_dim 16 and 32 (outside the reference criterion's own grid, which
    takes 64 and 128) on the MFMA kernels, at that criterion and its
    B, H = 4, 8."""
    B, H = 4, 8
    tol = get_tolerance(dtype)
    q, k, v, do = _inputs(B, T, H, D, dtype, seed=B + T + D, std=0.5)
    do = (do.float() * 2.0).to(dtype)
    errs = criterion_errors(q, k, v, do, lambda a, b, c: ts.sigmoid_attention(a, b, c, is_causal=causal),
                            dict(causal=causal))
    assert_reference_criterion(errs, tol)


# --- BASELINE parity bar: max-abs <= 2e-2 vs fp32 eager at N(0,1) --------------

def _fp32_reference(q, k, v, do, causal, chunk_b=1):
    outs, gq, gk, gv = [], [], [], []
    for b0 in range(0, q.shape[0], chunk_b):
        sl = slice(b0, b0 + chunk_b)
        qq, kk, vv = (t[sl].detach().float().requires_grad_(True) for t in (q, k, v))
        o = sigmoid_attention_eager(qq, kk, vv, causal=causal, upcast=True)
        o.backward(do[sl].float())
        outs.append(o.detach())
        gq.append(qq.grad)
        gk.append(kk.grad)
        gv.append(vv.grad)
        del o, qq, kk, vv
    return torch.cat(outs), torch.cat(gq), torch.cat(gk), torch.cat(gv)


@pytest.mark.parametrize("cfg", [
    dict(B=2, T=1024, H=8, D=64, dtype=torch.float16, causal=False),
    dict(B=2, T=1024, H=8, D=64, dtype=torch.float16, causal=True),
    dict(B=4, T=4096, H=16, D=128, dtype=torch.bfloat16, causal=True),
], ids=["c2-noncausal", "c2-causal", "c3-headline"])
def test_baseline_configs_within_2e2(cfg):
    B, T, H, D = cfg["B"], cfg["T"], cfg["H"], cfg["D"]
    q, k, v, do = _inputs(B, T, H, D, cfg["dtype"], seed=0)
    for t in (q, k, v):
        t.requires_grad_(True)
    o = ts.sigmoid_attention(q, k, v, is_causal=cfg["causal"])
    o.backward(do)
    ro, rq, rk, rv = _fp32_reference(q, k, v, do, cfg["causal"])
    for name, got, want in (("O", o, ro), ("dQ", q.grad, rq), ("dK", k.grad, rk), ("dV", v.grad, rv)):
        err = (got.float() - want).abs().max().item()
        assert err <= 2e-2, (name, err)


@pytest.mark.parametrize("B,T,H,ws_mb", [(2, 8192, 16, None), (1, 16384, 16, None), (1, 16384, 16, "0")],
                         ids=["L8192-two-pass", "L16384-two-pass", "L16384-recompute"])
def test_reference_grid_long_shapes(B, T, H, ws_mb, monkeypatch):
    """The long end of the reference's benchmark grid (bf16 D=128 non-causal,
    sigmoid_bias=0, B = 16384/L, H = 2048/D: benchmarks/benchmark_sigmoid.py:
    193,202), through the public API.  Under the default 2 GiB workspace cap
    the backward is the two-pass one in head groups: two groups of 8 heads at
    L=8192, four of 4 at L=16384 (whose dQ-from-dS launches take 256-row
    workgroups to fill the GPU); with no workspace allowed
    (SIGATTN_BWD_WORKSPACE_MB=0) the recompute backward runs.

    With sigmoid_bias=0 every P is near 1/2 and O sums thousands of them:
    |O| reaches ~150 and one bf16 rounding step there is 1.0, so an absolute
    2e-2 bound cannot hold for any bf16 kernel.  Each (batch, head) slice is
    held instead to the reference tests' relative criterion against fp32 eager
    (error <= 2x (forward) / 3x (backward) the mixed-precision eager path's
    error + tol, tests/test_sigmoid_dense.py:111-114,154-166) and to 2e-2 of
    the slice's largest fp32 magnitude."""
    from oracle.eager import mixed_fwd_bwd
    if ws_mb is not None:
        monkeypatch.setenv("SIGATTN_BWD_WORKSPACE_MB", ws_mb)
    D, tol = 128, get_tolerance(torch.bfloat16)
    q, k, v, do = _inputs(B, T, H, D, torch.bfloat16, seed=T)
    for t in (q, k, v):
        t.requires_grad_(True)
    o = ts.sigmoid_attention(q, k, v, sigmoid_bias=0.0)
    o.backward(do)
    ours = (o.detach(), q.grad, k.grad, v.grad)
    for b in range(B):
        for h in range(H):
            sl = (slice(b, b + 1), slice(None), slice(h, h + 1))
            qq, kk, vv = (t[sl].detach().float().requires_grad_(True) for t in (q, k, v))
            ro = sigmoid_attention_eager(qq, kk, vv, sigmoid_bias=0.0, upcast=True)
            ro.backward(do[sl].float())
            ref = (ro.detach(), qq.grad, kk.grad, vv.grad)
            mixed = mixed_fwd_bwd(*(t[sl].detach() for t in (q, k, v, do)), sigmoid_bias=0.0)
            for i, name in enumerate(("O", "dQ", "dK", "dV")):
                r = ref[i].float()
                err = (ours[i][sl].float() - r).abs().max().item()
                err_mixed = (mixed[i].float() - r).abs().max().item()
                f = 2.0 if name == "O" else 3.0
                assert err <= f * err_mixed + tol, (b, h, name, err, err_mixed)
                assert err <= 2e-2 * r.abs().max().item(), (b, h, name, err, r.abs().max().item())
            del ro, qq, kk, vv, ref, mixed


@pytest.mark.parametrize("causal", [False, True])
def test_c1_fp32_matches_oracle(causal):
    """fp32 B=2 L=256 H=4 D=64, q/k/v/dO ~ N(0,1)
    from a seed, scale 1/sqrt(D), default bias -log(L), fwd+bwd through the
    public API (the fp32 MFMA kernels) against the float64 oracle."""
    B, T, H, D = 2, 256, 4, 64
    q, k, v, do = _inputs(B, T, H, D, torch.float32, seed=0)
    for t in (q, k, v):
        t.requires_grad_(True)
    o = ts.sigmoid_attention(q, k, v, is_causal=causal)
    o.backward(do)
    bias = np.full(B, -math.log(T), dtype=np.float32).astype(np.float64)
    want_o, (dq, dk, dv) = oracle_fwd_bwd(q, k, v, do, scale=np.float32(1.0 / math.sqrt(D)), bias=bias,
                                          causal=causal)
    assert_close_to_oracle(o, want_o, torch.float32, "O")
    assert_close_to_oracle(q.grad, dq, torch.float32, "dQ")
    assert_close_to_oracle(k.grad, dk, torch.float32, "dK")
    assert_close_to_oracle(v.grad, dv, torch.float32, "dV")


def _off_boundary(t):
    """A contiguous copy of t whose data starts one element past a 16-byte
    boundary (a view one element into its storage), as a leaf."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:].copy_(t.reshape(-1))
    return buf[1:].view(t.shape).detach()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("causal", [False, True])
def test_rows_off_16_byte_boundaries_match_oracle(dtype, causal):
    """Q, K, V and dO whose rows do not start on 16-byte boundaries cannot be
    copied into LDS by the MFMA kernels' 16-byte tile copies; the portable
    kernels take them, with the same results."""
    B, T, H, D = 2, 130, 3, 64
    q, k, v, do = (_off_boundary(t) for t in _inputs(B, T, H, D, dtype, seed=21))
    assert all(t.data_ptr() % 16 != 0 for t in (q, k, v, do))
    for t in (q, k, v):
        t.requires_grad_(True)
    o = ts.sigmoid_attention(q, k, v, is_causal=causal)
    o.backward(do)
    bias = np.full(B, -math.log(T), dtype=np.float32).astype(np.float64)
    want_o, (dq, dk, dv) = oracle_fwd_bwd(q, k, v, do, scale=np.float32(1.0 / math.sqrt(D)), bias=bias,
                                          causal=causal)
    assert_close_to_oracle(o, want_o, dtype, "O")
    assert_close_to_oracle(q.grad, dq, dtype, "dQ")
    assert_close_to_oracle(k.grad, dk, dtype, "dK")
    assert_close_to_oracle(v.grad, dv, dtype, "dV")


@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (32, torch.bfloat16), (16, torch.bfloat16)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("with_mod", [False, True])
def test_one_launch_backward_equals_the_two_kernels(D, dtype, causal, with_mod):
    """At c2's size (B=2 L=1024 H=8: 128 dQ and 128 dK/dV workgroups) the
    recompute backward runs both kernels as one launch; its dQ, dK and dV
    equal those of the two kernels run alone (sigattn_bwd_dq,
    sigattn_bwd_dkdv) bit for bit."""
    lib = _capi.load_library()
    B, T, H = 2, 1024, 8
    q, k, v, do = _inputs(B, T, H, D, dtype, seed=D + 2 * causal + with_mod)
    bias = torch.full((B,), -math.log(T), device=DEV)
    scale = torch.tensor(1 / math.sqrt(D), device=DEV)
    sm = torch.randn((B, T), generator=torch.Generator().manual_seed(4)).to(DEV) if with_mod else None
    pr = _capi._problem(q, k, v, bias, sm, scale, None, None, causal)
    stream = torch.cuda.current_stream().cuda_stream
    one = [torch.full_like(q, float("nan")) for _ in range(3)]
    two = [torch.full_like(q, float("nan")) for _ in range(3)]
    assert lib.sigattn_bwd(ctypes.byref(pr), do.data_ptr(), *(t.data_ptr() for t in one), stream) == 0
    assert lib.sigattn_bwd_dq(ctypes.byref(pr), do.data_ptr(), two[0].data_ptr(), stream) == 0
    assert lib.sigattn_bwd_dkdv(ctypes.byref(pr), do.data_ptr(), two[1].data_ptr(), two[2].data_ptr(), stream) == 0
    torch.cuda.synchronize()
    for name, a, b in zip(("dQ", "dK", "dV"), one, two):
        assert torch.isfinite(a).all(), name
        assert torch.equal(a, b), name


# --- behaviour -----------------------------------------------------------------

def test_causal_past_outputs_ignore_future_keys():
    B, T, H, D = 1, 512, 2, 128
    q, k, v, _ = _inputs(B, T, H, D, torch.bfloat16, seed=3)
    o1 = ts.sigmoid_attention(q, k, v, is_causal=True)
    k2, v2 = k.clone(), v.clone()
    k2[:, 300:] = torch.randn_like(k2[:, 300:])
    v2[:, 300:] = torch.randn_like(v2[:, 300:])
    o2 = ts.sigmoid_attention(q, k2, v2, is_causal=True)
    assert torch.equal(o1[:, :300], o2[:, :300])
    assert not torch.equal(o1[:, 300:], o2[:, 300:])


@pytest.mark.parametrize("dtype", DTYPES)
def test_forward_and_backward_are_bitwise_deterministic(dtype):
    B, T, H, D = 2, 640, 4, 64
    q, k, v, do = _inputs(B, T, H, D, dtype, seed=4)
    res = []
    for _ in range(2):
        leaves = [t.detach().clone().requires_grad_(True) for t in (q, k, v)]
        o = ts.sigmoid_attention(*leaves, is_causal=True)
        o.backward(do)
        res.append([o.detach()] + [t.grad for t in leaves])
    for a, b in zip(*res):
        assert torch.equal(a, b)


def test_score_mod_zero_equals_none_and_constant_equals_bias():
    B, T, H, D = 2, 256, 2, 64
    q, k, v, _ = _inputs(B, T, H, D, torch.float16, seed=6)
    a = ts.sigmoid_attention(q, k, v)
    b = ts.sigmoid_attention(q, k, v, score_mod=torch.zeros(B, T, device=DEV))
    assert torch.equal(a, b)
    c = ts.sigmoid_attention(q, k, v, sigmoid_bias=-3.0, score_mod=torch.full((B, T), 1.0, device=DEV))
    d = ts.sigmoid_attention(q, k, v, sigmoid_bias=-2.0)
    torch.testing.assert_close(c, d, atol=2e-3, rtol=0)


def test_non_contiguous_inputs():
    B, T, H, D = 2, 200, 4, 64
    base = torch.randn(B, H, T, D, device=DEV, dtype=torch.bfloat16)
    q = base.transpose(1, 2)  # [B, T, H, D] view, not contiguous
    assert not q.is_contiguous()
    o = ts.sigmoid_attention(q, q, q)
    o2 = ts.sigmoid_attention(q.contiguous(), q.contiguous(), q.contiguous())
    assert torch.equal(o, o2)


def test_large_inputs_give_finite_gradients():
    B, T, H, D = 1, 256, 2, 64
    q, k, v, do = _inputs(B, T, H, D, torch.float16, seed=8)
    q, k, v = (t * 10 for t in (q, k, v))
    for t in (q, k, v):
        t.requires_grad_(True)
    o = ts.sigmoid_attention(q, k, v)
    o.backward(do)
    for t in (o, q.grad, k.grad, v.grad):
        assert torch.isfinite(t).all()
        assert t.abs().max() < 1e6


def test_zero_inputs():
    B, T, H, D = 1, 128, 2, 64
    z = torch.zeros(B, T, H, D, device=DEV, dtype=torch.float16, requires_grad=True)
    o = ts.sigmoid_attention(z, z, z)
    assert torch.equal(o, torch.zeros_like(o))
    o.sum().backward()
    assert torch.isfinite(z.grad).all()


def test_requires_grad_subsets():
    B, T, H, D = 1, 64, 2, 64
    q, k, v, do = _inputs(B, T, H, D, torch.bfloat16, seed=9)
    q.requires_grad_(True)
    o = ts.sigmoid_attention(q, k, v)
    o.backward(do)
    assert q.grad is not None and k.grad is None and v.grad is None


def test_empty_batch_and_length():
    for shape in [(0, 16, 2, 64), (2, 0, 2, 64)]:
        x = torch.randn(*shape, device=DEV, dtype=torch.float16)
        o = ts.sigmoid_attention(x, x, x)
        assert o.shape == x.shape


@pytest.mark.parametrize("T", [1, 7, 15, 33])
def test_tiny_sequence_lengths(T):
    B, H, D = 2, 2, 64
    q, k, v, do = _inputs(B, T, H, D, torch.float16, seed=T)
    o = ts.sigmoid_attention(q, k, v, is_causal=True)
    want, _ = oracle_fwd_bwd(q, k, v, do, scale=np.float32(1 / math.sqrt(D)),
                             bias=np.full(B, np.float32(-math.log(T))), causal=True, with_bwd=False)
    assert_close_to_oracle(o, want, torch.float16, "O")


# --- fp32 kernels: waves per row group, and values the bf16 splits cannot hold ---

@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("B,H,T", [(2, 3, 61), (2, 3, 257),      # four waves share 32 rows (two at D = 128)
                                   (4, 17, 161),                 # two waves share 64 rows: more than 256 blocks of 32
                                   (15, 18, 129)])               # one wave per 32 rows: 540 blocks of 128
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("with_mod", [False, True])
def test_fp32_waves_per_rows_match_oracle(B, H, T, D, causal, with_mod):
    """Each form of the fp32 kernels at remainders of its row blocks and
    streamed steps, padded lengths among them, on a few of the heads."""
    dtype = torch.float32
    q, k, v, do = _inputs(B, T, H, D, dtype, seed=B * T + D)
    g = torch.Generator().manual_seed(T)
    mod = torch.randn((B, T), generator=g).to(DEV) if with_mod else None
    lens = torch.randint(1, T + 1, (B,), generator=g, dtype=torch.int32)
    lens[0], lens[1] = T, max(1, T - 33)
    for t in (q, k, v):
        t.requires_grad_(True)
    ld = lens.to(DEV)
    o = ts.sigmoid_attention_padded(q, k, v, ld, ld, is_causal=causal, sigmoid_bias=-2.0, score_mod=mod)
    o.backward(do)
    for b, h in ((0, 0), (0, H - 1), (1, 1), (B - 1, H // 2)):
        n = int(lens[b])
        one = [t.detach()[b:b + 1, :n, h:h + 1] for t in (q, k, v, do)]
        want_o, grads = oracle_fwd_bwd(*one, scale=np.float32(1.0 / math.sqrt(D)), bias=np.full(1, -2.0),
                                       causal=causal, score_mod=None if mod is None else mod[b:b + 1, :n])
        for name, got, want in zip(("O", "dQ", "dK", "dV"), (o, q.grad, k.grad, v.grad), (want_o, *grads)):
            assert_close_to_oracle(got[b:b + 1, :n, h:h + 1], want, dtype, name)
            assert torch.all(got[b, n:] == 0)


@pytest.mark.parametrize("D", [32, 64, 128])  # 16 runs at width 32, where an infinity meets zeros
@pytest.mark.parametrize("T", [96, 320])  # whole tiles: a tail repeats the last row, and 0 * inf is NaN
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kind", ["nan", "inf", "-inf", "max", "tiny", "mask"])
def test_fp32_values_outside_the_split_match_the_portable_kernels(D, T, causal, kind):
    """Infinities, NaN, magnitudes above bf16's largest and below its smallest,
    and score_mod of the type's lowest value: the fp32 kernels against the
    portable ones (rows off 16-byte boundaries), which use plain FMAs."""
    B, H = 2, 3
    q, k, v, do = _inputs(B, T, H, D, torch.float32, seed=T + D)
    mod = torch.zeros((B, T), device=DEV)
    if kind == "tiny":
        v.mul_(1e-36)
        do.mul_(1e-36)
    elif kind == "mask":
        mod[:, T // 2:] = torch.finfo(torch.float32).min
        mod[1, 3] = float("-inf")
    else:
        x = float(kind) if kind != "max" else 3.4e38
        # The first key and the last query: no mask stands between them and any
        # other row (a masked pair's 0 * inf is NaN in whichever kernel's tile has it).
        q[0, T - 1, 0, 1] = x
        k[0, 0, 1, 2] = x
        v[1, 0, 1, 3] = x
        do[1, T - 1, 2, 0] = x
    lib = _capi.load_library()
    bias = torch.full((B,), -2.0, device=DEV)
    scale = torch.tensor(1 / math.sqrt(D), device=DEV)
    stream = torch.cuda.current_stream().cuda_stream

    def run(pad):
        # pad = 1: heads D + 1 floats apart, so most rows start off 16 bytes.
        ins = [torch.nn.functional.pad(t, (0, pad))[..., :D] for t in (q, k, v, do)]
        outs = [torch.nn.functional.pad(torch.full_like(t, 7.0), (0, pad))[..., :D] for t in (q, q, k, k)]
        pr = _capi._problem(*ins[:3], bias, mod, scale, None, None, causal)
        assert lib.sigattn_fwd(ctypes.byref(pr), outs[0].data_ptr(), stream) == 0
        assert lib.sigattn_bwd(ctypes.byref(pr), ins[3].data_ptr(), *(t.data_ptr() for t in outs[1:]), stream) == 0
        torch.cuda.synchronize()
        return outs

    for name, got, want in zip(("O", "dQ", "dK", "dV"), run(0), run(1)):
        assert torch.equal(torch.isnan(got), torch.isnan(want)), name
        assert torch.equal(torch.isinf(got), torch.isinf(want)), name
        fine = torch.isfinite(want)
        # fp32 sums of up to T and D terms in two orders: a few roundings of the largest value.
        top = want[fine].abs().max().item() if fine.any() else 0.0
        torch.testing.assert_close(got[fine], want[fine], rtol=0, atol=2 ** -24 * 64 * top)


def _fp32_and_portable(ins, mod, causal):
    """O, dQ, dK, dV of the fp32 kernels and of the portable ones (heads D + 1
    floats apart, so most rows start off 16 bytes), bias -2."""
    B, T, H, D = ins[0].shape
    lib = _capi.load_library()
    bias = torch.full((B,), -2.0, device=DEV)
    scale = torch.tensor(1 / math.sqrt(D), device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    both = []
    for pad in (0, 1):
        i = [torch.nn.functional.pad(t, (0, pad))[..., :D] for t in ins]
        o = [torch.nn.functional.pad(torch.full_like(t, 7.0), (0, pad))[..., :D] for t in ins]
        pr = _capi._problem(*i[:3], bias, mod, scale, None, None, causal)
        assert lib.sigattn_fwd(ctypes.byref(pr), o[0].data_ptr(), stream) == 0
        assert lib.sigattn_bwd(ctypes.byref(pr), i[3].data_ptr(), *(t.data_ptr() for t in o[1:]), stream) == 0
        torch.cuda.synchronize()
        both.append(o)
    return both


@pytest.mark.parametrize("D,B,H,T", [(32, 2, 3, 96), (64, 2, 3, 320), (64, 4, 64, 257), (128, 2, 3, 161)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kind", ["q", "k", "q-denormal", "do-v", "v-do", "do-k", "do-q", "one-key", "one-query",
                                  "probability"])
def test_fp32_tiny_operands_of_ordinary_results_match_the_portable_kernels(D, B, H, T, causal, kind):
    """Operands too small for three bf16 parts against large ones, so that the
    scores, dP or the results are of a size that shows nothing of it."""
    q, k, v, do = _inputs(B, T, H, D, torch.float32, seed=T + D)
    mod = None
    if kind == "q":
        q, k = q * 1e-35, k * 1e35
    elif kind == "k":
        q, k = q * 1e35, k * 1e-35
    elif kind == "q-denormal":
        q, k = q * 1e-38, k * 1e36
    elif kind == "do-v":
        do, v = do * 1e-36, v * 1e36
    elif kind == "v-do":
        do, v = do * 1e36, v * 1e-36
    elif kind == "do-k":
        do, q, k = do * 1e-36, q * 1e-12, k * 1e12
    elif kind == "do-q":
        do, q, k = do * 1e-36, q * 1e12, k * 1e-12
    elif kind == "probability":  # P and dS, not the inputs, are tiny
        q, k, v, do, mod = q * 1e-13, k * 1e12, v * 1e30, do * 1e-30, torch.full((B, T), -83.0, device=DEV)
    elif kind == "one-key":  # a single streamed (dQ) or stationary (dK, dV) row
        k[0, T - 2, 1] *= 1e-35
        q[0, :, 1, :3] *= 1e35
        k[0, :T - 2, 1, :3] = 0.0
        k[0, T - 1:, 1, :3] = 0.0
        q[0, :, 1, 3:] = 0.0
    else:
        q[0, T - 1, 1] *= 1e-35
        k[0, :, 1, :3] *= 1e35
        q[0, :T - 1, 1, :3] = 0.0
        k[0, :, 1, 3:] = 0.0
    got, want = _fp32_and_portable((q, k, v, do), mod, causal)
    for name, x, y in zip(("O", "dQ", "dK", "dV"), got, want):
        assert torch.isfinite(y).all(), name
        # fp32 sums of up to T and D terms in two orders: a few roundings of a head's largest value.
        # Scores near -83 are 2^7 as exponents of two, whose last bit is 2^-17: two of those in P.
        top = y.abs().amax(dim=(1, 3), keepdim=True)
        bound = 2 ** -24 * 64 + (2 ** -16 if kind == "probability" else 0)
        assert torch.all((x - y).abs() <= bound * top), (name, ((x - y).abs() / top).max().item())


# --- D <= 64 forward and dQ: two waves per 32 rows on small grids, one on larger ones ---

@pytest.mark.parametrize("D", [16, 32, 64])
@pytest.mark.parametrize("T", [63, 65, 96, 129, 257, 321])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("layout", ["dense", "mod", "padded"])
def test_wave_pairs_and_single_waves_match_oracle(D, T, causal, layout):
    """17 x 64 (batch, head) pairs are more than four blocks per compute unit
    (a wave per 32 rows); one pair alone is a small grid (two waves per 32 rows in
    the forward and, padded, in dQ).  Both against the oracle, on remainders of 32-, 64-,
    128- and 256-row blocks."""
    B, H, dtype = 17, 64, torch.bfloat16
    q, k, v, do = _inputs(B, T, H, D, dtype, seed=T + D)
    g = torch.Generator().manual_seed(T)
    mod = torch.randn((B, T), generator=g).to(DEV) if layout == "mod" else None
    lens = torch.full((B,), T, dtype=torch.int32)
    if layout == "padded":
        lens[1:] = torch.randint(1, T + 1, (B - 1,), generator=g, dtype=torch.int32)

    def run(bs, hs):
        ins = [t[bs, :, hs].contiguous().requires_grad_(True) for t in (q, k, v)]
        m = None if mod is None else mod[bs].contiguous()
        if layout == "padded":
            n = lens[bs].to(DEV)
            o = ts.sigmoid_attention_padded(*ins, n, n, is_causal=causal, sigmoid_bias=-2.0)
        else:
            o = ts.sigmoid_attention(*ins, is_causal=causal, sigmoid_bias=-2.0, score_mod=m)
        return (o, *torch.autograd.grad(o, ins, do[bs, :, hs].contiguous()))

    whole = run(slice(0, B), slice(0, H))
    for b, h in ((0, 0), (3, H - 1), (B - 1, 17)):
        n = int(lens[b])
        alone = run(slice(b, b + 1), slice(h, h + 1))
        one = [t[b:b + 1, :n, h:h + 1] for t in (q, k, v, do)]
        want_o, grads = oracle_fwd_bwd(*one, scale=np.float32(1.0 / math.sqrt(D)), bias=np.full(1, -2.0),
                                       causal=causal, score_mod=None if mod is None else mod[b:b + 1])
        for name, x, y, want in zip(("O", "dQ", "dK", "dV"), whole, alone, (want_o, *grads)):
            assert_close_to_oracle(x[b:b + 1, :n, h:h + 1], want, dtype, f"{name}, large grid")
            assert_close_to_oracle(y[:, :n], want, dtype, f"{name}, alone")
            assert torch.all(x[b, n:] == 0) and torch.all(y[:, n:] == 0)


@pytest.mark.parametrize("T", [961, 1000, 1023, 1024])  # remainders of 32-, 64-, 128- and 256-row blocks
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("layout", ["dense", "mod", "padded"])
def test_wide_waves_match_oracle(T, causal, layout):
    """Four blocks of 256 queries per compute unit (eight of padded ones) run 64
    queries per wave at D = 64: O of a few sequences and heads."""
    B, H, D, dtype = 32 if layout == "padded" else 16, 16, 64, torch.bfloat16
    q, k, v, _ = _inputs(B, T, H, D, dtype, seed=T)
    g = torch.Generator().manual_seed(T)
    mod = torch.randn((B, T), generator=g).to(DEV) if layout == "mod" else None
    lens = torch.full((B,), T, dtype=torch.int32)
    if layout == "padded":
        lens[1:] = torch.randint(1, T + 1, (B - 1,), generator=g, dtype=torch.int32)
        n = lens.to(DEV)
        o = ts.sigmoid_attention_padded(q, k, v, n, n, is_causal=causal, sigmoid_bias=-2.0)
    else:
        o = ts.sigmoid_attention(q, k, v, is_causal=causal, sigmoid_bias=-2.0, score_mod=mod)
    for b, h in ((0, 0), (3, H - 1), (B - 1, 7)):
        n = int(lens[b])
        one = [t[b:b + 1, :n, h:h + 1] for t in (q, k, v)]
        want, _ = oracle_fwd_bwd(*one, None, scale=np.float32(1.0 / math.sqrt(D)), bias=np.full(1, -2.0), causal=causal,
                                 score_mod=None if mod is None else mod[b:b + 1], with_bwd=False)
        assert_close_to_oracle(o[b:b + 1, :n, h:h + 1], want, dtype, "O")
        assert torch.all(o[b, n:] == 0)


@pytest.mark.parametrize("D", [16, 32, 64])
@pytest.mark.parametrize("B,H,T", [(10, 20, 63), (10, 10, 129), (5, 13, 321)])  # 200, 200 and 195 blocks of 128 rows
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("with_mod", [False, True])
def test_dq_wave_pairs_of_dense_grids_match_oracle(D, B, H, T, causal, with_mod):
    """Dense grids of up to one 128-row block per compute unit that do not fit
    the one-launch backward's single workgroup per unit run dQ in pairs of
    waves: two of the heads against the oracle, and the same bits apart."""
    dtype = torch.bfloat16
    q, k, v, do = _inputs(B, T, H, D, dtype, seed=T + D)
    g = torch.Generator().manual_seed(T)
    mod = torch.randn((B, T), generator=g).to(DEV) if with_mod else None
    bias = torch.full((B,), -2.0, device=DEV)
    scale = torch.tensor(1 / math.sqrt(D), device=DEV)
    lib = _capi.load_library()
    pr = _capi._problem(q, k, v, bias, mod, scale, None, None, causal)
    one = [torch.full_like(t, float("nan")) for t in (q, k, v)]
    two = [torch.full_like(t, float("nan")) for t in (q, k, v)]
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.sigattn_bwd(ctypes.byref(pr), do.data_ptr(), *(t.data_ptr() for t in one), stream) == 0
    assert lib.sigattn_bwd_dq(ctypes.byref(pr), do.data_ptr(), two[0].data_ptr(), stream) == 0
    assert lib.sigattn_bwd_dkdv(ctypes.byref(pr), do.data_ptr(), two[1].data_ptr(), two[2].data_ptr(), stream) == 0
    torch.cuda.synchronize()
    for a, b in zip(one, two):
        assert torch.equal(a, b)
    for b, h in ((0, H - 1), (B - 1, 1)):
        ins = [t[b:b + 1, :, h:h + 1] for t in (q, k, v, do)]
        _, grads = oracle_fwd_bwd(*ins, scale=np.float32(1.0 / math.sqrt(D)), bias=np.full(1, -2.0), causal=causal,
                                  score_mod=None if mod is None else mod[b:b + 1])
        for name, x, want in zip(("dQ", "dK", "dV"), one, grads):
            assert_close_to_oracle(x[b:b + 1, :, h:h + 1], want, dtype, name)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("B,H,T", [(15, 18, 33), (10, 18, 100), (15, 18, 100), (9, 12, 130)])
@pytest.mark.parametrize("causal", [False, True])
def test_fp32_short_padded_rows_match_oracle(D, B, H, T, causal):
    """Short streamed rows: index order (WorkOrder's from 129 on) and one wave per
    32 rows of D = 128 grids of more than half a block per compute unit."""
    test_fp32_waves_per_rows_match_oracle(B, H, T, D, causal, False)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,T", [(10, 18, 100), (10, 14, 200), (5, 9, 400)])  # 180, 280 and 180 blocks of 128 rows
@pytest.mark.parametrize("causal", [False, True])
def test_fp32_dense_waves_per_rows_match_oracle(D, B, H, T, causal):
    dtype = torch.float32
    q, k, v, do = _inputs(B, T, H, D, dtype, seed=T + D)
    for t in (q, k, v):
        t.requires_grad_(True)
    o = ts.sigmoid_attention(q, k, v, is_causal=causal, sigmoid_bias=-2.0)
    o.backward(do)
    for b, h in ((0, H - 1), (B - 1, 0)):
        one = [t.detach()[b:b + 1, :, h:h + 1] for t in (q, k, v, do)]
        want_o, grads = oracle_fwd_bwd(*one, scale=np.float32(1.0 / math.sqrt(D)), bias=np.full(1, -2.0), causal=causal)
        for name, got, want in zip(("O", "dQ", "dK", "dV"), (o, q.grad, k.grad, v.grad), (want_o, *grads)):
            assert_close_to_oracle(got[b:b + 1, :, h:h + 1], want, dtype, name)
