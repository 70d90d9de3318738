"""GPU parity tests for the split-KV forward (decode shapes: Tq <= 32 queries
against Tk >= 256 keys, non-causal), which sigmoid_attention_padded and
sigmoid_attention_varlen take automatically.  The reference has no separate
decode path: its padded forward (sigmoid_triton_padded.py:24-171) computes
these shapes with one program per 16..128-query block, so the semantics, and
the float64 oracle they are checked against, are the padded forward's."""

import ctypes
import math

import numpy as np
import pytest
import torch

import triton_sigmoid as ts
from helpers import assert_close_to_oracle, oracle_fwd_bwd, randn
from triton_sigmoid import _capi

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(B, Tq, Tk, H, D, dtype, seed, full=False):
    g = torch.Generator().manual_seed(seed)
    q = randn((B, Tq, H, D), dtype, DEV, g)
    k = randn((B, Tk, H, D), dtype, DEV, g)
    v = randn((B, Tk, H, D), dtype, DEV, g)
    sk = torch.full((B,), Tk, dtype=torch.int32) if full else torch.randint(1, Tk + 1, (B,), generator=g,
                                                                             dtype=torch.int32)
    sq = torch.full((B,), Tq, dtype=torch.int32) if full else torch.randint(0, Tq + 1, (B,), generator=g,
                                                                             dtype=torch.int32)
    for b in range(B):  # padding holds NaN: it must never be read
        k[b, sk[b]:] = float("nan")
        v[b, sk[b]:] = float("nan")
        q[b, sq[b]:] = float("nan")
    return q, k, v, sq, sk


def _clean(t, lens):
    t = t.detach().clone()
    for b in range(t.shape[0]):
        t[b, int(lens[b]):] = 0
    return t




@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("Tq,Tk", [(1, 256), (1, 4099), (5, 1000), (32, 20000), (17, 300)])
def test_decode_matches_oracle(dtype, D, Tq, Tk):
    # D = 16 and 32, and fp32, have no split-KV kernel: one MFMA forward
    # workgroup per 128 queries.
    B, H = 3, 4
    q, k, v, sq, sk = _case(B, Tq, Tk, H, D, dtype, seed=Tq * 1000 + Tk + D)
    o = ts.sigmoid_attention_padded(q, k, v, seq_lens_k=sk.to(DEV), seq_lens_q=sq.to(DEV))
    bias = (-torch.log(sk.float())).double().numpy()
    want, _ = oracle_fwd_bwd(_clean(q, sq), _clean(k, sk), _clean(v, sk), None,
                             scale=np.float32(1 / math.sqrt(D)), bias=bias, seq_lens_q=sq, seq_lens_k=sk,
                             with_bwd=False)
    assert_close_to_oracle(o, want, dtype, "O")
    for b in range(B):
        assert torch.all(o[b, sq[b]:] == 0)


@pytest.mark.parametrize("D", [64, 128])
def test_decode_score_mod_matches_oracle(D):
    B, Tq, Tk, H = 2, 3, 3000, 2
    q, k, v, sq, sk = _case(B, Tq, Tk, H, D, torch.bfloat16, seed=7)
    g = torch.Generator().manual_seed(8)
    sm = torch.randn((B, Tk), generator=g).to(DEV)
    o = ts.sigmoid_attention_padded(q, k, v, seq_lens_k=sk.to(DEV), seq_lens_q=sq.to(DEV), score_mod=sm,
                                    sigmoid_bias=-4.0)
    want, _ = oracle_fwd_bwd(_clean(q, sq), _clean(k, sk), _clean(v, sk), None,
                             scale=np.float32(1 / math.sqrt(D)), bias=np.full(B, -4.0), score_mod=sm,
                             seq_lens_q=sq, seq_lens_k=sk, with_bwd=False)
    assert_close_to_oracle(o, want, torch.bfloat16, "O")


@pytest.mark.parametrize("D", [64, 128])
def test_split_and_single_chunk_agree(D):
    """With a workspace the keys are cut into chunks; without one each
    (batch, head) is one chunk.  Both are deterministic and agree up to the
    fp32 summation order (a few bf16 ulps at most)."""
    lib = _capi.load_library()
    B, Tq, Tk, H = 2, 4, 9000, 2
    q, k, v, sq, sk = _case(B, Tq, Tk, H, D, torch.bfloat16, seed=D, full=True)
    bias = torch.full((B,), -math.log(Tk), device=DEV)
    scale = torch.tensor(1 / math.sqrt(D), device=DEV)
    sq_d, sk_d = sq.to(DEV), sk.to(DEV)   # the problem holds raw pointers: keep them alive
    pr = _capi._problem(q, k, v, bias, None, scale, sq_d, sk_d, False)
    nbytes = lib.sigattn_fwd_workspace_bytes(ctypes.byref(pr))
    assert nbytes > 0
    ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    outs = []
    for w in (ws, ws, None):
        o = torch.full_like(q, float("nan"))
        rc = lib.sigattn_fwd_ws(ctypes.byref(pr), o.data_ptr(), None if w is None else w.data_ptr(),
                                0 if w is None else nbytes, stream)
        assert rc == 0
        outs.append(o)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    torch.testing.assert_close(outs[0], outs[2], atol=2 ** -7 * outs[2].abs().max().item(), rtol=0)
    want, _ = oracle_fwd_bwd(q, k, v, None, scale=np.float32(1 / math.sqrt(D)),
                             bias=np.full(B, -math.log(Tk), dtype=np.float32).astype(np.float64),
                             seq_lens_q=sq, seq_lens_k=sk, with_bwd=False)
    assert_close_to_oracle(outs[0], want, torch.bfloat16, "split")
    assert_close_to_oracle(outs[2], want, torch.bfloat16, "single chunk")


def test_decode_packed_sequences():
    """Packed layout: one query per sequence against its own cache."""
    B, H, D = 6, 4, 128
    g = torch.Generator().manual_seed(12)
    lens_k = torch.randint(200, 5000, (B,), generator=g)
    cu_k = torch.cat([torch.zeros(1, dtype=torch.int64), lens_k.cumsum(0)]).to(torch.int32)
    cu_q = torch.arange(B + 1, dtype=torch.int32)
    q = randn((B, H, D), torch.bfloat16, DEV, g)
    k = randn((int(cu_k[-1]), H, D), torch.bfloat16, DEV, g)
    v = randn((int(cu_k[-1]), H, D), torch.bfloat16, DEV, g)
    o = ts.sigmoid_attention_varlen(q, k, v, cu_q.to(DEV), cu_k.to(DEV), 1, int(lens_k.max()))
    for b in range(B):
        ks, ke = int(cu_k[b]), int(cu_k[b + 1])
        want, _ = oracle_fwd_bwd(q[b:b + 1, None], k[None, ks:ke], v[None, ks:ke], None,
                                 scale=np.float32(1 / math.sqrt(D)),
                                 bias=(-torch.log(torch.tensor([float(ke - ks)]))).double().numpy(),
                                 with_bwd=False)
        assert_close_to_oracle(o[b:b + 1, None], want, torch.bfloat16, f"seq {b}")


def test_decode_backward_through_autograd():
    """Decode-shaped problems keep the standard backward kernels."""
    B, Tq, Tk, H, D = 2, 4, 1500, 2, 64
    q, k, v, sq, sk = _case(B, Tq, Tk, H, D, torch.float16, seed=5, full=True)
    g = torch.Generator().manual_seed(6)
    do = randn((B, Tq, H, D), torch.float16, DEV, g)
    for t in (q, k, v):
        t.requires_grad_(True)
    o = ts.sigmoid_attention_padded(q, k, v, seq_lens_k=sk.to(DEV), seq_lens_q=sq.to(DEV))
    o.backward(do)
    want_o, (dq, dk, dv) = oracle_fwd_bwd(q, k, v, do, scale=np.float32(1 / math.sqrt(D)),
                                          bias=(-torch.log(sk.float())).double().numpy(),
                                          seq_lens_q=sq, seq_lens_k=sk)
    assert_close_to_oracle(o, want_o, torch.float16, "O")
    assert_close_to_oracle(q.grad, dq, torch.float16, "dQ")
    assert_close_to_oracle(k.grad, dk, torch.float16, "dK")
    assert_close_to_oracle(v.grad, dv, torch.float16, "dV")


def test_decode_long_cache_sum_of_halves():
    """Size-independent check at a long cache (B=1, H=8, Tk=131072): O over
    the whole cache equals O over its two halves summed (same bias), within
    the bf16 rounding of the three outputs."""
    B, Tq, Tk, H, D = 1, 1, 131072, 8, 128
    q, k, v, sq, sk = _case(B, Tq, Tk, H, D, torch.bfloat16, seed=99, full=True)
    f = lambda kk, vv: ts.sigmoid_attention_padded(q, kk, vv, sigmoid_bias=-math.log(Tk)).float()
    whole = f(k, v)
    h1, h2 = f(k[:, :Tk // 2], v[:, :Tk // 2]), f(k[:, Tk // 2:], v[:, Tk // 2:])
    mag = max(t.abs().max().item() for t in (whole, h1, h2))
    torch.testing.assert_close(whole, h1 + h2, atol=3 * 2 ** -8 * mag, rtol=0)


@pytest.mark.parametrize("B,H,Tq,Tk,D,packed,mod", [
    (8, 16, 1, 2100, 64, False, False),    # chunks of at least 256 keys
    (10, 13, 3, 2111, 128, False, True),   # units not a multiple of the workgroup's four
    (8, 16, 32, 8200, 64, False, True),    # all 32 query rows
    (9, 16, 2, 3001, 128, True, True),     # packed rows
    (16, 128, 2, 300, 64, False, False),   # one chunk per (batch, head): no partials
    (64, 16, 1, 2100, 64, False, False),   # a sequence per lane, 2 rows of partials each
    (65, 16, 1, 2100, 64, False, False),   # one more: chunks of one length for all
    (12, 16, 32, 12000, 64, False, False), # keys for one round of waves, not for two
    (3, 16, 1, 30000, 128, False, True),   # ... and long sequences
])
def test_decode_wave_per_chunk_matches_the_general_path(B, H, Tq, Tk, D, packed, mod):
    """sigattn_fwd_decode's plan (a wave per chunk) against sigattn_fwd_ws and
    the oracle: ragged and empty caches, short last chunks and blocks."""
    lib = _capi.load_library()
    g = torch.Generator().manual_seed(B * Tk + D)
    lens = torch.randint(1, Tk + 1, (B,), generator=g)
    lens[0], lens[1], lens[2] = Tk, 0, 33
    rows = int(lens.sum())
    q = randn((B * Tq, H, D) if packed else (B, Tq, H, D), torch.bfloat16, DEV, g)
    k, v = (randn((rows, H, D) if packed else (B, Tk, H, D), torch.bfloat16, DEV, g) for _ in range(2))
    sm = torch.randn((rows,) if packed else (B, Tk), generator=g).to(DEV) if mod else None
    bias = torch.full((B,), -3.0, device=DEV)
    scale = torch.tensor(1 / math.sqrt(D), device=DEV)
    cu_q = (torch.arange(B + 1) * Tq).to(DEV, torch.int32)
    cu_k = torch.cat([torch.zeros(1, dtype=torch.int64), lens.cumsum(0)]).to(DEV, torch.int32)
    sq = torch.full((B,), Tq, dtype=torch.int32, device=DEV)
    sk = lens.to(DEV, torch.int32)
    if packed:
        pr = _capi._problem(q, k, v, bias, sm, scale, None, None, False, packed=(cu_q, cu_k, Tq, Tk))
    else:
        pr = _capi._problem(q, k, v, bias, sm, scale, sq, sk, False)
    stream = torch.cuda.current_stream().cuda_stream
    outs = []
    for size, run in ((lib.sigattn_fwd_decode_workspace_bytes, lib.sigattn_fwd_decode),
                      (lib.sigattn_fwd_workspace_bytes, lib.sigattn_fwd_ws)):
        n = size(ctypes.byref(pr))
        ws = torch.full((max(n, 1),), 255, dtype=torch.uint8, device=DEV)  # NaN bytes
        o = torch.full_like(q, float("nan"))
        assert run(ctypes.byref(pr), o.data_ptr(), ws.data_ptr(), n, stream) == 0
        outs.append(o.view(B, Tq, H, D))
    torch.cuda.synchronize()
    # One rounding to bf16 of sums in another order: at most one bf16 step of the largest value.
    torch.testing.assert_close(outs[0], outs[1], atol=2 ** -7 * outs[1].abs().max().item(), rtol=0)
    heads = slice(0, H, max(1, H // 2))
    qs = q.view(B, Tq, H, D)
    for b in range(min(B, 4)):
        n, first = int(lens[b]), int(cu_k[b])
        ks, vs = (t[first:first + n] if packed else t[b, :n] for t in (k, v))
        if n == 0:
            assert torch.all(outs[0][b] == 0)
            continue
        ms = None if sm is None else (sm[first:first + n] if packed else sm[b, :n])[None]
        want, _ = oracle_fwd_bwd(qs[b:b + 1, :, heads], ks[None, :, heads], vs[None, :, heads], None,
                                 scale=np.float32(1 / math.sqrt(D)), bias=np.full(1, -3.0), score_mod=ms,
                                 with_bwd=False)
        assert_close_to_oracle(outs[0][b:b + 1, :, heads], want, torch.bfloat16, f"sequence {b}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Tq,Tk,D", [(16, 128, 2, 300, 64), (16, 128, 1, 257, 128),  # enough (batch, head) pairs
                                         (8, 128, 32, 1000, 64)])                        # one chunk of 32 Tq keys
@pytest.mark.parametrize("mod", [False, True])
def test_decode_wave_per_pair_is_what_callers_without_a_workspace_get(dtype, B, H, Tq, Tk, D, mod):
    """One chunk per (batch, head) needs no partials: the public entry and a call
    without a workspace run the same kernel as one that is handed some memory."""
    lib = _capi.load_library()
    g = torch.Generator().manual_seed(Tk + D)
    lens = torch.randint(1, Tk + 1, (B,), generator=g)
    lens[0], lens[1], lens[2] = Tk, 0, 33
    q = randn((B, Tq, H, D), dtype, DEV, g)
    k, v = (randn((B, Tk, H, D), dtype, DEV, g) for _ in range(2))
    sm = torch.randn((B, Tk), generator=g).to(DEV) if mod else None
    bias = torch.full((B,), -3.0, device=DEV)
    scale = torch.tensor(1 / math.sqrt(D), device=DEV)
    sq = torch.full((B,), Tq, dtype=torch.int32, device=DEV)
    sk = lens.to(DEV, torch.int32)
    pr = _capi._problem(q, k, v, bias, sm, scale, sq, sk, False)
    assert lib.sigattn_fwd_decode_workspace_bytes(ctypes.byref(pr)) == 0
    stream = torch.cuda.current_stream().cuda_stream
    some = torch.zeros(256, dtype=torch.uint8, device=DEV)
    want, got, other = (torch.full_like(q, float("nan")) for _ in range(3))
    assert lib.sigattn_fwd_decode(ctypes.byref(pr), want.data_ptr(), some.data_ptr(), 0, stream) == 0
    assert lib.sigattn_fwd_decode(ctypes.byref(pr), got.data_ptr(), None, 0, stream) == 0
    assert lib.sigattn_fwd(ctypes.byref(pr), other.data_ptr(), stream) == 0
    api = ts.sigmoid_attention_padded(q, k, v, sk, sq, sigmoid_bias=-3.0, score_mod=sm)
    torch.cuda.synchronize()
    assert torch.equal(got, want) and torch.equal(api, want)
    # The shared form adds in another order: one rounding of the largest value.
    torch.testing.assert_close(want, other, atol=2 ** -7 * other.abs().max().item(), rtol=0)
    assert not torch.equal(want, other)


def _plan_bytes(B, H, Tq, Tk, D):
    """Workspace of the decode plan and of the shared form."""
    lib = _capi.load_library()
    q = torch.empty((B, Tq, H, D), dtype=torch.bfloat16, device=DEV)
    k = torch.empty((B, Tk, H, D), dtype=torch.bfloat16, device=DEV)
    n = torch.empty((B,), dtype=torch.int32, device=DEV)
    f = torch.empty((B,), dtype=torch.float32, device=DEV)
    pr = _capi._problem(q, k, k, f, None, f[0], n, n, False)
    return tuple(int(fn(ctypes.byref(pr))) for fn in (lib.sigattn_fwd_decode_workspace_bytes,
                                                      lib.sigattn_fwd_workspace_bytes))


@pytest.mark.parametrize("B,H,Tq,Tk,D", [(24, 32, 16, 581, 64), (48, 32, 1, 469, 64), (80, 16, 4, 378, 64),
                                         (64, 8, 2, 672, 64), (128, 4, 32, 2614, 64), (16, 32, 1, 299, 128)])
def test_short_caches_of_many_pairs_need_no_partials(B, H, Tq, Tk, D):
    """From 512 (batch, head) pairs on the shared form writes O itself; caches
    that are read in less time than the partials take keep it."""
    assert _plan_bytes(B, H, Tq, Tk, D) == (0, 0)


@pytest.mark.parametrize("B,H,Tq,Tk,D,chunks", [(65, 16, 1, 2100, 64, 3), (80, 16, 1, 8192, 128, 3),
                                                (72, 8, 2, 2600, 128, 5), (80, 4, 1, 6000, 64, 7),
                                                (256, 1, 1, 20000, 64, 7), (70, 8, 1, 3000, 64, 5)])
def test_batches_of_more_than_a_lane_each_take_an_odd_number_of_chunks(B, H, Tq, Tk, D, chunks):
    """An even number would put the last, short chunks of all sequences on the
    same XCDs."""
    assert _plan_bytes(B, H, Tq, Tk, D)[0] == chunks * B * H * Tq * D * 4


@pytest.mark.parametrize("B,H,Tq,Tk,D,packed,mod", [
    (65, 16, 1, 2100, 64, False, True),   # three chunks of one length for all
    (72, 8, 2, 2600, 128, True, False),   # five, packed rows
    (80, 4, 1, 6000, 64, False, False),
])
def test_decode_large_batches_match_the_general_path(B, H, Tq, Tk, D, packed, mod):
    test_decode_wave_per_chunk_matches_the_general_path(B, H, Tq, Tk, D, packed, mod)
