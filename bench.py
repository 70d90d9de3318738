#!/usr/bin/env python3
"""Benchmark: fused sigmoid attention fwd and fwd+bwd TFLOPS on one MI355X.

Default workload (the headline config): dense bf16
B=4 L=4096 H=16 D=128, causal, q/k/v/dO ~ N(0,1) from a seeded CPU generator,
scale = 1/sqrt(D), default bias -log(L).  One step = forward + backward through
the public API (`sigmoid_attention(...)` then `out.backward(dO)`), i.e. the fwd
kernel, the dQ kernel and the dK/dV kernel, with inputs resident in HBM.

FLOPs (algorithmic, extending the reference's benchmarks/benchmark_sigmoid.py
:252-260): per (b, h) and visible (query, key) pair, fwd = 4·D, bwd = 10·D,
fwd+bwd = 14·D; causal counts L²/2 pairs.  Recomputed or masked work is not
credited.

Padded workloads (--config c4 / c5, BASELINE.json configs[3] / [4]): seq_lens_q
= seq_lens_k ~ U[lo, Lmax] per batch element from the same seeded generator,
padding rows filled with N(0,1) noise; FLOPs count only valid (query, key)
pairs, and the same run times the dense kernels at the full shape to report
the padded path's TFLOPS per valid token as a fraction of dense.  The default
run (c3) measures c4 and c5 the same way after the headline and reports them
under "padded" in the same JSON line (--no-padded skips them), and the step
time of BASELINE.json configs[1] (dense fp16 B=2 L=1024 H=8 D=64, non-causal
c2 and causal c2c) under "small" (--no-small skips it).

Prints ONE JSON line on stdout; details go to stderr.
"""

from __future__ import annotations

import argparse
import itertools
import json
import math
import os
import re
import statistics
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT / "triton-sigmoid_amd"))
sys.path.insert(0, str(ROOT))

PEAK_BF16_TFLOPS = 2516.6  # MI355X dense fp16/bf16 MFMA: 256 CU x 2.4 GHz x 4096 FLOP/clk
PEAK_F32_TFLOPS = 157.3    # MI355X dense fp32 MFMA (v_mfma_f32_32x32x2_f32)
HBM_PEAK_TBPS = 8.0        # MI355X HBM3E
METRIC = "fwd & fwd+bwd TFLOPS + % of fp16 MFMA peak, dense/padded L=4096 D=128"

CONFIGS = {
    "c2": dict(B=2, L=1024, H=8, D=64, dtype="float16", causal=False),
    "c2c": dict(B=2, L=1024, H=8, D=64, dtype="float16", causal=True),
    "c3": dict(B=4, L=4096, H=16, D=128, dtype="bfloat16", causal=True),
    "c3nc": dict(B=4, L=4096, H=16, D=128, dtype="bfloat16", causal=False),
    # padded fp16, seq_lens ~ U[512, 2048], causal.
    "c4": dict(B=8, L=2048, H=8, D=64, dtype="float16", causal=True, padded=True, lo=512),
    # padded bf16 long context, seq_lens ~ U[1024, 8192],
    # non-causal, through torch.compile(sigmoid_attention_padded).
    "c5": dict(B=4, L=8192, H=12, D=64, dtype="bfloat16", causal=False, padded=True, lo=1024,
               compiled=True),
    # The other head dims and fp32 at the headline's shape (not BASELINE
    # configs; they time the D = 32 instances, head_dim 16 inside them, and
    # the fp32 MFMA kernels).
    "d32": dict(B=4, L=4096, H=16, D=32, dtype="bfloat16", causal=True),
    "d16": dict(B=4, L=4096, H=16, D=16, dtype="bfloat16", causal=True),
    "f32": dict(B=4, L=4096, H=16, D=128, dtype="float32", causal=True),
    "f32d64": dict(B=4, L=4096, H=16, D=64, dtype="float32", causal=True),
}


def peak_tflops(cfg) -> float:
    """Dense MFMA peak of the config's dtype."""
    return PEAK_F32_TFLOPS if cfg["dtype"] == "float32" else PEAK_BF16_TFLOPS


DTYPE_LABEL = {"bfloat16": "bf16", "float16": "fp16", "float32": "fp32"}


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def pairs(L: int, causal: bool) -> float:
    return L * L / 2.0 if causal else float(L * L)


def make_inputs(cfg, device):
    import torch
    dtype = getattr(torch, cfg["dtype"])
    g = torch.Generator().manual_seed(0)
    shape = (cfg["B"], cfg["L"], cfg["H"], cfg["D"])
    return [torch.randn(shape, generator=g, dtype=torch.float32).to(dtype).to(device) for _ in range(4)]


def make_seq_lens(cfg, device):
    """Per-batch valid lengths ~ U[lo, L] (int32) for the padded configs, else None."""
    import torch
    if not cfg.get("padded"):
        return None
    g = torch.Generator().manual_seed(1)
    return torch.randint(cfg["lo"], cfg["L"] + 1, (cfg["B"],), generator=g, dtype=torch.int32).to(device)


def valid_pairs(cfg, seq_lens) -> float:
    """(query, key) pairs the kernels must compute, summed over batch and heads."""
    if seq_lens is None:
        return pairs(cfg["L"], cfg["causal"]) * cfg["B"] * cfg["H"]
    return sum(pairs(int(n), cfg["causal"]) for n in seq_lens.tolist()) * cfg["H"]


def time_region(fn, iters: int, warmup: int):
    """Median per-call ms over `iters` calls bracketed by events on the current stream."""
    import torch
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    times = []
    for _ in range(iters):
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        fn()
        e.record()
        e.synchronize()
        times.append(s.elapsed_time(e))
    return statistics.median(times), times


def bench_like_reference(fn, warmup_ms: float = 100.0, rep_ms: float = 250.0, grad_to_none=()):
    """Median ms per call, timed the way the reference's sweep times it
    (benchmarks/benchmark_sigmoid.py:249, triton.testing.do_bench with
    warmup=100 ms, rep=250 ms, return_mode='median'): call counts from a
    5-call estimate, and before every timed call the gradients are reset and
    a 512 MiB buffer is zeroed so no operand is still in the L2 or the
    256 MB last-level cache; calls are queued back to back and the events
    read after one final synchronisation."""
    import torch
    flush = torch.empty(512 << 20, dtype=torch.uint8, device="cuda")
    fn()
    torch.cuda.synchronize()
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    for _ in range(5):
        flush.zero_()
        fn()
    e.record()
    torch.cuda.synchronize()
    est = s.elapsed_time(e) / 5
    n_warm, n_rep = max(1, int(warmup_ms / est)), max(1, int(rep_ms / est))
    for _ in range(n_warm):
        fn()
    starts = [torch.cuda.Event(enable_timing=True) for _ in range(n_rep)]
    ends = [torch.cuda.Event(enable_timing=True) for _ in range(n_rep)]
    for i in range(n_rep):
        for t in grad_to_none:
            t.grad = None
        flush.zero_()
        starts[i].record()
        fn()
        ends[i].record()
    torch.cuda.synchronize()
    del flush
    return statistics.median(a.elapsed_time(b) for a, b in zip(starts, ends))


KERNELS = ("fwd", "bwd_dq", "bwd_dkdv")


def kernel_times(cfg, q, k, v, do, iters: int, seq_lens=None, packed=False):
    """Average duration of each kernel, launched one at a time through the C ABI
    on torch's current stream and bracketed by HIP events on that stream, and
    of the whole backward ("bwd") as the public API launches it (on small
    dense grids at D <= 64, one launch running both kernels' items).
    packed=True runs the same sequences in the packed [rows, H, D] layout
    (cu_seqlens = [0, cumsum(seq_lens)]) instead of the padded one."""
    import ctypes
    import torch
    from triton_sigmoid import _capi
    lib = _capi.load_library()
    B, L, H, D = q.shape
    if seq_lens is None:
        bias = torch.full((B,), -math.log(L), dtype=torch.float32, device=q.device)
    else:
        bias = -torch.log(seq_lens.float())
    scale = torch.full((), 1.0 / math.sqrt(D), dtype=torch.float32, device=q.device)
    if packed:
        lens = seq_lens.tolist()
        q, k, v, do = (torch.cat([t[b, :n] for b, n in enumerate(lens)], 0) for t in (q, k, v, do))
        cu = torch.tensor([0] + list(itertools.accumulate(lens)), dtype=torch.int32, device=q.device)
        pr = _capi._problem(q, k, v, bias, None, scale, None, None, cfg["causal"],
                            packed=(cu, cu, max(lens), max(lens)))
    else:
        pr = _capi._problem(q, k, v, bias, None, scale, seq_lens, seq_lens, cfg["causal"])
    o, dq, dk, dv = (torch.empty_like(q) for _ in range(4))
    stream = torch.cuda.current_stream().cuda_stream
    # The forward the public API runs: with the workspace the library asks
    # for (the split-KV kernel at decode shapes, the range split of small
    # dense grids; none otherwise).
    fbytes = int(lib.sigattn_fwd_workspace_bytes(ctypes.byref(pr)))
    fws = torch.empty(max(fbytes, 16), dtype=torch.uint8, device=q.device)
    calls = {"fwd": lambda: lib.sigattn_fwd_ws(ctypes.byref(pr), o.data_ptr(), fws.data_ptr() if fbytes else None,
                                               fbytes, stream)}
    # The backward the public API runs: the range-split recompute kernels
    # where a small grid splits, else two-pass (dK/dV storing dS, then dQ
    # from dS) where _capi uses it, else the recompute kernels.
    sbytes = int(lib.sigattn_bwd_split_workspace_bytes(ctypes.byref(pr)))
    nbytes = 0
    if sbytes == 0 and D in _capi.TWO_PASS_HEAD_DIMS:
        nbytes = int(lib.sigattn_bwd_workspace_bytes(ctypes.byref(pr)))
    if 0 < nbytes <= _capi.bwd_workspace_limit():
        ws = torch.empty(nbytes, dtype=torch.uint8, device=q.device)
        calls["bwd_dkdv"] = lambda: lib.sigattn_bwd_dkdv_ws(ctypes.byref(pr), do.data_ptr(), dk.data_ptr(),
                                                            dv.data_ptr(), ws.data_ptr(), nbytes, stream)
        calls["bwd_dq"] = lambda: lib.sigattn_bwd_dq_ws(ctypes.byref(pr), dq.data_ptr(), ws.data_ptr(), nbytes,
                                                        stream)
        calls["bwd"] = lambda: lib.sigattn_bwd_ws(ctypes.byref(pr), do.data_ptr(), dq.data_ptr(), dk.data_ptr(),
                                                  dv.data_ptr(), ws.data_ptr(), nbytes, stream)
    else:
        # The recompute kernels, range-split where the public API splits them
        # (each half of sigattn_bwd_split on the whole workspace; the timing
        # includes its counter-clearing launch).
        nbytes = 0
        sws = torch.empty(max(sbytes, 16), dtype=torch.uint8, device=q.device)
        sptr = sws.data_ptr() if sbytes else None
        calls["bwd_dq"] = lambda: lib.sigattn_bwd_split(ctypes.byref(pr), do.data_ptr(), dq.data_ptr(), None, None,
                                                        sptr, sbytes, stream)
        calls["bwd_dkdv"] = lambda: lib.sigattn_bwd_split(ctypes.byref(pr), do.data_ptr(), None, dk.data_ptr(),
                                                          dv.data_ptr(), sptr, sbytes, stream)
        # The whole backward as the public API runs it: on small dense grids
        # at D <= 64 the library runs both kernels as one launch.
        calls["bwd"] = lambda: lib.sigattn_bwd_split(ctypes.byref(pr), do.data_ptr(), dq.data_ptr(), dk.data_ptr(),
                                                     dv.data_ptr(), sptr, sbytes, stream)
    # Median of five timed runs of `iters` launches each: the first kernel
    # timed after a long step loop, or early in a process, can read 5-20 %
    # slow on its own.
    out = {}
    for name, fn in calls.items():
        for _ in range(3):
            assert fn() == 0
        torch.cuda.synchronize()
        runs = []
        for _ in range(5):
            s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            s.record()
            for _ in range(iters):
                fn()
            e.record()
            e.synchronize()
            runs.append(s.elapsed_time(e) / iters)
        out[name] = statistics.median(runs)
        log(f"[bench] kernel {name}: runs {', '.join(f'{r:.4f}' for r in runs)} ms")
    if nbytes:
        log(f"[bench] two-pass backward: dS workspace {nbytes / 1e9:.3f} GB; dQ-from-dS reads it at "
            f"{nbytes / (out['bwd_dq'] * 1e-3) / 1e12:.2f} TB/s")
    return {n: out[n] for n in ("fwd", "bwd_dq", "bwd_dkdv", "bwd")}


def cpu_model() -> str:
    """The host CPU's model name (first 'model name' line of /proc/cpuinfo)."""
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(cfg, budget_s: float = 20.0):
    """fp32 eager forward + autograd backward of the oracle's restatement of the
    reference's sigmoid_attention_ref, on the host cores, over a bounded slice
    of the same workload: as many heads of one batch element, then as many
    batch elements (one at a time, so the L x L intermediates of only one are
    live), as fit about `budget_s` over the three timed runs."""
    import torch
    from oracle.eager import fwd_bwd_fp32
    torch.set_num_threads(os.cpu_count() or 1)
    L, D, causal = cfg["L"], cfg["D"], cfg["causal"]
    g = torch.Generator().manual_seed(0)
    heads = 1
    q, k, v, do = (torch.randn((1, L, heads, D), generator=g) for _ in range(4))
    fwd_bwd_fp32(q, k, v, do, causal=causal)  # warm-up (thread pool, allocator)
    t0 = time.perf_counter()
    fwd_bwd_fp32(q, k, v, do, causal=causal)
    one = time.perf_counter() - t0
    heads = max(1, min(cfg["H"], int(budget_s / 3.0 / max(one, 1e-3))))
    nb = max(1, min(cfg["B"], int(budget_s / 3.0 / max(one * heads, 1e-3))))
    batches = [[torch.randn((1, L, heads, D), generator=g) for _ in range(4)] for _ in range(nb)]
    runs = []
    for _ in range(3):
        t0 = time.perf_counter()
        for q, k, v, do in batches:
            fwd_bwd_fp32(q, k, v, do, causal=causal)
        runs.append(time.perf_counter() - t0)
    t = statistics.median(runs)
    flops = 14 * D * pairs(L, causal) * heads * nb
    return {
        "value": round(flops / t / 1e12, 4),
        "unit": "TFLOPS",
        "cores": torch.get_num_threads(),
        "host_cpu_count": os.cpu_count(),
        "cpu_model": cpu_model(),
        "kind": "port",
        "sample": f"fp32 eager fwd+bwd (oracle/eager.py) on B={nb} H={heads} (one batch element at a time) "
                  f"of the same L={L} D={D} causal={causal} workload, median of 3 after warm-up, "
                  f"{t:.2f} s each",
    }


def copy_calibration(nbytes: int = 1 << 30) -> None:
    """Runs one plain device copy of `nbytes` (read nbytes + write nbytes) so
    rocprofv3's FETCH_SIZE / WRITE_SIZE counters can be scaled to bytes."""
    import torch
    x = torch.ones(nbytes // 4, dtype=torch.float32, device="cuda")
    y = torch.empty_like(x)
    y.copy_(x)
    torch.cuda.synchronize()
    log(f"[bench] copy calibration: {nbytes} bytes read, {nbytes} bytes written")


def mfma_ceiling(n: int = 8192, iters: int = 20):
    """Practical MFMA rate of this GPU: hipBLASLt's bf16 GEMM (torch.matmul,
    n x n x n, fp32 accumulation) on N(0,1) operands and on all-zero
    operands.  The chip's power limit lowers the clock with data activity, so
    the random-operand rate is the ceiling a dense bf16 kernel can reach on
    this box; the zero-operand rate shows how far the spec clock is from it."""
    import torch
    g = torch.Generator().manual_seed(0)
    out = {}
    for name in ("random", "zero"):
        a = torch.randn((n, n), generator=g).to(torch.bfloat16).cuda()
        b = torch.randn((n, n), generator=g).to(torch.bfloat16).cuda()
        if name == "zero":
            a.zero_()
            b.zero_()
        ms, _ = time_region(lambda: torch.matmul(a, b), iters, 5)
        out[name] = {"ms": round(ms, 4), "tflops": round(2 * n ** 3 / ms / 1e9, 1)}
        del a, b
    return {"gemm": f"torch.matmul bf16 {n}x{n}x{n}", "peak_tflops": PEAK_BF16_TFLOPS,
            "random_operands": out["random"], "zero_operands": out["zero"],
            "random_frac_of_peak": round(out["random"]["tflops"] / PEAK_BF16_TFLOPS, 4)}


def kernel_source_digest() -> str:
    """sha256 over the device sources (csrc/*.hip, *.h) in name order: the
    identity of the kernels a traffic measurement belongs to."""
    import hashlib
    h = hashlib.sha256()
    for f in sorted((ROOT / "triton-sigmoid_amd" / "csrc").glob("*")):
        if f.suffix in (".hip", ".h"):
            h.update(f.name.encode())
            h.update(f.read_bytes())
    return h.hexdigest()[:16]


def _pmc_rows(path: str, counter: str) -> dict:
    """{kernel name: [value per dispatch]} of one counter from a rocprofv3
    --pmc csv (<dir>/<name>_counter_collection.csv)."""
    import csv
    out: dict = {}
    with open(path, newline="") as f:
        for row in csv.DictReader(f):
            if row.get("Counter_Name") != counter:
                continue
            out.setdefault(row["Kernel_Name"], []).append(float(row["Counter_Value"]))
    return out


def traffic_json(config: str, fetch_csv: str, write_csv: str, cal_fetch_csv: str, cal_write_csv: str) -> dict:
    """profiles/hbm_traffic.json from four rocprofv3 --pmc runs: FETCH_SIZE and
    WRITE_SIZE of `bench.py --config <config> --kernels dense`, and the same two
    counters of `bench.py --copy-calibration` (one 1 GiB device copy).  Bytes
    per launch = counter KiB x 1024 x (1 GiB / the copy's reading of it); the
    median over the dispatches of each kernel.  Records the kernel-source
    digest, so bench.py reports the traffic only for these kernels."""
    cfg = CONFIGS[config]
    one_gib = float(1 << 30)
    def copy_kib(path, counter):
        rows = [v for k, vs in _pmc_rows(path, counter).items() if "copyBuffer" in k for v in vs]
        if not rows:
            raise SystemExit(f"{path}: no {counter} row of the calibration copy (__amd_rocclr_copyBuffer)")
        return statistics.median(rows)

    fcal, wcal = copy_kib(cal_fetch_csv, "FETCH_SIZE"), copy_kib(cal_write_csv, "WRITE_SIZE")
    ffac, wfac = one_gib / (fcal * 1024), one_gib / (wcal * 1024)
    fetch, write = _pmc_rows(fetch_csv, "FETCH_SIZE"), _pmc_rows(write_csv, "WRITE_SIZE")
    B, L, H, D = cfg["B"], cfg["L"], cfg["H"], cfg["D"]
    tensor = B * L * H * D * 2
    nqb = -(-L // 32)
    ds_tiles = nqb * (nqb + 1) // 2 if cfg["causal"] else nqb * nqb
    ds_bytes = B * H * ds_tiles * 2048 if D == 128 else 0
    algo = {"fwd": 4 * tensor, "bwd_dkdv": 6 * tensor + ds_bytes,
            "bwd_dq": (2 * tensor + ds_bytes) if ds_bytes else 5 * tensor}
    # Without the two-pass backward's dS stream (written by dK/dV, read back
    # by dQ): only the operator's own tensors each kernel reads or writes.
    compulsory = {"fwd": 4 * tensor, "bwd_dkdv": 6 * tensor, "bwd_dq": 2 * tensor if ds_bytes else 5 * tensor}
    out = {"src_digest": kernel_source_digest(), "config": config,
           "calibration": {"copy_bytes": int(one_gib), "fetch_kib": fcal, "write_kib": wcal,
                           "fetch_factor": round(ffac, 4), "write_factor": round(wfac, 4)}}
    entry = {}
    for name in ("fwd", "bwd_dkdv", "bwd_dq"):
        fks = [(k, vs) for k, vs in fetch.items() if _kernel_matches(name, k)]
        wks = [(k, vs) for k, vs in write.items() if _kernel_matches(name, k)]
        if not fks or not wks:
            continue
        fk = statistics.median(v for _, vs in fks for v in vs)
        wk = statistics.median(v for _, vs in wks for v in vs)
        nbytes = fk * 1024 * ffac + wk * 1024 * wfac
        entry[name] = {"kernel": _kernel_base(fks[0][0]), "bytes_per_launch": int(nbytes),
                       "fetch_kib": round(fk, 1), "write_kib": round(wk, 1),
                       "algorithmic_bytes": int(algo[name]), "ratio": round(nbytes / algo[name], 3),
                       "compulsory_bytes": int(compulsory[name]),
                       "ratio_to_compulsory": round(nbytes / compulsory[name], 3)}
    out[config] = entry
    return out


# Function names of the kernels bench.py times under each name (rocprofv3
# reports some kernel names mangled, some demangled, so they are searched for).
_KERNEL_NAMES = {
    "fwd": ("fwd_mfma_kernel", "fwd_splitkv_kernel", "fwd_generic_kernel"),
    "bwd_dkdv": ("bwd_dkdv_pair_kernel", "bwd_dkdv_kernel", "dkdv_generic_kernel"),
    "bwd_dq": ("bwd_dq_ds_kernel", "bwd_dq_kernel", "dq_generic_kernel"),
}


def _kernel_base(kernel: str):
    """The library kernel function a profiled kernel name refers to
    ('_ZN7sigattn15fwd_mfma_kernelI...' or 'void sigattn::fwd_mfma_kernel<...>(...)'),
    or None for other kernels."""
    m = re.match(r"_ZN7sigattn(\d+)", kernel)
    if m:
        name = kernel[m.end():m.end() + int(m.group(1))]
    else:
        m = re.search(r"sigattn::(\w+)", kernel)
        name = m.group(1) if m else None
    return name if any(name in names for names in _KERNEL_NAMES.values()) else None


def _kernel_matches(name: str, kernel: str) -> bool:
    """Whether a profiled kernel is one bench.py times as `name`."""
    return _kernel_base(kernel) in _KERNEL_NAMES[name]


def load_traffic(kernel: str, config: str):
    """HBM bytes per launch of `kernel` measured with rocprofv3 --pmc FETCH_SIZE
    and WRITE_SIZE (scaled by the copy calibration), from
    profiles/hbm_traffic.json -- only when that file was measured on the
    kernels built from the current sources (its src_digest matches), else
    None."""
    path = ROOT / "profiles" / "hbm_traffic.json"
    if not path.exists():
        return None
    data = json.loads(path.read_text())
    if data.get("src_digest") != kernel_source_digest():
        log(f"[bench] profiles/hbm_traffic.json was measured on other kernel sources "
            f"({data.get('src_digest')} != {kernel_source_digest()}): traffic not reported")
        return None
    entry = data.get(config, {}).get(kernel)
    return None if entry is None else entry.get("bytes_per_launch")


# The reference's published chart (benchmarks/results/H100/tflops_comparison.png,
# read off the chart +-5 TFLOPS): bf16, non-causal, sigmoid_bias = 0,
# B = 16384/L, H = 2048/D; "bwd" = backward-only time credited with 2.5x the
# forward FLOPs (benchmarks/benchmark_sigmoid.py:193,202,232,252-260).
H100_CHART = {
    ("fwd", 64, 0): [347, 381, 395, 423, 437, 445], ("bwd", 64, 0): [270, 294, 293, 309, 316, 325],
    ("fwd", 128, 0): [371, 435, 466, 479, 486, 514], ("bwd", 128, 0): [278, 319, 334, 364, 367, 370],
    ("fwd", 64, 25): [300, 350, 377, 411, 416, 428], ("bwd", 64, 25): [231, 253, 274, 285, 262, 300],
    ("fwd", 128, 25): [312, 365, 380, 445, 428, 479], ("bwd", 128, 25): [244, 283, 304, 327, 326, 354],
}
SWEEP_L = [512, 1024, 2048, 4096, 8192, 16384]


def sweep():
    """The reference benchmark's grid (benchmarks/benchmark_sigmoid.py:193-260) on
    this GPU: D in {64, 128}, L in SWEEP_L with B = 16384/L and H = 2048/D, bf16,
    non-causal, sigmoid_bias = 0, padding 0 % (dense API), 25 % and 50 % (padded
    API, seq_lens ~ U[(1 - p) L, L] from a seeded CPU generator,
    benchmarks/benchmark_sigmoid.py:91-93); fwd and backward-only
    (o.backward(dO, retain_graph=True)), timed by bench_like_reference.
    The H100 chart has no 50 % panel, so those rows carry no comparison."""
    return [sweep_row(hd, pad, L) for hd in (64, 128) for pad in (0, 25, 50) for L in SWEEP_L]


def sweep_row(hd: int, pad: int, L: int) -> dict:
    """One point of the reference benchmark's grid (see sweep)."""
    import torch
    import triton_sigmoid as ts
    dev = torch.device("cuda", 0)
    li = SWEEP_L.index(L)
    B, H = 16384 // L, 2048 // hd
    g = torch.Generator().manual_seed(L * 1000 + hd * 10 + pad)
    q, k, v = (torch.randn((B, L, H, hd), generator=g).to(torch.bfloat16).to(dev).requires_grad_(True)
               for _ in range(3))
    if pad:
        lo = max(1, int(L * (1 - pad / 100)))
        sl = torch.randint(lo, L + 1, (B,), generator=g, dtype=torch.int32).to(dev)
        attn = lambda: ts.sigmoid_attention_padded(q, k, v, seq_lens_k=sl, seq_lens_q=sl,  # noqa: E731
                                                   is_causal=False, sigmoid_bias=0.0)
        flops_fwd = 4 * H * hd * float((sl.double() ** 2).sum().item())
    else:
        attn = lambda: ts.sigmoid_attention(q, k, v, sigmoid_bias=0.0)  # noqa: E731
        flops_fwd = 4.0 * B * H * L * L * hd
    ms_f = bench_like_reference(attn, grad_to_none=(q, k, v))
    o = attn()
    do = torch.randn(o.shape, generator=g).to(torch.bfloat16).to(dev)
    ms_b = bench_like_reference(lambda: o.backward(do, retain_graph=True), grad_to_none=(q, k, v))
    h100 = {m: H100_CHART[(m, hd, pad)][li] if (m, hd, pad) in H100_CHART else None for m in ("fwd", "bwd")}
    row = {"D": hd, "L": L, "B": B, "H": H, "padding_pct": pad,
           "fwd_ms": round(ms_f, 4), "bwd_ms": round(ms_b, 4),
           "fwd_tflops": round(flops_fwd / ms_f / 1e9, 1),
           "bwd_tflops": round(2.5 * flops_fwd / ms_b / 1e9, 1),
           "h100_fwd": h100["fwd"], "h100_bwd": h100["bwd"]}
    log(f"[sweep] D={hd} L={L} B={B} H={H} pad={pad}%: fwd {row['fwd_tflops']} TFLOPS "
        f"(H100 {row['h100_fwd']}), bwd {row['bwd_tflops']} (H100 {row['h100_bwd']})")
    del q, k, v, o, do
    torch.cuda.empty_cache()
    return row


# Points of the reference grid every default run reports (the "grid" block):
# D = 128, the chart's L = 4096 (dense and 25 % padding, the shape the
# reference's published utilisation is read at) and its long end, and D = 64
# at L = 4096.
GRID_DEFAULT = [(128, 0, 4096), (128, 25, 4096), (128, 0, 8192), (128, 0, 16384), (64, 0, 4096)]


# Decode shapes for the split-KV forward (bench.py --decode): bf16, Tq new
# queries per sequence against a KV cache, non-causal; "lo" = cache lengths
# ~ U[lo, Tk] per sequence (seeded), else every cache is Tk long.
DECODE_CONFIGS = [
    dict(B=16, H=32, D=128, Tq=1, Tk=8192),
    dict(B=16, H=32, D=128, Tq=1, Tk=8192, lo=1024),
    dict(B=1, H=32, D=128, Tq=1, Tk=131072),
    dict(B=32, H=32, D=64, Tq=4, Tk=4096),
    dict(B=8, H=16, D=128, Tq=32, Tk=16384),
]


def decode_bench(iters: int = 20):
    """Split-KV forward at decode shapes through the C ABI: average kernel time
    (the chunk kernel and the partial sum) by the plan the public APIs launch
    (sigattn_fwd_decode), by sigattn_fwd_ws with the workspace it asks for, and
    with none (one chunk per (batch, head)), on torch's current stream
    between HIP events.  The kernel is HBM-bound: its algorithmic traffic is
    K and V of the valid cache (2 * D * 2 bytes per key, batch and head) plus
    Q and O."""
    import ctypes
    import torch
    from triton_sigmoid import _capi
    lib = _capi.load_library()
    dev = torch.device("cuda", 0)
    rows = []
    for cfg in DECODE_CONFIGS:
        B, H, D, Tq, Tk = cfg["B"], cfg["H"], cfg["D"], cfg["Tq"], cfg["Tk"]
        g = torch.Generator(device=dev).manual_seed(B * Tk + D)
        q = torch.randn((B, Tq, H, D), generator=g, device=dev, dtype=torch.bfloat16)
        k = torch.randn((B, Tk, H, D), generator=g, device=dev, dtype=torch.bfloat16)
        v = torch.randn((B, Tk, H, D), generator=g, device=dev, dtype=torch.bfloat16)
        gc = torch.Generator().manual_seed(Tk + B)
        lens = (torch.randint(cfg["lo"], Tk + 1, (B,), generator=gc, dtype=torch.int32) if "lo" in cfg
                else torch.full((B,), Tk, dtype=torch.int32))
        sk = lens.to(dev)
        sq = torch.full((B,), Tq, dtype=torch.int32, device=dev)
        bias = -torch.log(sk.float())
        scale = torch.full((), 1.0 / math.sqrt(D), dtype=torch.float32, device=dev)
        pr = _capi._problem(q, k, v, bias, None, scale, sq, sk, False)
        out = torch.empty_like(q)
        nbytes = int(lib.sigattn_fwd_workspace_bytes(ctypes.byref(pr)))
        dbytes = int(lib.sigattn_fwd_decode_workspace_bytes(ctypes.byref(pr)))
        ws = torch.empty(max(nbytes, dbytes, 16), dtype=torch.uint8, device=dev)
        stream = torch.cuda.current_stream().cuda_stream
        kv_keys = int(lens.sum())
        traffic = 2 * D * 2 * kv_keys * H + 2 * B * Tq * H * D * 2
        flops = 4 * D * Tq * kv_keys * H
        row = dict(cfg, workspace_bytes=nbytes, decode_workspace_bytes=dbytes)
        for name, fwd, wbytes in (("decode", lib.sigattn_fwd_decode, dbytes), ("split", lib.sigattn_fwd_ws, nbytes),
                                  ("one_chunk", lib.sigattn_fwd_ws, 0)):
            wptr = ws.data_ptr() if wbytes else None
            call = lambda: fwd(ctypes.byref(pr), out.data_ptr(), wptr, wbytes, stream)
            for _ in range(3):
                assert call() == 0
            torch.cuda.synchronize()
            s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            s.record()
            for _ in range(iters):
                call()
            e.record()
            e.synchronize()
            ms = s.elapsed_time(e) / iters
            row[name] = dict(ms=round(ms, 4), gbps=round(traffic / ms / 1e6, 1),
                             hbm_frac=round(traffic / ms / 1e6 / (HBM_PEAK_TBPS * 1e3), 4),
                             tflops=round(flops / ms / 1e9, 1))
        rows.append(row)
        log(f"[decode] {cfg}: decode {row['decode']} | split {row['split']} | one chunk {row['one_chunk']}")
        del q, k, v, out, ws
        torch.cuda.empty_cache()
    return rows


def workload_name(name, cfg) -> str:
    shape = f"B={cfg['B']} L={cfg['L']} H={cfg['H']} D={cfg['D']} {cfg['dtype']} causal={cfg['causal']}"
    if cfg.get("padded"):
        how = "torch.compile(sigmoid_attention_padded)" if cfg.get("compiled") else "sigmoid_attention_padded"
        tag = {"c4": " (BASELINE.json configs[3])", "c5": " (BASELINE.json configs[4])"}.get(name, "")
        return f"padded sigmoid attention fwd+bwd via {how}, {shape}, seq_lens ~ U[{cfg['lo']}, {cfg['L']}]{tag}"
    tag = {"c3": " (BASELINE.json configs[2])", "c2": " (BASELINE.json configs[1])",
           "c2c": " (BASELINE.json configs[1])"}.get(name, "")
    return f"dense sigmoid attention fwd+bwd, {shape}{tag}"


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    # The warm-up covers the GPU's power-management settling: at c3 the step
    # time swings from 1.18 to 1.5 ms over the first steps of a process and
    # settles at its steady value after about 40 (measured over 400 steps:
    # steps 20-39 average 1.230 ms, every later block of 20 1.203-1.212 ms).
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=50)
    ap.add_argument("--config", default="c3", choices=sorted(CONFIGS))
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-padded", action="store_true",
                    help="with the default c3 config: skip the c4 / c5 padded-vs-dense measurements")
    ap.add_argument("--no-small", action="store_true",
                    help="with the default c3 config: skip the c2 / c2c small-problem step measurements")
    ap.add_argument("--no-grid", action="store_true",
                    help="skip the points of the reference benchmark's grid that ride along with c3")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only run a 1 GiB device copy (for rocprofv3 counter scaling)")
    ap.add_argument("--sweep", action="store_true",
                    help="the reference benchmark's L/D/padding grid, beside its published H100 chart")
    ap.add_argument("--sweep-point", nargs=3, type=int, metavar=("D", "PAD_PCT", "L"),
                    help="one point of that grid")
    ap.add_argument("--decode", action="store_true",
                    help="split-KV forward at decode shapes (HBM GB/s)")
    ap.add_argument("--ceiling", action="store_true",
                    help="hipBLASLt bf16 GEMM TFLOPS on random and on zero operands (the box's practical MFMA rate)")
    ap.add_argument("--kernels", choices=("dense", "padded", "packed"),
                    help="only time the config's kernels through the C ABI in this layout (a program to "
                         "profile: no API steps, no CPU baseline)")
    ap.add_argument("--traffic-json", nargs=4, metavar=("FETCH_CSV", "WRITE_CSV", "CAL_FETCH_CSV", "CAL_WRITE_CSV"),
                    help="write profiles/hbm_traffic.json for --config from rocprofv3 --pmc FETCH_SIZE / "
                         "WRITE_SIZE csvs of `--kernels dense` and of `--copy-calibration`")
    args = ap.parse_args()
    if args.traffic_json:
        data = traffic_json(args.config, *args.traffic_json)
        path = ROOT / "profiles" / "hbm_traffic.json"
        path.write_text(json.dumps(data, indent=1) + "\n")
        print(json.dumps(data), flush=True)
        return
    if args.ceiling:
        print(json.dumps({"metric": "practical MFMA rate (bf16 GEMM)", "unit": "TFLOPS", **mfma_ceiling()}),
              flush=True)
        return
    if args.copy_calibration:
        copy_calibration()
        return
    if args.decode:
        rows = decode_bench()
        print(json.dumps({"metric": "split-KV decode forward: HBM GB/s of K, V, Q, O", "unit": "GB/s",
                          "peak_tbps": HBM_PEAK_TBPS, "rows": rows}), flush=True)
        return
    if args.sweep_point:
        hd, pad, L = args.sweep_point
        if hd not in (64, 128) or pad not in (0, 25, 50) or L not in SWEEP_L:
            sys.exit(f"--sweep-point: D in (64, 128), PAD_PCT in (0, 25, 50), L in {SWEEP_L}")
    if args.sweep or args.sweep_point:
        rows = sweep() if args.sweep else [sweep_row(*args.sweep_point)]
        print(json.dumps({"metric": "reference benchmark grid: fwd and bwd-only TFLOPS, bf16 non-causal",
                          "unit": "TFLOPS", "rows": rows}), flush=True)
        return

    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) > 1:
        print("bench.py measures one GPU only: this build has no multi-GPU path "
              "(every (batch, head) pair is independent, so the work would shard across GPUs by heads). "
              "Run with --gpus 1.", file=sys.stderr)
        sys.exit(2)

    import torch

    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    if args.kernels:
        cfg = CONFIGS[args.config]
        q, k, v, do = make_inputs(cfg, dev)
        sl = make_seq_lens(cfg, dev) if args.kernels != "dense" else None
        if args.kernels != "dense" and sl is None:
            sys.exit(f"--kernels {args.kernels} needs a padded config")
        kt = kernel_times(cfg, q, k, v, do, iters=args.steps, seq_lens=sl, packed=args.kernels == "packed")
        print(json.dumps({"config": args.config, "layout": args.kernels, "kernel_ms": kt}), flush=True)
        return
    res = measure_config(args.config, args.steps, args.warmup)
    B, L, H, D, causal = (res["cfg"][n] for n in ("B", "L", "H", "D", "causal"))
    kt, P, dominant = res["kernel_ms"], res["pairs"], res["dominant"]
    credit = {"fwd": 4 * D * P, "bwd_dq": 2 * D * P, "bwd_dkdv": 8 * D * P}
    achieved = credit[dominant] / (kt[dominant] * 1e-3) / 1e12
    bwd_ms = kt["bwd"]  # the backward as the public API launches it
    fb_tflops = res["fb_tflops"]

    # The padded configs ride along with the headline run, so their padded /
    # dense ratio (the north-star target, >= 0.85) is measured by every
    # default run, c5 through torch.compile.
    padded = {}
    if res.get("padded") is not None:
        padded[args.config] = res["padded"]
    elif args.config == "c3" and not args.no_padded:
        for name in ("c4", "c5"):
            torch.cuda.empty_cache()
            r = measure_config(name, args.steps, args.warmup)
            padded[name] = dict(r["padded"], step_ms=round(r["ms_step"], 4),
                                step_tflops_valid_pairs=round(r["fb_tflops"], 2),
                                step_pct_of_peak=round(100 * r["fb_tflops"] / PEAK_BF16_TFLOPS, 2),
                                workload=workload_name(name, CONFIGS[name]))

    # BASELINE configs[1] (dense fp16 B=2 L=1024 H=8 D=64, non-causal and
    # causal) rides along too: a small problem whose step time is set by the
    # host path and the grid's fill of the GPU as much as by the kernels.
    small = {}
    if args.config == "c3" and not args.no_small:
        for name in ("c2", "c2c"):
            torch.cuda.empty_cache()
            r = measure_config(name, max(args.steps, 200), args.warmup)
            small[name] = dict(step_ms=round(r["ms_step"], 4), step_tflops=round(r["fb_tflops"], 2),
                               kernel_ms={n: round(t, 4) for n, t in r["kernel_ms"].items()},
                               workload=workload_name(name, CONFIGS[name]))

    # A few points of the reference benchmark's own grid (fwd and backward-only
    # TFLOPS, bf16 non-causal, sigmoid_bias = 0, timed as the reference times
    # them) beside the H100 chart's values: the long end the sweep reaches.
    grid = []
    if args.config == "c3" and not args.no_grid:
        for hd, pad, L in GRID_DEFAULT:
            torch.cuda.empty_cache()
            grid.append(sweep_row(hd, pad, L))

    cpu = None
    if not args.no_cpu_baseline:
        cpu = cpu_baseline(res["cfg"])
        log(f"[bench] cpu baseline {cpu}")

    cfg = res["cfg"]
    line = {
        "metric": METRIC,
        "value": round(fb_tflops, 2),
        "unit": "TFLOPS",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(res["ms_step"], 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": DTYPE_LABEL[cfg["dtype"]],
        "data": "synthetic: q,k,v,dO ~ N(0,1) from torch.Generator seed 0",
        "config": {
            "workload": workload_name(args.config, cfg),
            "batch": B, "seq_len": L, "heads": H, "head_dim": D, "causal": causal,
        },
        "pct_of_peak": round(100 * fb_tflops / peak_tflops(cfg), 2),
        "fwd_tflops": round(res["fwd_tflops"], 2),
        "fwd_pct_of_peak": round(100 * res["fwd_tflops"] / peak_tflops(cfg), 2),
        "bwd_only_tflops": round(10 * D * P / (bwd_ms * 1e-3) / 1e12, 2),
        "kernel_ms": {n: round(t, 4) for n, t in kt.items()},
        "roofline": {
            "kernel": dominant,
            "bound": "mfma",
            "achieved": round(achieved, 2),
            "peak": peak_tflops(cfg),
            "unit": "TFLOP/s",
            "frac": round(achieved / peak_tflops(cfg), 4),
            "traffic": load_traffic(dominant, args.config),
        },
        "cpu_baseline": cpu,
    }
    if padded:
        line["padded"] = padded
    if small:
        line["small"] = small
    if grid:
        line["grid"] = grid
    print(json.dumps(line), flush=True)


def measure_config(name: str, steps: int, warmup: int) -> dict:
    """Times one config: `steps` fwd+bwd steps through the public API (after
    `warmup` untimed ones), the forward alone, and each kernel through the C
    ABI; padded configs add the padded / dense ratios (padded_block)."""
    import torch
    import triton_sigmoid as ts

    cfg = CONFIGS[name]
    dev = torch.device("cuda", 0)
    q, k, v, do = make_inputs(cfg, dev)
    for t in (q, k, v):
        t.requires_grad_(True)
    B, L, H, D, causal = cfg["B"], cfg["L"], cfg["H"], cfg["D"], cfg["causal"]
    sl = make_seq_lens(cfg, dev)
    P = valid_pairs(cfg, sl)
    fwd_flops, fb_flops = 4 * D * P, 14 * D * P

    if sl is None:
        attn = lambda: ts.sigmoid_attention(q, k, v, is_causal=causal)
    else:
        padded = ts.sigmoid_attention_padded
        if cfg.get("compiled"):
            padded = torch.compile(ts.sigmoid_attention_padded, fullgraph=True)
        attn = lambda: padded(q, k, v, seq_lens_k=sl, seq_lens_q=sl, is_causal=causal)

    def fwd():
        with torch.no_grad():
            attn()

    def step():
        q.grad = k.grad = v.grad = None
        o = attn()
        o.backward(do)

    # The per-kernel and forward-only timings run first.  Besides their own
    # figures they take the GPU through its power-management settling (a
    # process's first steps run at the cold clock, the next ones throttled),
    # so the K timed steps below measure the steady state a training loop
    # runs at rather than the first tens of milliseconds of a process.
    kt = kernel_times(cfg, q.detach(), k.detach(), v.detach(), do, iters=max(10, steps), seq_lens=sl)
    fwd_ms, _ = time_region(fwd, iters=max(10, steps), warmup=3)
    fwd_tflops = fwd_flops / (fwd_ms * 1e-3) / 1e12

    # Whole-job timing of K fwd+bwd steps after W untimed ones.
    for _ in range(warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        step()
    torch.cuda.synchronize()
    ms_step = (time.perf_counter() - t0) * 1e3 / steps
    fb_tflops = fb_flops / (ms_step * 1e-3) / 1e12
    dominant = max(KERNELS, key=kt.get)
    log(f"[bench] config={name} {cfg}")
    log(f"[bench] step {ms_step:.3f} ms -> fwd+bwd {fb_tflops:.1f} TFLOPS ({100 * fb_tflops / peak_tflops(cfg):.1f}% peak)")
    log(f"[bench] fwd {fwd_ms:.3f} ms -> {fwd_tflops:.1f} TFLOPS; kernels (ms): "
        + ", ".join(f"{n}={t:.3f}" for n, t in kt.items()))
    out = dict(cfg=cfg, pairs=P, ms_step=ms_step, fb_tflops=fb_tflops, fwd_tflops=fwd_tflops, kernel_ms=kt,
               dominant=dominant, padded=None)
    if sl is not None:
        out["padded"] = padded_block(cfg, q.detach(), k.detach(), v.detach(), do, sl, kt, P, max(10, steps))
    del q, k, v, do
    return out


def padded_block(cfg, q, k, v, do, sl, kt, P, iters) -> dict:
    """The padded path's TFLOPS per valid token as a fraction of dense: the
    dense kernels at the full shape and the padded kernels, timed in the same
    run through the C ABI, plus the packed layout (the same sequences as
    [rows, H, D] with cu_seqlens).  padded_vs_dense times the forward and the
    whole backward as the library launches them for the public API (for large
    ragged non-causal problems its two kernels run concurrently);
    kernel_sum_padded_vs_dense the three kernels launched one at a time."""
    B, L, H, D, causal = cfg["B"], cfg["L"], cfg["H"], cfg["D"], cfg["causal"]
    kd = kernel_times(cfg, q, k, v, do, iters=iters)
    Pd = pairs(L, causal) * B * H
    kp = kernel_times(cfg, q, k, v, do, iters=iters, seq_lens=sl, packed=True)
    log("[bench] packed layout kernels (ms): " + ", ".join(f"{n}={t:.3f}" for n, t in kp.items()))

    def tflops(pairs_, kt_, parts):
        return 14 * D * pairs_ / (sum(kt_[n] for n in parts) * 1e-3) / 1e12

    launched, kernels = ("fwd", "bwd"), KERNELS
    dense_tf, padded_tf, packed_tf = tflops(Pd, kd, launched), tflops(P, kt, launched), tflops(P, kp, launched)
    dense_ks, padded_ks, packed_ks = tflops(Pd, kd, kernels), tflops(P, kt, kernels), tflops(P, kp, kernels)
    credit = {"fwd": 4 * D * P, "bwd_dq": 2 * D * P, "bwd_dkdv": 8 * D * P}
    credit_d = {"fwd": 4 * D * Pd, "bwd_dq": 2 * D * Pd, "bwd_dkdv": 8 * D * Pd}
    info = {
        "seq_lens": sl.tolist(),
        "valid_pair_fraction": round(P / Pd, 4),
        "padded_vs_dense": round(padded_tf / dense_tf, 4),
        "packed_vs_dense": round(packed_tf / dense_tf, 4),
        "kernel_sum_padded_vs_dense": round(padded_ks / dense_ks, 4),
        "kernel_sum_packed_vs_dense": round(packed_ks / dense_ks, 4),
        "per_kernel_padded_vs_dense": {
            n: round((credit[n] / kt[n]) / (credit_d[n] / kd[n]), 4) for n in ("fwd", "bwd_dq", "bwd_dkdv")},
        "padded_kernel_ms": {n: round(t, 4) for n, t in kt.items()},
        "dense_kernel_ms": {n: round(t, 4) for n, t in kd.items()},
        "packed_kernel_ms": {n: round(t, 4) for n, t in kp.items()},
        "padded_kernel_tflops": round(padded_tf, 2),
        "padded_kernel_pct_of_peak": round(100 * padded_tf / PEAK_BF16_TFLOPS, 2),
        "dense_kernel_tflops": round(dense_tf, 2),
        "packed_kernel_tflops": round(packed_tf, 2),
        "note": "padded_vs_dense: fwd + the whole backward as the library launches it, through the C ABI; "
                "kernel_sum_*: fwd + dQ + dK/dV launched one at a time; padded and packed (the same "
                "sequences as [rows, H, D] with cu_seqlens) count valid pairs only",
    }
    log(f"[bench] padded {info}")
    return info


if __name__ == "__main__":
    main()
