"""Pairs that fail at many elements (what dense items leave, and where items go back
and forth between the dense form and the queue) against the oracle (needs an
MI355X): shares of mismatches among identical pairs and among noise, zero and
partly zero tolerances, identical infinities and NaN, sections of different kinds
within one pair, fp32, bf16 and fp16, single and batched, and the tolerant
policy's near-zero diagnostics.  Also order statistics among the captured values
just below a capture threshold."""

import numpy as np
import pytest
import torch

from golden_io import same_value
from kernelverse_amd import verdict
from kernelverse_amd.correctness_policy import resolve_correctness_policy
from oracle import torch_verdict as tv
from parity_util import meta_problems, record_vs_oracle
from test_gpu_input_select import _fp32_noise, _pivot_positions

pytestmark = pytest.mark.gpu

DEV = "cuda"
DTYPES = [torch.float32, torch.bfloat16, torch.float16]
NAMES = {torch.float32: "FP32", torch.bfloat16: "BF16", torch.float16: "FP16"}
DEFAULT = {torch.float32: (1e-5, 1e-5), torch.bfloat16: (1.6e-2, 1e-2), torch.float16: (1e-3, 1e-3)}
NOISE = {torch.float32: 2e-7, torch.bfloat16: 4e-3, torch.float16: 5e-4}


def _pair(kind, n, dtype, seed):
    """(generated, reference, (rtol, atol))"""
    gen = torch.Generator().manual_seed(seed)
    x, u, e = torch.randn(n, generator=gen), torch.rand(n, generator=gen), torch.randn(n, generator=gen)
    r = x.to(dtype)
    near = (x * (1 + NOISE[dtype] * e)).to(dtype)
    far = (x + 0.2 * torch.sign(e) * (1 + u) + 0.1 * x * e).to(dtype)
    tol = DEFAULT[dtype]
    if kind.startswith("miss"):
        return torch.where(u < int(kind[4:]) / 100, far, r), r, tol
    if kind.startswith("noisymiss"):
        return torch.where(u < int(kind[9:]) / 100, far, near), r, tol
    if kind.startswith("zerotol"):
        return torch.where(u < int(kind[7:]) / 100, near, r), r, (0.0, 0.0)
    if kind == "atol0":
        zero = torch.zeros((), dtype=dtype)
        sign = torch.where(e < 0, -zero, zero)
        return torch.where(u < 0.5, sign, near), torch.where(u < 0.5, zero, r), (tol[0], 0.0)
    if kind in ("mask", "noisymask"):
        inf = torch.tensor(float("-inf"), dtype=dtype)
        return torch.where(u < 0.5, inf, near if kind == "noisymask" else r), torch.where(u < 0.5, inf, r), tol
    if kind == "nan":
        nan = torch.tensor(float("nan"), dtype=dtype)
        return torch.where(u < 0.4, nan, near), torch.where((u > 0.1) & (u < 0.5), nan, r), tol
    if kind == "equalsum":
        # mismatches of one abs_diff and one rel_diff: every tie of both
        r = torch.where(u < 0.5, 1.0, 2.0).to(dtype)
        return torch.where(u < 0.9, r * 2, r), r, tol
    # sections of a few items each, in turn: noise, all beyond the tolerance, identical, masked, half beyond
    section = (torch.arange(n) // 5000) % 5
    inf = torch.tensor(float("inf"), dtype=dtype)
    g = torch.where(section == 0, near, torch.where(section == 1, far, r))
    g = torch.where((section == 4) & (u < 0.5), far, g)
    masked = section == 3
    return torch.where(masked, inf, g), torch.where(masked, inf, r), tol


KINDS = ["miss25", "miss50", "miss100", "noisymiss10", "noisymiss50", "zerotol25", "zerotol50", "zerotol100", "atol0", "mask",
         "noisymask", "nan", "equalsum", "sections"]


def _problems(rec, g, r, tol):
    probs = record_vs_oracle(rec, g, r, tol)
    mm = tv.mismatch_stats(g, r, tol)
    for k in ("mismatch_count", "first_mismatch_index"):
        if rec[k] != mm[k]:
            probs.append(f"{k}: device {rec[k]} != oracle {mm[k]}")
    for k in ("mismatch_max_abs", "mismatch_max_rel"):
        if mm["mismatch_count"] and not same_value(float(rec[k]), mm[k]):
            probs.append(f"{k}: device {rec[k]!r} != oracle {mm[k]!r}")
    return probs


def _tol(dtype, tol):
    return {NAMES[dtype]: {"rtol": tol[0], "atol": tol[1]}}


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("kind", KINDS)
def test_single(kind, dtype):
    # one wave's items, partial items, and several items per wave
    for n in (1024, 5_003, 1_000_003, 7_340_033):
        if n > 2_000_000 and kind not in ("noisymiss10", "sections", "noisymask"):
            continue
        g, r, tol = _pair(kind, n, dtype, n + len(kind))
        print("dense rest", kind, dtype, n, flush=True)
        rec = verdict.verdict_record(g.to(DEV), r.to(DEV), _tol(dtype, tol))
        probs = _problems(rec, g, r, _tol(dtype, tol))
        assert not probs, probs


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
def test_batch(dtype):
    """Enough large pairs that their p99 comes from captured values, small ones between them."""
    jobs = []
    for i in range(300):
        n = 8_300 + 997 * (i % 40) if i % 4 else 300 + 37 * i
        jobs.append(_pair(KINDS[i % len(KINDS)], n, dtype, i))
    print("dense rest batch", dtype, len(jobs), flush=True)
    recs = verdict.verdict_records([(g.to(DEV), r.to(DEV), _tol(dtype, t)) for g, r, t in jobs])
    for i, ((g, r, t), rec) in enumerate(zip(jobs, recs)):
        probs = _problems(rec, g, r, _tol(dtype, t))
        a, b, _, _ = tv.mismatch_parts(g, r, _tol(dtype, t))
        for k, vals in (("p99_abs", a), ("p99_rel", b)):
            if not same_value(float(rec[k]), float(tv.p99_meta(vals))):
                probs.append(f"{k}: device {rec[k]!r} != oracle {tv.p99_meta(vals)!r}")
        assert not probs, (KINDS[i % len(KINDS)], g.numel(), probs)


@pytest.mark.parametrize("dtype", DTYPES[1:], ids=str)
@pytest.mark.parametrize("kind", KINDS)
def test_tolerant_meta(kind, dtype):
    policy = resolve_correctness_policy({"category": "gemm", "op_name": "x"})
    g, r, tol = _pair(kind, 600_001, dtype, 5)
    print("dense rest tolerant", kind, dtype, flush=True)
    got = verdict._compare_tensors(g.to(DEV), r.to(DEV), "output", _tol(dtype, tol), policy)
    want = tv.compare_tensors(g, r, "output", _tol(dtype, tol), policy)
    assert got[0] == want[0]
    assert not meta_problems(got[2], want[2], g, r)


def test_order_statistic_below_the_rel_threshold():
    """Dense fp32 items capture rel_diff a few roundings below the pivot threshold; a p99 among those captured
    values falls back.  The pivot runs hold the rel_diff v = 0.5 (abs_diff 0.5), the other elements v - 2^-23 to
    v - 4 * 2^-23 (abs_diff near 2, captured); and rel_diffs below 2^-80, where every nonzero value is captured."""
    rng = np.random.default_rng(12)
    n = 600_000  # (1 % of them more than the pivot's 4,096)
    special = []
    for steps in (1, 4):
        r = np.full(n, 4.0, np.float32)
        k = rng.integers(1, steps + 1, n).astype(np.float32)
        g = r + (np.float32(2.0) - k * np.float32(2.0 ** -21))
        pos = _pivot_positions(n)
        r[pos], g[pos] = 1.0, 1.5
        special.append((torch.from_numpy(g), torch.from_numpy(r)))
    r = (1e-37 * (1 + rng.random(n))).astype(np.float32)
    g = (r.view(np.int32) + rng.integers(1, 5_000, n).astype(np.int32)).view(np.float32)
    special.append((torch.from_numpy(g), torch.from_numpy(r)))
    pairs = special + [_fp32_noise(int(rng.integers(8_300, 12_000)), rng) for _ in range(270)]
    print("below the threshold", len(pairs), flush=True)
    recs = verdict.verdict_records([(g.to(DEV), r.to(DEV)) for g, r in pairs])
    for (g, r), rec in zip(special, recs):
        a, b, _, _ = tv.mismatch_parts(g, r)
        assert same_value(float(rec["p99_abs"]), float(tv.p99_meta(a)))
        assert same_value(float(rec["p99_rel"]), float(tv.p99_meta(b)))
        assert not record_vs_oracle(rec, g, r)
