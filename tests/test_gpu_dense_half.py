"""16-bit pairs that differ at many elements (the dense items of the main pass)
against the oracle (needs an MI355X): fp16 and bf16, distances in every ULP
bucket, sign changes (signed zeros among them), NaN and Inf on either side,
ties of the largest rel_diff and abs_diff, mismatches, sizes that leave partial
items and vectors, and the near-zero diagnostics of the tolerant policy.

Records are exact except the fp64 sums (parity_util's bounds)."""

import pytest
import torch

from kernelverse_amd import verdict
from kernelverse_amd.correctness_policy import resolve_correctness_policy
from oracle import torch_verdict as tv
from parity_util import meta_problems, record_vs_oracle

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = {"BF16": {"rtol": 1.6e-2, "atol": 1e-2}, "FP16": {"rtol": 1e-3, "atol": 1e-3}}
# items of 2048 elements: one item, partial vectors, partial items, several items per wave, a strided sample
SIZES = [2048, 2049, 40_003, 600_000, 7_340_033]


def _steps(r, gen, frac, top):
    """r with `frac` of its codes moved by 1..top steps of magnitude (kept finite), either way."""
    codes = r.view(torch.int16)
    mag = codes & 0x7FFF
    step = torch.randint(1, top + 1, r.shape, generator=gen).to(torch.int16)
    step = torch.where(torch.rand(r.shape, generator=gen) < frac, step, torch.zeros_like(step))
    down = (torch.rand(r.shape, generator=gen) < 0.5) & (mag >= step)
    limit = 0x7F80 if r.dtype == torch.bfloat16 else 0x7C00
    up_ok = mag.int() + step < limit
    moved = torch.where(down, codes - step, torch.where(up_ok, codes + step, codes))
    return moved.view(r.dtype)


def _pair(kind, n, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    r = (torch.randn(n, generator=gen) * 2).to(dtype)
    if kind == "ulp1":
        return _steps(r, gen, 0.5, 1), r
    if kind == "wide":
        return _steps(r, gen, 0.9, 3000), r
    if kind == "signs":
        g = _steps(r, gen, 0.6, 3)
        flip = torch.rand(n, generator=gen) < 0.05
        g = torch.where(flip, -g, g)
        zero = torch.rand(n, generator=gen) < 0.05
        r = torch.where(zero, torch.zeros_like(r), r)
        g = torch.where(zero, torch.where(torch.rand(n, generator=gen) < 0.5, -torch.zeros_like(g), torch.zeros_like(g)), g)
        tiny = torch.rand(n, generator=gen) < 0.02
        r = torch.where(tiny, (r.float() * 1e-7).to(dtype), r)
        return torch.where(tiny, -r, g), r
    if kind == "nonfinite":
        g = _steps(r, gen, 0.5, 2)
        for side, share in ((g, 0.002), (r, 0.002)):
            for v in (float("nan"), float("inf"), float("-inf")):
                side[torch.rand(n, generator=gen) < share] = v
        same = torch.rand(n, generator=gen) < 0.002
        g[same] = r[same] = float("nan")
        return g, r
    if kind == "ties":
        # every pair one of few values: the largest abs_diff and rel_diff repeat
        r = torch.tensor([1.0, 2.0, -4.0, 0.5])[torch.randint(0, 4, (n,), generator=gen)].to(dtype)
        return _steps(r, gen, 0.7, 1), r
    # far: half of the pairs beyond the tolerance
    return (r.float() * (1 + 0.2 * (torch.rand(n, generator=gen) < 0.5))).to(dtype), r


KINDS = ["ulp1", "wide", "signs", "nonfinite", "ties", "far"]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("kind", KINDS)
def test_dense_half_record(kind, dtype):
    for n in SIZES if kind in ("ulp1", "nonfinite") else SIZES[2:4]:
        print("dense half", kind, dtype, n, flush=True)
        g, r = _pair(kind, n, dtype, n + len(kind))
        rec = verdict.verdict_record(g.to(DEV), r.to(DEV), TOL)
        assert not record_vs_oracle(rec, g, r, TOL)


@pytest.mark.parametrize("kind", KINDS)
def test_dense_half_tolerant_meta(kind):
    policy = resolve_correctness_policy({"category": "gemm", "op_name": "x"})
    for dtype, n in ((torch.bfloat16, 600_001), (torch.float16, 2_500_000)):
        g, r = _pair(kind, n, dtype, 77)
        print("dense half tolerant", kind, dtype, n, flush=True)
        got = verdict._compare_tensors(g.to(DEV), r.to(DEV), "output", TOL, policy)
        want = tv.compare_tensors(g, r, "output", TOL, policy)
        assert got[0] == want[0]
        assert not meta_problems(got[2], want[2], g, r)
