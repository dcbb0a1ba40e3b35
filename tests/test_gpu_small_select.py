"""The block select of small groups (needs an MI355X): its rank's bin collected
and ranked by comparison, or binned again when it holds more values than that
takes; sizes at the edges of the value groups, ties around the candidates'
limit, ranks far apart, and the same through many-group batches, whose captured
values the same select reads."""

import pytest
import torch

from kernelverse_amd import verdict
from oracle import torch_verdict as tv
from parity_util import record_vs_oracle

pytestmark = pytest.mark.gpu

DEV = "cuda"
SIZES = [1, 2, 3, 101, 255, 256, 257, 2047, 2048, 2049, 4096, 6145, 8191, 8192]


def _diffs(kind, n, gen):
    d = torch.randn(n, generator=gen).abs() * 1e-3 + 1e-6
    k = n - 1 - int(0.99 * (n - 1))
    order = torch.randperm(n, generator=gen)
    if kind == "apart":
        # the two order statistics in bins far apart
        d[order[:k]] = 1000.0 + torch.arange(k, dtype=torch.float32)
    elif kind == "zeros":
        d[order[k:]] = 0.0
    elif kind.startswith("ties"):
        # values of one bin around the rank: that many equal ones, or distinct neighbours
        m = min(n, int(kind[4:]))
        d[order[:m]] = 0.5 + (torch.arange(m) % 3) * 2.0 ** -24
    elif kind == "crowd":
        d = 0.5 + torch.randint(0, 64, (n,), generator=gen).float() * 2.0 ** -23
        d[order[0]] = 1e30
        d[order[-1]] = 1e-30
    return d


KINDS = ["noise", "apart", "zeros", "ties254", "ties255", "ties256", "ties257", "ties600", "crowd"]


@pytest.mark.parametrize("kind", KINDS)
def test_small_group(kind):
    for n in SIZES:
        gen = torch.Generator().manual_seed(n)
        # (a zero reference: abs_diff is exactly the drawn value)
        g = _diffs(kind, n, gen)
        r = torch.zeros(n)
        print(kind, n, flush=True)
        assert not record_vs_oracle(verdict.verdict_record(g.to(DEV), r.to(DEV)), g, r)


def test_captured_groups():
    gen = torch.Generator().manual_seed(7)
    pairs = []
    for i in range(300):
        n = 9000 + 311 * i
        g = _diffs(KINDS[i % len(KINDS)], n, gen)
        r = torch.zeros(n) if i % 2 else torch.randn(n, generator=gen)
        pairs.append(((r + g) if i % 2 == 0 else g, r))
    got = verdict._compare_outputs([g.to(DEV) for g, _ in pairs], [r.to(DEV) for _, r in pairs])
    for meta, (g, r) in zip(got[2], pairs):
        want = tv.compare_tensors(g, r, "output")[2]
        assert meta["p99_abs"] == want["p99_abs"] and meta["p99_rel"] == want["p99_rel"]
