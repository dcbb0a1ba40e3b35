"""Row-layout pairs (contiguous rows under outer strides) against the oracle
(needs an MI355X): one to four outer dims, permuted and pitched views, an
expanded (stride 0) reference, rows shorter and longer than a wave's vectors,
odd dims, single calls and a batch of all of them."""

import pytest
import torch

from kernelverse_amd import verdict
from parity_util import record_vs_oracle

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _heads(t):
    b, h, s, d = t.shape
    return t.transpose(1, 2).contiguous().transpose(1, 2)


def _pitched(pad):
    def f(t):
        base = torch.zeros(*t.shape[:-1], t.shape[-1] + pad, dtype=t.dtype, device=t.device)
        v = base[..., :t.shape[-1]]
        v.copy_(t)
        return v
    return f


def _outer_swapped(t):
    return t.transpose(0, -2).contiguous().transpose(0, -2)


CASES = [
    ((3, 5, 7, 64), torch.float16, _heads),            # three outer dims, odd sizes
    ((2, 16, 33, 128), torch.bfloat16, _heads),
    ((4, 3, 129, 8), torch.float32, _heads),           # rows of two vectors
    ((1000, 24), torch.float32, _pitched(8)),          # one outer dim
    ((17, 4096), torch.bfloat16, _pitched(64)),        # rows of whole items
    ((3, 50, 40), torch.float16, _pitched(24)),        # two outer dims that do not merge
    ((2, 3, 4, 5, 32), torch.float16, _outer_swapped),  # four outer dims: the divisions
    ((6, 700, 16), torch.int8, _outer_swapped),
]


def _pair(shape, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    if dtype == torch.int8:
        r = torch.randint(-100, 100, shape, generator=gen, dtype=torch.int8)
        g = r + (torch.rand(shape, generator=gen) < 0.05).to(torch.int8) * 3
        return g, r
    r = torch.randn(shape, generator=gen).to(dtype)
    g = (r.float() * (1 + 0.02 * torch.randn(shape, generator=gen) * (torch.rand(shape, generator=gen) < 0.3))).to(dtype)
    return g, r


@pytest.mark.parametrize("k", range(len(CASES)))
def test_row_view_matches_oracle(k):
    shape, dtype, lay = CASES[k]
    g, r = _pair(shape, dtype, k)
    print("row view", shape, dtype, flush=True)
    gd, rd = lay(g.to(DEV)), lay(r.to(DEV))
    for a, b in ((gd, rd), (g.to(DEV), rd), (gd, r.to(DEV))):
        assert not record_vs_oracle(verdict.verdict_record(a, b), g, r)


def test_row_view_expanded_reference():
    g = torch.randn(300, 64)
    r = torch.randn(1, 64).expand(300, 64)
    rec = verdict.verdict_record(g.to(DEV), r[:1].to(DEV).expand(300, 64))
    assert not record_vs_oracle(rec, g, r.contiguous())


def test_row_views_in_a_batch():
    pairs, want = [], []
    for k, (shape, dtype, lay) in enumerate(CASES):
        g, r = _pair(shape, dtype, 100 + k)
        pairs.append((lay(g.to(DEV)), lay(r.to(DEV))))
        want.append((g, r))
    for rec, (g, r) in zip(verdict.verdict_records(pairs), want):
        assert not record_vs_oracle(rec, g, r)
