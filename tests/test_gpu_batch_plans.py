"""The nested-output plans kept between calls (needs an MI355X): repeated calls
with new tensors of the same layouts, calls that differ only in policy, dtype,
stride or alignment, an empty leaf, more distinct sequences than are kept, and
single-pair calls in between; every meta equals the one from fresh buffers."""

import pytest
import torch

from kernelverse_amd import verdict
from kernelverse_amd.correctness_policy import resolve_correctness_policy

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _pair(shape, dtype, seed, offset=False):
    gen = torch.Generator().manual_seed(seed)
    r = torch.randn(shape, generator=gen)
    g = r + 0.02 * torch.randn(shape, generator=gen) * (torch.rand(shape, generator=gen) < 0.2)
    out = []
    for t in (g, r):
        t = t.to(dtype).to(DEV)
        if offset:
            base = torch.zeros(t.numel() + 1, dtype=dtype, device=DEV)
            base[1:] = t.reshape(-1)
            t = base[1:].view(shape)
        out.append(t)
    return out


def _call(spec, seed, policy):
    pairs = [_pair(shape, dtype, seed + i, off) for i, (shape, dtype, off) in enumerate(spec)]
    outs, refs = tuple(p[0] for p in pairs), tuple(p[1] for p in pairs)
    got = verdict._compare_outputs(outs, refs, correctness_policy=policy)
    verdict._compare_tensors(*pairs[0], "x", None, policy)
    again = verdict._compare_outputs(outs, refs, correctness_policy=policy)
    verdict.release_buffers()
    want = verdict._compare_outputs(outs, refs, correctness_policy=policy)
    assert repr(got) == repr(want) and repr(again) == repr(want)
    return outs, refs, want


def test_kept_batch_plans():
    f32, bf, h = torch.float32, torch.bfloat16, torch.float16
    specs = [[((64, 80), f32, False), ((3000,), bf, False)], [((64, 80), f32, True), ((3000,), bf, False)],
             [((64, 80), f32, False), ((3000,), h, False)], [((64, 80), f32, False), ((0, 4), bf, False), ((40_000,), h, False)]]
    calls = []
    for k, spec in enumerate(specs):
        for name in ("gemm", "activation"):
            policy = resolve_correctness_policy({"category": name, "op_name": "x"})
            for seed in (1, 100):
                calls.append((*_call(spec, seed + k, policy), policy))
    # all of them again on one set of buffers, each plan now met with the pointers of another call
    for outs, refs, want, policy in calls + calls[::-1]:
        assert repr(verdict._compare_outputs(outs, refs, correctness_policy=policy)) == repr(want)


def test_more_sequences_than_are_kept():
    for n in range(40):
        a, b = _pair((100 + n,), torch.float32, n), _pair((50,), torch.float32, n + 1)
        got = verdict._compare_outputs([a[0], b[0]], [a[1], b[1]])
        one = verdict._compare_tensors(a[0], a[1], "output[0]")
        assert repr(got[2][0]) == repr(one[2])
    buf = verdict._stream_buffers(torch.device("cuda", torch.cuda.current_device()))
    assert len(buf.batch_plans) <= verdict._MAX_BATCH_PLANS
