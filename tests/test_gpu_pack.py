"""Pairs copied into the workspace before the main pass (layouts without
16-byte vectors) against the oracle and the scalar main pass (needs an MI355X):
transposed, channels-last, sliced, stepped, misaligned and broadcast views of
one or both tensors, every element size, sizes at the edges of the copy's 64 x
64 tiles and of its vectors, and a workspace without room for the copies."""

import ctypes

import pytest
import torch

from kernelverse_amd import _lib, verdict
from kernelverse_amd.correctness_policy import resolve_correctness_policy
from oracle import torch_verdict as tv
from parity_util import meta_problems, record_vs_oracle

pytestmark = pytest.mark.gpu

DEV = "cuda"
DTYPES = [torch.float32, torch.bfloat16, torch.float16, torch.float64, torch.float8_e5m2, torch.int8, torch.int32,
          torch.int64, torch.bool]


def _transposed(t):
    return t.transpose(0, -1).contiguous().transpose(0, -1)


def _swapped_outer(t):
    return t.transpose(0, 1).contiguous().transpose(0, 1)


def _channels_last(t):
    return t.movedim(1, -1).contiguous().movedim(-1, 1)


def _sliced(t):
    base = torch.zeros(*t.shape[:-1], t.shape[-1] + 1, dtype=t.dtype, device=t.device)
    base[..., 1:] = t
    return base[..., 1:]


def _stepped(t):
    base = torch.zeros(*t.shape[:-1], 2 * t.shape[-1], dtype=t.dtype, device=t.device)
    base[..., ::2] = t
    return base[..., ::2]


def _offset(t):
    base = torch.zeros(t.numel() + 1, dtype=t.dtype, device=t.device)
    base[1:] = t.reshape(-1)
    return base[1:].view(t.shape)


def _pair(shape, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    r = torch.randn(shape, generator=gen) * 20
    moved = torch.rand(shape, generator=gen) < 0.1
    if dtype == torch.bool:
        r = r > 0
        return r ^ moved, r
    if not dtype.is_floating_point:
        r = r.to(dtype)
        return r + moved.to(dtype) * 3, r
    g = torch.where(moved, r * 1.05, r)
    return g.to(dtype), r.to(dtype)


CASES = [((64, 64), _transposed), ((65, 63), _transposed), ((129, 40), _transposed), ((33, 1000), _transposed),
         ((3, 17, 70), _transposed), ((2, 20, 9, 31), _channels_last), ((1, 64, 30, 30), _channels_last),
         ((40, 33), _sliced), ((7, 5, 129), _sliced), ((300, 17), _stepped), ((513,), _offset), ((70_001,), _offset),
         ((5, 7, 41), _swapped_outer), ((514, 2), _transposed)]


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
def test_packed_pair_matches_oracle(dtype):
    for k, (shape, lay) in enumerate(CASES):
        g, r = _pair(shape, dtype, k)
        print("pack", dtype, shape, lay.__name__, flush=True)
        gd, rd = g.to(DEV), r.to(DEV)
        for a, b in ((gd, lay(rd)), (lay(gd), rd), (lay(gd), lay(rd))):
            assert not record_vs_oracle(verdict.verdict_record(a, b), g, r)


def test_packed_broadcast_reference():
    g, _ = _pair((600, 50), torch.float32, 1)
    row = torch.randn(600, 1)
    rec = verdict.verdict_record(g.to(DEV), row.to(DEV).expand(600, 50))
    assert not record_vs_oracle(rec, g, row.expand(600, 50).contiguous())


def test_packed_tolerant_meta():
    policy = resolve_correctness_policy({"category": "gemm", "op_name": "x"})
    tol = {"BF16": {"rtol": 1.6e-2, "atol": 1e-2}}
    g, r = _pair((1500, 1001), torch.bfloat16, 5)
    g, r = g / 20, r / 20
    got = verdict._compare_tensors(g.to(DEV), _transposed(r.to(DEV)), "output", tol, policy)
    want = tv.compare_tensors(g, r, "output", tol, policy)
    assert got[0] == want[0] and not meta_problems(got[2], want[2], g, r)


@pytest.mark.parametrize("shape", [(64, 70), (1200, 1100)])
def test_workspace_without_room_for_the_copies(shape):
    """The least workspace takes the scalar pass: the same record (fp64 sums within their bound)."""
    lib = _lib.load()
    g, r = _pair(shape, torch.float32, 9)
    gd, rd = g.to(DEV), _transposed(r.to(DEV))
    gt, rt = verdict._kvv_tensor(gd), verdict._kvv_tensor(rd)
    job = verdict._Job(gd, rd, "output", None, None, verdict.MAX_SAMPLES)
    size = ctypes.c_size_t()
    _lib.check(lib.kvv_workspace_size(gt, rt, job.kpolicy, ctypes.byref(size)), "kvv_workspace_size")
    copy = g.numel() * 4
    assert size.value > copy
    out = torch.empty(ctypes.sizeof(_lib.KvvResult), dtype=torch.uint8, pin_memory=True)
    recs = []
    for room in (size.value, size.value - 256):
        ws = torch.empty(room, dtype=torch.uint8, device=DEV)
        _lib.check(lib.kvv_verdict(gt, rt, job.kpolicy, out.data_ptr(), ws.data_ptr(), room,
                                   torch.cuda.current_stream().cuda_stream), "kvv_verdict")
        torch.cuda.synchronize()
        recs.append(_lib.KvvResult.from_buffer_copy(out.numpy().tobytes()).to_dict())
    for rec in recs:
        assert not record_vs_oracle(rec, g, r)
    exact = [k for k, v in recs[0].items() if isinstance(v, (int, list))] + ["p99_abs", "p99_rel", "max_abs", "max_rel"]
    assert all(recs[0][k] == recs[1][k] for k in exact)


def test_device_without_room_for_the_copies(monkeypatch):
    """A drop-in verdict whose workspace cannot be allocated with room for the copies runs with the least one."""
    g, r = _pair((5000, 4100), torch.float32, 3)
    gd, rd = g.to(DEV), _transposed(r.to(DEV))
    want = verdict._compare_tensors(gd, rd, "output")
    verdict.release_buffers()
    empty = torch.empty

    def short(n, *args, **kw):
        if kw.get("dtype") == torch.uint8 and not kw.get("pin_memory") and n > verdict._LEAST_WS:
            raise torch.OutOfMemoryError("no room")
        return empty(n, *args, **kw)

    monkeypatch.setattr(torch, "empty", short)
    for _ in range(2):
        assert repr(verdict._compare_tensors(gd, rd, "output")) == repr(want)
    monkeypatch.undo()
    assert repr(verdict._compare_tensors(gd, rd, "output")) == repr(want)
    verdict.release_buffers()
