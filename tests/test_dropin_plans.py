"""The drop-in's kept plans meet a pair whose tensors differ in shape or type: the
call is refused before anything is launched, whatever plans earlier calls left.
Runs on the CPU: the library plans for real (no device is needed for that) and its
two launching entry points are replaced by recorders."""

import ctypes

import pytest
import torch

from kernelverse_amd import _lib, verdict


class _OnDevice(torch.Tensor):
    """A CPU tensor that gives a device index and a made-up address."""

    def get_device(self):
        return 0

    def data_ptr(self):
        return self.address


def _on_device(shape, dtype, address):
    t = torch.empty_strided(shape, (80, 1), dtype=dtype).as_subclass(_OnDevice)
    t.address = address
    return t


class _Stream:
    cuda_stream = 0

    def synchronize(self):
        pass


class _Recorder:
    """libkvv with its launches recorded instead of issued."""

    def __init__(self, lib):
        self._lib, self.launched = lib, []

    def __getattr__(self, name):
        return getattr(self._lib, name)

    def kvv_verdict(self, *args):
        self.launched.append("kvv_verdict")
        return 0

    def kvv_verdict_batch(self, *args):
        self.launched.append("kvv_verdict_batch")
        return 0


@pytest.fixture
def recorder(monkeypatch):
    rec = _Recorder(_lib.load())
    buf = verdict._Buffers(_Stream())
    host = ctypes.create_string_buffer(64 * verdict._REC_SIZE)

    def ensure(b, dev, ws_bytes, records, *more):
        b.ws, b.ws_bytes, b.ws_ptr = host, 1 << 40, 4096
        b.out, b.out_ptr = host, ctypes.addressof(host)
        b.out_rec = (ctypes.c_char * verdict._REC_SIZE).from_buffer(host)

    monkeypatch.setattr(_lib, "load", lambda: rec)
    monkeypatch.setattr(verdict, "_GET_DEVICE", lambda: 0)
    monkeypatch.setattr(verdict, "_stream_buffers", lambda dev: buf)
    monkeypatch.setattr(verdict, "_ensure", ensure)
    return rec


def _pair(address, shape=(64, 80), dtype=torch.float64):
    """A float64 pair of 64 x 80 whose reference has the given shape and type."""
    return (_on_device((64, 80), torch.float64, address), _on_device(shape, dtype, address + (1 << 20)))


DIFFERING = {"shape": {"shape": (32, 80)}, "dtype": {"dtype": torch.float32}}


@pytest.mark.parametrize("pairs", [1, 3])
@pytest.mark.parametrize("what", ["shape", "dtype"])
def test_kept_plan_refuses_a_differing_pair(recorder, pairs, what):
    entry = "kvv_verdict" if pairs == 1 else "kvv_verdict_batch"
    same = [_pair(4096 * (1 + i)) for i in range(pairs)]
    mixed = same[:-1] + [_pair(4096 * pairs, **DIFFERING[what])]
    # (fp64 and fp32 share a tolerance: the two calls' policy keys are equal)
    jobs = [verdict._Job(*p, "output", None, None, verdict.MAX_SAMPLES) for p in (same[-1], mixed[-1])]
    assert jobs[0].pkey == jobs[1].pkey
    with pytest.raises(_lib.KvvLibraryError, match=f"{what}s differ"):
        verdict.verdict_records(mixed)
    assert recorder.launched == []
    verdict.verdict_records(same)
    verdict.verdict_records(same)
    assert recorder.launched == [entry, entry]
    with pytest.raises(_lib.KvvLibraryError, match=f"{what}s differ"):
        verdict.verdict_records(mixed)
    assert recorder.launched == [entry, entry]
