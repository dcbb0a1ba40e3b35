"""The drop-in's kept plans and workspaces, on the CPU: the library plans for real
(no device is needed for that), its launching entry points are replaced by
recorders and device allocations by plain sizes with a limit.

* A pair whose tensors differ in shape or type is refused before anything is
  launched, whatever plans earlier calls left.
* A pair whose workspace holds copies of its tensors runs without them where the
  device has no room, does not ask for that room again on each call, and keeps no
  large copies between calls."""

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


def _on_device(shape, dtype, address, strides=(80, 1)):
    t = torch.empty_strided(shape, strides, dtype=dtype, device="meta").as_subclass(_OnDevice)
    t.address = address
    return t


class _Stream:
    cuda_stream = 0

    def synchronize(self):
        pass


class _Recorder:
    """libkvv with its launches recorded (entry point, workspace bytes) instead of issued."""

    def __init__(self, lib):
        self._lib, self.launched = lib, []

    def __getattr__(self, name):
        return getattr(self._lib, name)

    def kvv_verdict(self, gen, ref, policy, out, ws, ws_bytes, stream):
        least, copies = ctypes.c_size_t(), ctypes.c_size_t()
        assert self._lib.kvv_workspace_parts(gen, ref, policy, least, copies) == 0
        assert ws_bytes >= least.value  # (what the library itself would refuse)
        self.launched.append(("kvv_verdict", ws_bytes))
        return 0

    def kvv_verdict_batch(self, count, gens, refs, policies, out, ws, ws_bytes, stream):
        self.launched.append(("kvv_verdict_batch", ws_bytes))
        return 0


class _Block:
    """A device allocation of n bytes."""

    def __init__(self, n):
        self.n = n

    def numel(self):
        return self.n

    def data_ptr(self):
        return 1 << 40


class _Device:
    """Allocations of up to ``room`` bytes succeed; ``asked`` holds every size asked for."""

    def __init__(self, empty):
        self.empty, self.room, self.asked = empty, 1 << 50, []

    def __call__(self, n, *args, **kw):
        if kw.pop("pin_memory", False):
            return self.empty(n, *args, **kw).zero_()
        self.asked.append(n)
        if n > self.room:
            raise torch.OutOfMemoryError("no room")
        return _Block(n)


@pytest.fixture
def device(monkeypatch):
    dev = _Device(torch.empty)
    dev.lib = _Recorder(_lib.load())
    dev.buf = verdict._Buffers(_Stream())
    monkeypatch.setattr(torch, "empty", dev)
    monkeypatch.setattr(_lib, "load", lambda: dev.lib)
    monkeypatch.setattr(verdict, "_GET_DEVICE", lambda: 0)
    monkeypatch.setattr(verdict, "_stream_buffers", lambda d: dev.buf)
    return dev


def _pair(address, shape=(64, 80), dtype=torch.float64):
    """A float64 pair of 64 x 80 whose reference has the given shape and type."""
    return (_on_device((64, 80), torch.float64, address), _on_device(shape, dtype, address + (1 << 20)))


DIFFERING = {"shape": {"shape": (32, 80)}, "dtype": {"dtype": torch.float32}}


@pytest.mark.parametrize("pairs", [1, 3])
@pytest.mark.parametrize("what", ["shape", "dtype"])
def test_kept_plan_refuses_a_differing_pair(device, pairs, what):
    entry = "kvv_verdict" if pairs == 1 else "kvv_verdict_batch"
    same = [_pair(4096 * (1 + i)) for i in range(pairs)]
    mixed = same[:-1] + [_pair(4096 * pairs, **DIFFERING[what])]
    # (fp64 and fp32 share a tolerance: the two calls' policy keys are equal)
    jobs = [verdict._Job(*p, "output", None, None, verdict.MAX_SAMPLES) for p in (same[-1], mixed[-1])]
    assert jobs[0].pkey == jobs[1].pkey
    with pytest.raises(_lib.KvvLibraryError, match=f"{what}s differ"):
        verdict.verdict_records(mixed)
    assert device.lib.launched == []
    verdict.verdict_records(same)
    verdict.verdict_records(same)
    assert [name for name, _ in device.lib.launched] == [entry, entry]
    with pytest.raises(_lib.KvvLibraryError, match=f"{what}s differ"):
        verdict.verdict_records(mixed)
    assert [name for name, _ in device.lib.launched] == [entry, entry]


def _transposed(rows, cols):
    return (_on_device((rows, cols), torch.float32, 4096, (cols, 1)), _on_device((rows, cols), torch.float32, 8192, (1, rows)))


@pytest.mark.parametrize("max_samples,room", [(1_000_000, 64 << 20), (1 << 24, 200 << 20)])
def test_device_without_room_for_the_copies(device, max_samples, room):
    """The fallback holds the pair's own samples (2 x 64 MiB at the largest max_samples), and the size that found no
    room is asked for again only after _SHORT_CALLS calls."""
    pair = _transposed(5000, 4100)
    device.room = room
    for _ in range(1 + verdict._SHORT_CALLS):
        verdict.verdict_records([pair], max_samples=max_samples)
    full = max(device.asked)
    assert full > room and device.asked.count(full) == 1
    assert all(b <= room for _, b in device.lib.launched)
    device.room = 1 << 50
    verdict.verdict_records([pair], max_samples=max_samples)
    assert device.lib.launched[-1][1] == full


def test_contiguous_pair_without_room_raises(device):
    device.room = 1 << 20
    g = _on_device((5000, 4100), torch.float32, 4096, (4100, 1))
    with pytest.raises(torch.OutOfMemoryError):
        verdict.verdict_records([(g, g)])
    assert device.lib.launched == []


def test_large_copies_are_not_kept(device):
    small, large = _transposed(2000, 3000), _transposed(16384, 16384)
    verdict.verdict_records([small])
    held = device.buf.ws_bytes
    for _ in range(2):
        verdict.verdict_records([large])
        assert device.lib.launched[-1][1] > 1 << 30 and device.buf.ws_bytes == held and device.buf.kept
    verdict.verdict_records([small])
    assert device.lib.launched[-1][1] <= held
