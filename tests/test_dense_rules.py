"""The rules of the main pass's dense items on the host (no GPU): csrc/kvv_bounds.h,
what the kernels call, built with g++.

* The one-compare test (lean_tol, lean_close) passes only pairs that torch's
  isclose calls close, and passes every finite pair of equal values, whatever the
  tolerances.
* dense_pays takes an item over where that is the cheaper way, and not where most
  of what it would skip fails the test anyway.
"""

import ctypes
import itertools
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parents[1] / "kernelverse_amd" / "csrc"

HARNESS = r"""
#include "kvv_bounds.h"
extern "C" void closes(int n, const float* g, const float* r, float rtol, float atol, uint8_t* out) {
  const kvv::LeanTol t = kvv::lean_tol(rtol, atol, rtol == 0.0f && atol == 0.0f);
  for (int i = 0; i < n; ++i) out[i] = kvv::lean_close(fabsf(g[i] - r[i]), g[i], t.rtol, t.atol);
}
extern "C" int pays(int fp32, int capture, uint32_t slow, uint32_t pairs, uint32_t lanes, uint32_t pass, uint32_t miss) {
  return kvv::dense_surely_pays(fp32, slow, pairs) || kvv::dense_pays(fp32, capture, slow, pairs, lanes, pass, miss);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("dense")
    src = d / "h.cpp"
    src.write_text(HARNESS)
    so = d / "h.so"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", f"-I{CSRC}", str(src), "-o", str(so)], check=True)
    return ctypes.CDLL(str(so))


def _closes(lib, g, r, rtol, atol):
    out = np.zeros(g.size, np.uint8)
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    lib.closes(ctypes.c_int(g.size), p(g), p(r), ctypes.c_float(rtol), ctypes.c_float(atol), p(out))
    return out.astype(bool)


TOLERANCES = [(1e-5, 1e-5), (1.6e-2, 1e-2), (0.0, 1e-3), (1e-3, 0.0), (0.0, 0.0), (1e-35, 0.0), (0.0, 1e-40), (1e31, 1e-5),
              (2.0 ** -100, 2.0 ** -100), (1.0, 0.0), (2.0 ** -20, 0.0)]


@pytest.mark.parametrize("rtol,atol", TOLERANCES)
def test_passing_pairs_are_close(lib, rtol, atol):
    rng = np.random.default_rng(3)
    f = np.float32
    rt, at = f(rtol), f(atol)
    n = 200_000
    # magnitudes over the whole range, denormals and zeros among them
    g = (rng.standard_normal(n) * np.exp2(rng.integers(-149, 120, n).astype(np.float64))).astype(f)
    g[::50] = 0
    with np.errstate(all="ignore"):
        allowed = at + np.abs(rt * g)
        # references at the allowed bound, a few floats to either side, and equal
        step = rng.integers(-4, 5, n).astype(np.int32)
        edge = (g + np.where(rng.random(n) < 0.5, allowed, -allowed)).astype(f)
        r = (edge.view(np.int32) + step).view(f)
        r = np.where(np.isfinite(r), r, g).astype(f)
        r[::7] = g[::7]
        ad = np.abs(g - r)
        close = (g == r) if rtol == 0.0 and atol == 0.0 else (g == r) | (np.isfinite(ad) & (ad <= allowed))
    got = _closes(lib, g, r, rtol, atol)
    assert not (got & ~close).any()
    assert got[g == r].all()


@pytest.mark.parametrize("rtol,atol", TOLERANCES)
def test_non_finite_pairs_never_pass(lib, rtol, atol):
    inf, nan = np.float32(np.inf), np.float32(np.nan)
    pairs = [p for p in itertools.product([inf, -inf, nan, np.float32(0), np.float32(1)], repeat=2)
             if not (np.isfinite(p[0]) and np.isfinite(p[1]))]
    g, r = (np.array(x, np.float32) for x in zip(*pairs))
    assert not _closes(lib, g, r, rtol, atol).any()


# (fp32, capture, share of slow pairs, of which pass, of which miss): the others are not finite
TAKEN = [(1, 0, 1.0, 1.0, 0.0), (0, 0, 1.0, 1.0, 0.0), (0, 0, 0.3, 1.0, 0.0), (1, 0, 0.3, 1.0, 0.0),
         (0, 0, 0.5, 0.8, 0.2), (1, 0, 1.0, 0.0, 1.0),   # noise with a tenth of mismatches; fp32 all beyond the tolerance
         (0, 0, 0.75, 0.33, 0.0), (1, 0, 0.95, 0.5, 0.0),  # half masked, noise elsewhere
         (1, 1, 0.5, 0.0, 0.0)]                            # half masked, capture segment
LEFT = [(0, 0, 0.5, 0.0, 1.0), (0, 0, 1.0, 0.0, 1.0),      # 16-bit: all that differs is beyond the tolerance
        (1, 0, 0.3, 0.0, 1.0), (0, 0, 0.3, 0.0, 1.0),
        (0, 0, 0.5, 0.0, 0.0), (1, 0, 0.5, 0.0, 0.0),      # half masked, identical elsewhere
        (0, 0, 0.2, 1.0, 0.0), (1, 0, 0.2, 1.0, 0.0)]


@pytest.mark.parametrize("pairs", [256, 512, 1024, 2048])
@pytest.mark.parametrize("taken", [True, False])
def test_dense_pays(lib, taken, pairs):
    for fp32, capture, slow, passing, miss in TAKEN if taken else LEFT:
        for lanes in (64, 40):
            got = lib.pays(fp32, capture, round(slow * pairs), pairs, lanes, round(passing * lanes), round(miss * lanes))
            assert bool(got) == taken, (fp32, capture, slow, passing, miss, pairs, lanes)
