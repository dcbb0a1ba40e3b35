"""The multiply-and-shift quotients of the row addressing (no GPU).

kvv::row_magic (csrc/kvv_bounds.h, what the host plans and the kernels use)
against integer division, over every small divisor, powers of two and their
neighbours, and random divisors, at multiples, just below them and at the top
of the 31-bit range.
"""

import ctypes
import subprocess
from pathlib import Path

import numpy as np

CSRC = Path(__file__).resolve().parents[1] / "kernelverse_amd" / "csrc"

HARNESS = r"""
#include "kvv_bounds.h"
extern "C" long bad(int n, const uint32_t* d, const uint32_t* x, int per) {
  long bad = 0;
  for (int i = 0; i < n; ++i) {
    uint32_t mul, sh;
    kvv::row_magic(d[i], mul, sh);
    for (int k = 0; k < per; ++k) {
      const uint32_t v = x[(long)i * per + k];
      bad += ((uint32_t)(((uint64_t)v * mul) >> 32) >> sh) != v / d[i];
    }
  }
  return bad;
}
"""


def test_quotients_are_exact(tmp_path):
    src = tmp_path / "h.cpp"
    src.write_text(HARNESS)
    so = tmp_path / "h.so"
    subprocess.run(["g++", "-O2", "-shared", "-fPIC", f"-I{CSRC}", str(src), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    lib.bad.restype = ctypes.c_long
    rng = np.random.default_rng(3)
    top = (1 << 31) - 1
    pows = np.array([1 << k for k in range(1, 31)], dtype=np.int64)
    d = np.concatenate([np.arange(2, 6000), pows, pows + 1, pows[1:] - 1, [top, top - 1],
                        np.exp(rng.uniform(np.log(2), np.log(top), 40_000)).astype(np.int64)])
    d = np.clip(d, 2, top)
    q = rng.integers(0, top // d[:, None] + 1, size=(d.size, 12))
    x = np.concatenate([q * d[:, None], np.maximum(q * d[:, None] - 1, 0), np.full((d.size, 1), top),
                        rng.integers(0, top + 1, size=(d.size, 8))], axis=1)
    x = np.minimum(x, top)
    dd, xx = np.ascontiguousarray(d, dtype=np.uint32), np.ascontiguousarray(x, dtype=np.uint32)
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    assert lib.bad(ctypes.c_int(d.size), p(dd), p(xx), ctypes.c_int(x.shape[1])) == 0
