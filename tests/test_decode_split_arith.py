"""The stream-K split's 32-bit arithmetic, compiled for the CPU from the kernel's own header (csrc/sk_split.hpp).

The kernel divides with one fp32 product by an approximate reciprocal (v_rcp_f32: within one ulp) and a correction.
Here the reciprocals are off by up to one ulp either way, and the results are compared with exact integer division over
work lines, grids (up to the launch's cap) and positions of every size class.
"""

from __future__ import annotations

import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT

SOURCE = """
#define __host__
#define __device__
#define __forceinline__ inline
#include "sk_split.hpp"
extern "C" int cap() { return sia::kMaxSplitGroups; }
extern "C" void lo(int n, const int* g, int* out, int W, int G, float rG, float rW) {
  const sia::SkSplit s = sia::sk_split(W, G, rG, rW);
  for (int i = 0; i < n; ++i) out[i] = sia::sk_lo(s, g[i]);
}
extern "C" void group(int n, const int* x, int* out, int W, int G, float rG, float rW) {
  const sia::SkSplit s = sia::sk_split(W, G, rG, rW);
  for (int i = 0; i < n; ++i) out[i] = sia::sk_group(s, x[i]);
}
"""
F = np.float32


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("split")
    (d / "split.cpp").write_text(SOURCE)
    csrc = os.path.join(ROOT, "simple-inference-autoresearch_amd", "csrc")
    # (the fp32 steps as written: no contraction)
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", csrc, "-o",
                    str(d / "split.so"), str(d / "split.cpp")], check=True)
    return ctypes.CDLL(str(d / "split.so"))


def rcp(x, ulps):
    r = F(1.0) / F(x)
    for _ in range(abs(ulps)):
        r = np.nextafter(r, F(np.inf if ulps > 0 else 0))
    return r


def run(f, v, W, G, ulps):
    v = np.ascontiguousarray(v, dtype=np.int32)
    out = np.empty_like(v)
    p = ctypes.POINTER(ctypes.c_int)
    f(len(v), v.ctypes.data_as(p), out.ctypes.data_as(p), ctypes.c_int(W), ctypes.c_int(G),
      ctypes.c_float(rcp(G, ulps)), ctypes.c_float(rcp(W, ulps)))
    return out.astype(np.int64)


def test_cap_keeps_products_below_2_to_24(lib):
    assert (lib.cap() - 1) * lib.cap() < 1 << 24


def test_split_equals_integer_division(lib):
    rng = np.random.default_rng(0)
    for G in (1, 2, 3, 7, 64, 255, 256, 257, 511, 512, 1000, 1024, lib.cap()):
        for W in (1, 2, 5, 63, 255, 256, 4097, 100003, (1 << 24) - 1, (1 << 24) + 1, 1 << 30, (1 << 31) - 1):
            for ulps in (-1, 0, 1):
                g = np.arange(G + 1, dtype=np.int64)
                assert np.array_equal(run(lib.lo, g, W, G, ulps), g * W // G), (W, G, ulps)
                x = np.unique(np.concatenate([rng.integers(0, W, 400), [0, W - 1], np.clip(g * W // G, 0, W - 1),
                                              np.clip(g * W // G - 1, 0, W - 1)])).astype(np.int64)
                want = -(-(x + 1) * G // W) - 1
                assert np.array_equal(run(lib.group, x, W, G, ulps), want), (W, G, ulps)
