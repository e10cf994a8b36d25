"""The stream-K split's 32-bit arithmetic (csrc/decode_kernel.hpp, sk_split / sk_lo / sk_group), on the CPU.

The kernel divides with one fp32 product by an approximate reciprocal
(v_rcp_f32: within one ulp) and a correction.  Here the same steps run in numpy
with the reciprocal off by up to one ulp either way and are compared with exact
integer division over work lines, grids and positions of every size class.
"""

from __future__ import annotations

import numpy as np

F = np.float32


def rcp(x, ulps):
    r = F(1.0) / F(x)
    for _ in range(abs(ulps)):
        r = np.nextafter(r, F(np.inf if ulps > 0 else 0))
    return r


def lo(g, W, G, ulps):
    Q, R = W // G, W % G
    n = g * R
    assert np.all(n < 1 << 24)
    q = (n.astype(F) * rcp(G, ulps)).astype(np.int64)
    r = n - q * G
    q = q + np.where(r >= G, 1, np.where(r < 0, -1, 0))
    return g * Q + q


def group(x, W, G, ulps):
    est = np.ceil((x + 1).astype(F) * (F(G) * rcp(W, ulps))).astype(np.int64) - 1
    g = np.clip(est, 0, G - 1)
    g = np.where((g > 0) & (lo(g, W, G, ulps) > x), g - 1, g)
    return np.where((g + 1 < G) & (lo(np.minimum(g + 1, G - 1), W, G, ulps) <= x), g + 1, g)


def test_split_equals_integer_division():
    rng = np.random.default_rng(0)
    for G in (1, 2, 3, 7, 64, 255, 256, 257, 511, 512, 1000, 1024, 4095):
        for W in (1, 2, 5, 63, 255, 256, 4097, 100003, (1 << 24) - 1, (1 << 24) + 1, 1 << 30, (1 << 31) - 1):
            for ulps in (-1, 0, 1):
                g = np.arange(G + 1, dtype=np.int64)
                assert np.array_equal(lo(g, W, G, ulps), g * W // G), (W, G, ulps)
                x = np.unique(np.concatenate([rng.integers(0, W, 400), [0, W - 1], np.clip(g * W // G, 0, W - 1),
                                              np.clip(g * W // G - 1, 0, W - 1)])).astype(np.int64)
                want = -(-(x + 1) * G // W) - 1
                assert np.array_equal(group(x, W, G, ulps), want), (W, G, ulps)
