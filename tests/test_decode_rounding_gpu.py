"""One rounding of the quotient ahead of the 16-bit one: averages of L float16 values whose exact mean is a tie between
two float16 values come out rounded to even, bit for bit (K is zero, so the weights are 1 and the sums exact).  A
product with a rounded 1 / L misses hundreds of these ties.  128 sequences of 8 KV heads: 2 waves per unit, merged and
stored by decode_main."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import announce

pytestmark = pytest.mark.gpu
DEV = "cuda"


def values_with_mean(m: int, L: int):
    """L float16 values (as multiples of 1/2048) whose mean is m/2048, m odd in [2049, 4095]."""
    for rem in range(2047, 2030, -2):
        x = 2 * m - L + 2 - rem
        if float(np.float16(x / 2048)) * 2048 == x:
            return [m + 1] * (L - 2) + [x, rem]
    raise AssertionError((m, L))


@pytest.mark.parametrize("L", [7, 15, 41, 61])
def test_ties(gpu_pkg, L):
    announce(f"ties of means of {L} values")
    B, H, D = 128, 8, 128
    odd = [m for m in range(2049, 4096, 2)
           if np.float16(np.float32(L * m / 2048) * (np.float32(1) / np.float32(L))) != np.float16(m / 2048)]
    m = np.resize(odd, D)                                 # the ties that 1 / L misses, one per dimension
    cols = np.array([values_with_mean(int(x), L) for x in m]).T / 2048
    v = torch.tensor(cols, dtype=torch.float16, device=DEV).expand(B, H, L, D).contiguous()
    q = torch.randn(B, H, 1, D, device=DEV, dtype=torch.float16)
    kl = torch.tensor([L], dtype=torch.int32, device=DEV)
    out = gpu_pkg.attention_flash_decode(q, torch.zeros_like(v), v, kl)
    want = torch.tensor(m / 2048, dtype=torch.float16, device=DEV).expand_as(out)   # round to nearest even
    assert torch.equal(out, want)
