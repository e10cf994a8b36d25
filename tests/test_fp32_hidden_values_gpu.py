"""fp32 prompts with Inf and NaN among the values: a key's value reaches exactly the query rows that see the key.

The rows of 32 (row, head) columns share a work-group and its tiles of 32 keys, where a key that some of them do not see
weighs 0 (and 0 times Inf is NaN).  Reference: finite values through a masked softmax in float64, the others added to
the rows that see them.  Bar 1e-5, the fp32 path's for N(0, 1) inputs; Inf and NaN are compared exactly."""

from __future__ import annotations

import pytest
import torch

from helpers import announce

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("Hq,Hkv", [(4, 1), (2, 2)])
@pytest.mark.parametrize("Tq,Tk,causal,keys", [
    (70, 70, True, [0, 33, 40, 69]),      # tiles on the diagonal, the last row's key
    (100, 100, True, [99]),
    (20, 100, True, [3, 84, 90]),         # a prompt's next part
    (40, 45, False, [44]),                # the last key of a partial tile, seen by every row
    (30, 10, True, [2, 9]),               # rows that see no key
])
def test_rows_that_see_the_key(gpu_pkg, D, Hq, Hkv, Tq, Tk, causal, keys):
    announce(f"fp32 values not finite D={D} {Hq}/{Hkv} {Tq}/{Tk} causal={causal} keys={keys}")
    g = torch.Generator(device=DEV).manual_seed(D + Tq)
    q, k, v = (torch.randn(1, H, T, D, generator=g, device=DEV) for H, T in ((Hq, Tq), (Hkv, Tk), (Hkv, Tk)))
    special = [float("inf"), float("nan"), float("-inf")]
    for i, key in enumerate(keys):
        v[:, :, key, (5 * i + 1) % D] = special[i % 3]
        v[:, :, key, D - 1 - i] = special[(i + 1) % 3]
    out = gpu_pkg.attention_flash_triton(q, k, v, causal).double()
    kd, vd = (x.double().repeat_interleave(Hq // Hkv, 1) for x in (k, v))
    s = (q.double()[:, :, :, None] * kd[:, :, None]).sum(-1) * D ** -0.5
    seen = torch.ones(Tq, Tk, dtype=torch.bool, device=DEV)
    if causal:
        seen = torch.arange(Tk, device=DEV)[None] <= torch.arange(Tq, device=DEV)[:, None] + (Tk - Tq)
    w = torch.softmax(s.masked_fill(~seen, float("-inf")), -1).nan_to_num(0.0)      # (rows without a key: zeros)
    ref = (w[..., None] * vd.nan_to_num(0.0, 0.0, 0.0)[:, :, None]).sum(3)
    for key in keys:
        x = torch.where(vd[:, :, key].isfinite(), 0.0, vd[:, :, key])               # (1, Hq, D)
        ref += torch.where(seen[:, key][None, None, :, None], x[:, :, None], 0.0)
    torch.testing.assert_close(out, ref, rtol=0, atol=1e-5, equal_nan=True)
