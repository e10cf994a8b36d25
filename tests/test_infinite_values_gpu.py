"""Infinities in V where split pieces are merged: an Inf in one piece's values comes out as Inf in its dimension and
nowhere else (the merges read their last piece again to fill a batch: weighed with 0, that Inf would give NaN).
K is zero, so every weight is 1/n.  float16 and float32 (bf16 weights are split in two parts, one of them 0)."""

from __future__ import annotations

import pytest
import torch

from helpers import announce

pytestmark = pytest.mark.gpu
DEV = "cuda"


def check(out, v, dim, tol):
    """out (..., D) of uniform weights over v (B, Hkv, T, D), every head alike but for the group."""
    G = out.shape[1] // v.shape[1]
    ref = v.double().mean(2).repeat_interleave(G, 1)[:, :, None].expand(out.shape)
    assert torch.isposinf(out[..., dim]).all()
    keep = [d for d in range(v.shape[-1]) if d != dim]
    torch.testing.assert_close(out[..., keep].double(), ref[..., keep], rtol=0, atol=tol)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("B", [64, 128])     # 4 and 2 waves (two and one at head_dim 256) per unit
def test_decode_waves(gpu_pkg, B, D):
    announce(f"Inf in a wave's share B={B} D={D}")
    T = 64
    q = torch.randn(B, 8, 1, D, device=DEV, dtype=torch.float16)
    v = torch.randn(B, 8, T, D, device=DEV, dtype=torch.float16)
    v[:, :, T - 3, 5] = float("inf")
    kl = torch.tensor([T], dtype=torch.int32, device=DEV)
    out = gpu_pkg.attention_flash_decode(q, torch.zeros_like(v), v, kl).transpose(1, 2)
    check(out, v, 5, 2e-3)


@pytest.mark.parametrize("D", [16, 64, 128, 256])
@pytest.mark.parametrize("pieces", [2, 7, 8, 9])
def test_fp32_pieces(gpu_pkg, D, pieces):
    announce(f"Inf in the last fp32 piece of {pieces}, D={D}")
    T = 16 * pieces
    q = torch.randn(2, 6, 1, D, device=DEV)
    v = torch.randn(2, 2, T, D, device=DEV)
    v[:, :, T - 9, 5] = float("inf")
    kl = torch.tensor([T], dtype=torch.int32, device=DEV)
    with gpu_pkg.decode_options(tiles_per_split=1):
        out = gpu_pkg.attention_flash_decode(q, torch.zeros_like(v), v, kl).transpose(1, 2)
    check(out, v, 5, 1e-5)


@pytest.mark.parametrize("D,Tk", [(64, 8192), (128, 8192), (128, 3072), (256, 6016)])
def test_prefill_runs(gpu_pkg, D, Tk):
    announce(f"Inf in the last run of keys D={D} Tk={Tk}")
    q = torch.randn(1, 8, 5, D, device=DEV, dtype=torch.float16)
    v = torch.randn(1, 2, Tk, D, device=DEV, dtype=torch.float16)
    v[:, :, Tk - 3, 5] = float("inf")
    check(gpu_pkg.attention_flash_triton(q, torch.zeros_like(v), v, False), v, 5, 2e-3)
