"""fp32 prefill at the edges of its tiles: 32 columns (query rows x heads) and 32 keys, 4 waves of every fourth tile.

Bar: that of the fp32 path, max-abs 1e-5 against the float64 oracle for N(0, 1)
inputs (fp32 sums of at most 256 products per score and a few hundred weights
per output, each within some 1e-6 of the exact value).
"""

from __future__ import annotations

import pytest
import torch

from oracle import attention as O
from helpers import announce, assert_close, f64

pytestmark = pytest.mark.gpu
DEV = "cuda"
FP32_TOL = 1e-5


def run(gpu_pkg, B, Hq, Hkv, Tq, Tk, D, causal, view, seed):
    announce(f"fp32 prefill tiles B={B} {Hq}/{Hkv} Tq={Tq} Tk={Tk} D={D} causal={causal} {view}")
    g = torch.Generator(device=DEV).manual_seed(seed)

    def t(H, T):
        x = torch.randn(B, H, T, D, generator=g, device=DEV)
        if view == "token_major":
            return x.transpose(1, 2).contiguous().transpose(1, 2)
        if view == "padded":
            big = torch.full((B, H, T + 5, D + 4), float("nan"), device=DEV)
            big[:, :, :T, :D] = x
            return big[:, :, :T, :D]
        return x

    q, k, v = t(Hq, Tq), t(Hkv, Tk), t(Hkv, Tk)
    out = gpu_pkg.attention_flash_triton(q, k, v, causal=causal, out_token_major=view == "token_major")
    torch.cuda.synchronize()
    got = out.transpose(1, 2) if view == "token_major" else out
    assert_close(got.contiguous(), O.flash_attention(f64(q), f64(k), f64(v), causal), FP32_TOL, "fp32 prefill")


@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("Hq,Hkv,Tq", [(4, 4, 31), (4, 4, 32), (4, 4, 33), (12, 4, 11), (8, 1, 9), (64, 1, 2)])
@pytest.mark.parametrize("Tk", [31, 32, 33, 127, 129, 260])
def test_tile_edges(gpu_pkg, D, Hq, Hkv, Tq, Tk):
    causal = (Tq + Tk) % 2 == 0
    run(gpu_pkg, 1, Hq, Hkv, Tq, Tk, D, causal, "padded" if Tk % 2 else "token_major", Tk + Tq)


@pytest.mark.parametrize("Hq,Hkv,Tq,Tk,D", [(32, 8, 512, 512, 64),     # two groups per CU, folded order
                                            (32, 8, 300, 300, 128),
                                            (8, 8, 1100, 1100, 64),    # folded, units not a power of two apart
                                            (6, 3, 700, 600, 64),      # fully masked leading rows, folded
                                            (16, 16, 700, 700, 64)])   # more than two groups per CU
def test_grid_orders(gpu_pkg, Hq, Hkv, Tq, Tk, D):
    run(gpu_pkg, 2 if Hkv == 3 else 1, Hq, Hkv, Tq, Tk, D, True, "plain", Tq)
