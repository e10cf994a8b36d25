"""Split fp32 decode: the merge reads 8 pieces at a time, and a row's dot products are summed across its lanes.

Numbers of pieces around the batch's edges, empty pieces among them, against
the float64 oracle at the fp32 path's bar (max-abs 1e-5 for N(0, 1) inputs).
"""

from __future__ import annotations

import pytest
import torch

from oracle import attention as O
from helpers import announce, assert_close, f64

pytestmark = pytest.mark.gpu
DEV = "cuda"
FP32_TOL = 1e-5


@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("pieces", [2, 7, 8, 9, 17])
def test_pieces(gpu_pkg, D, pieces):
    announce(f"fp32 decode of {pieces} pieces, D={D}")
    B, Hq, Hkv, S = 3, 6, 2, 16 * pieces
    g = torch.Generator(device=DEV).manual_seed(D + pieces)
    q = torch.randn(B, Hq, 1, D, generator=g, device=DEV)
    k, v = (torch.randn(B, Hkv, S, D, generator=g, device=DEV) for _ in range(2))
    lens = [S, 16 * (pieces // 2) + 3, 0]              # every piece, empty pieces behind, no key at all
    kv_len = torch.tensor(lens, dtype=torch.int32, device=DEV)
    with gpu_pkg.decode_options(tiles_per_split=1):
        out = gpu_pkg.attention_flash_decode(q, k, v, kv_len)
    torch.cuda.synchronize()
    assert not out[2].any()
    assert_close(out, O.gqa_decode(f64(q), f64(k), f64(v), lens), FP32_TOL, f"{pieces} pieces D={D}")
