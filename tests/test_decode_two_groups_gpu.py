"""int8 decode at head_dim 64 around the work from which a CU runs two work-groups (5 tiles per wave of 512 groups),
and one segment per CU of equal lengths (256 segments).  Bar: 2e-3 before one output rounding, against the
dequantised cache."""

from __future__ import annotations

import pytest
import torch

from helpers import announce, assert_close, f64
from oracle import attention as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,Hq,Hkv,lens", [
    (8, 32, 8, [5120] * 7 + [4900]),      # 8 waves per unit, 64 segments: just below the line
    (8, 32, 8, [5120] * 7 + [5400]),      # just above it
    (40, 32, 8, [1900, 2100, 7, 0] * 10),
    (64, 32, 8, [1024] * 64),             # one segment per CU: whole segments
    (64, 32, 8, [1009 + i % 16 for i in range(64)]),
    (64, 32, 8, [1024] * 63 + [1025]),
    (512, 4, 1, [33] * 512),              # more segments than CUs
])
@pytest.mark.parametrize("paged", [True, False])
@pytest.mark.parametrize("scales", [torch.float16, torch.float32])
def test_grid(gpu_pkg, B, Hq, Hkv, lens, paged, scales):
    announce(f"two groups B={B} {Hq}/{Hkv} lens={lens[:4]}..{lens[-1]} paged={paged} {scales}")
    P, D = 32, 64
    nb = (max(lens) + P - 1) // P
    S = nb * P
    g = torch.Generator(device=DEV).manual_seed(B + lens[-1])
    codes, sc, ref = [], [], []
    for _ in range(2):
        c = torch.randint(-127, 128, (B, Hkv, S, D), generator=g, device=DEV, dtype=torch.int8)
        s = ((0.5 + torch.rand(B, Hkv, S, generator=g, device=DEV)) / 64).to(scales)
        codes.append(c), sc.append(s), ref.append(f64(c) * f64(s)[..., None])
    q = torch.randn(B, Hq, 1, D, generator=g, device=DEV).to(torch.bfloat16)
    kl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    if paged:
        bt = torch.randperm(B * nb, generator=g, device=DEV).to(torch.int32).view(B, nb)

        def pool(x):   # (B, Hkv, nb, P, ...) -> physical pages in the block table's order
            y = x.unflatten(2, (nb, P)).transpose(1, 2).flatten(0, 1)
            out = torch.empty_like(y, memory_format=torch.contiguous_format)
            out[bt.flatten().long()] = y
            return out
        out = gpu_pkg.paged_gqa_int8_flash_decode(q, pool(codes[0]), pool(codes[1]), pool(sc[0]), pool(sc[1]), bt, kl, P)
    else:
        out = gpu_pkg.attention_flash_decode_int8(q, *codes, *sc, kl)
    torch.cuda.synchronize()
    assert_close(out, O.gqa_decode(f64(q), ref[0], ref[1], lens), 2e-3, "decode")
