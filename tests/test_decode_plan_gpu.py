"""Decode batches at the edges of the plan: batch sizes around one wave (64) and the coarse search, empty and
one-token sequences, lengths on both sides of a 16-token tile, shared lengths whose segments are given a whole
number of work-groups, and 2, 4 and 8 waves per unit.  Bar: 2e-3 before one output rounding (int8 K/V the same,
against the dequantised cache)."""

from __future__ import annotations

import pytest
import torch

from helpers import announce, assert_close, f64
from oracle import attention as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def cache(B, Hkv, S, D, kv, g):
    k, v = (torch.randn(B, Hkv, S, D, generator=g, device=DEV) for _ in range(2))
    if kv != "int8":
        dt = torch.bfloat16 if kv == "bf16" else torch.float16
        k, v = k.to(dt), v.to(dt)
        return (k, v), (f64(k), f64(v))
    out, ref = [], []
    for x in (k, v):
        s = x.abs().amax(-1) / 127.0
        c = torch.round(x / s[..., None]).clamp(-127, 127).to(torch.int8)
        out += [c, s.float()]
        ref.append(f64(c) * f64(s)[..., None])
    return (out[0], out[2], out[1], out[3]), tuple(ref)


def check(gpu_pkg, B, Hq, Hkv, D, S, lens, shared, kv, seed):
    announce(f"decode plan B={B} {Hq}/{Hkv} D={D} S={S} {kv} shared={shared} lens={lens[:6]}")
    g = torch.Generator(device=DEV).manual_seed(seed)
    t, (kr, vr) = cache(B, Hkv, S, D, kv, g)
    q = torch.randn(B, Hq, 1, D, generator=g, device=DEV).to(torch.float16 if kv == "fp16" else torch.bfloat16)
    kl = torch.tensor(lens[:1] if shared else lens, dtype=torch.int32, device=DEV)
    f = gpu_pkg.attention_flash_decode_int8 if kv == "int8" else gpu_pkg.attention_flash_decode
    out = f(q, *t, kl)
    torch.cuda.synchronize()
    assert_close(out, O.gqa_decode(f64(q), kr, vr, lens), 2e-3, "decode plan")


@pytest.mark.parametrize("B", [1, 2, 63, 64, 65, 129, 300])
@pytest.mark.parametrize("kv,D", [("bf16", 64), ("fp16", 128), ("int8", 128), ("bf16", 256)])
def test_ragged_batches(gpu_pkg, B, kv, D):
    """Lengths 0, 1, 15, 16, 17, ... in turn: empty sequences at both ends and in runs."""
    some = [0, 1, 15, 16, 17, 0, 0, 33, 150, 31, 32, 0]
    lens = [some[(i * 7 + (i // 12)) % 12] for i in range(B)]
    if B > 2:
        lens[0] = lens[-1] = 0
    check(gpu_pkg, B, 8, 2, D, 160, lens, False, kv, B)


@pytest.mark.parametrize("B,Hq,Hkv", [(1, 4, 1), (3, 8, 4), (8, 32, 8), (24, 32, 8), (5, 6, 6), (9, 64, 4)])
@pytest.mark.parametrize("n", [1, 16, 17, 100, 700, 1009])
@pytest.mark.parametrize("kv,D", [("bf16", 64), ("int8", 128), ("fp16", 256)])
def test_shared_lengths(gpu_pkg, B, Hq, Hkv, n, kv, D):
    check(gpu_pkg, B, Hq, Hkv, D, 1010, [n] * B, True, kv, n)
