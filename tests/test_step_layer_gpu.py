"""Decode steps over a cache's whole pools against the same calls on views cut in Python: equal bit for bit.

Layers other than the first, counted from the end too, and batches smaller
than the cache's, in contiguous and paged caches of both kinds.
"""

from __future__ import annotations

import pytest
import torch

from helpers import announce

pytestmark = pytest.mark.gpu
DEV = "cuda"
Hq, Hkv, D, LAYERS, MAX_B = 8, 2, 64, 3, 4


def inputs(B, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    qkv = torch.randn(B, 1, Hq + 2 * Hkv, D, generator=g, device=DEV).to(torch.bfloat16)
    ang = torch.rand(512, D, generator=g, device=DEV)
    return (*qkv.split([Hq, Hkv, Hkv], dim=2), ang.cos().to(torch.bfloat16), ang.sin().to(torch.bfloat16), g)


def fill(cache, names, g):
    for n in names:
        t = getattr(cache, n)
        x = torch.randn(t.shape, generator=g, device=DEV)
        t.copy_((x * 40).clamp(-127, 127).round() if t.dtype == torch.int8 else x.abs() * 0.02 if "scale" in n else x)


def clone(cache, names):
    return [getattr(cache, n).clone() for n in names]


@pytest.mark.parametrize("cap", [256, 400])            # a 16-bit cache, an int8 one
@pytest.mark.parametrize("layer,B", [(0, 4), (1, 3), (2, 1), (-1, 4), (-3, 2)])
def test_contiguous(gpu_pkg, cap, layer, B):
    announce(f"contiguous step layer={layer} B={B} cap={cap}")
    q, k, v, cos, sin, g = inputs(B, 7 * B + layer)
    cache = gpu_pkg.KVCache(LAYERS, MAX_B, cap, Hkv, D, device=DEV)
    names = ["k_cache", "v_cache"] + (["k_scale", "v_scale"] if cache.is_int8 else [])
    fill(cache, names, g)
    ctx = gpu_pkg.DecodeCtx(D, DEV)
    ctx.set_position(99)
    ref = clone(cache, names)
    views = [t[layer, :B] for t in ref] + [None] * (4 - len(ref))
    q_rot = gpu_pkg.rope_kv_write(q, k, v, cos, sin, *views, start_pos=ctx.pos_index)
    qh = q_rot.transpose(1, 2)
    want = (gpu_pkg.attention_flash_decode_int8(qh, *views, ctx.kv_len) if cache.is_int8
            else gpu_pkg.attention_flash_decode(qh, *views[:2], ctx.kv_len))
    got = gpu_pkg.rope_decode_step_attention(q, k, v, cos, sin, cache, layer, ctx)
    assert torch.equal(got, want)
    for n, t in zip(names, ref):                       # (the other layers and sequences untouched among them)
        assert torch.equal(getattr(cache, n), t), n


@pytest.mark.parametrize("kv_dtype", [torch.bfloat16, torch.int8])
@pytest.mark.parametrize("layer,B", [(0, 4), (1, 3), (-1, 1)])
def test_paged(gpu_pkg, kv_dtype, layer, B):
    announce(f"paged step layer={layer} B={B} {kv_dtype}")
    q, k, v, cos, sin, g = inputs(B, 11 * B + layer)
    cache = gpu_pkg.PagedKVCache(LAYERS, MAX_B, 200, Hkv, D, device=DEV, kv_dtype=kv_dtype)
    cache.allocate(MAX_B, cache.max_blocks_per_seq)
    names = ["k_pool", "v_pool"] + (["k_scale_pool", "v_scale_pool"] if cache.is_int8 else [])
    fill(cache, names, g)
    cache.seq_lens.copy_(torch.tensor([1, 77, 160, 200], dtype=torch.int32))
    ref = clone(cache, names)
    views = [t[layer] for t in ref] + [None] * (4 - len(ref))
    table, lens, P = cache.block_tables[:B], cache.seq_lens[:B], cache.block_size
    want_q = gpu_pkg.rope_kv_write(q, k, v, cos, sin, *views, block_table=table, start_pos=lens, start_offset=-1,
                                   page_size=P)
    qh = want_q.transpose(1, 2)
    want = (gpu_pkg.paged_gqa_int8_flash_decode(qh, *views, table, lens, P) if cache.is_int8
            else gpu_pkg.paged_attention_flash_decode(qh, *views[:2], table, lens, P))
    got_q = cache.write_decode_rope(layer, q, k, v, cos, sin)
    got = cache.decode_attention(layer, got_q.transpose(1, 2))
    assert torch.equal(got_q, want_q) and torch.equal(got, want)
    for n, t in zip(names, ref):
        assert torch.equal(getattr(cache, n), t), n


@pytest.mark.parametrize("layer", [LAYERS, -LAYERS - 1])
def test_layer_out_of_range(gpu_pkg, layer):
    announce(f"layer {layer} of {LAYERS}")
    q, k, v, cos, sin, _ = inputs(1, 0)
    cache = gpu_pkg.KVCache(LAYERS, MAX_B, 256, Hkv, D, device=DEV)
    with pytest.raises(IndexError):
        cache.write_decode_rope(layer, gpu_pkg.DecodeCtx(D, DEV).pos_index, q, k, v, cos, sin)
