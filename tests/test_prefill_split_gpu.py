"""GPU parity of the prefill whose keys are split over work-groups (few query rows, many keys).

The library takes that route when the workspace also holds the partials
(``sia_attention_flash_fwd_workspace_size``) and runs the call whole with the
smaller workspace of ``sia_prefill_workspace_size``: the two are compared with
each other and with the float64 oracle.  Bars: the prefill bar of
``helpers.allowed_error`` at 2e-3 against the oracle; between the two routes
(each within 2e-3 of the exact value before its own rounding) twice that.
"""

from __future__ import annotations

import ctypes
from importlib import import_module

import numpy as np
import pytest
import torch

from helpers import allowed_error, announce, assert_close, f64
from oracle import attention as O

DEV = "cuda"


def workspace_sizes(lm, q, k):
    """(bytes of the whole call, bytes with room for the partials) for these tensors."""
    lib = lm.load_library()
    whole, split = ctypes.c_size_t(0), ctypes.c_size_t(0)
    B, Hkv, Tk, D = k.shape
    assert lib.sia_prefill_workspace_size(B, Hkv, Tk, D, ctypes.byref(whole)) == 0
    dq, dk = lm.desc(q), lm.desc(k)
    assert lib.sia_attention_flash_fwd_workspace_size(ctypes.byref(dq), ctypes.byref(dk), ctypes.byref(split)) == 0
    return whole.value, split.value


def whole_call(lm, q, k, v, causal):
    """The call through the C ABI with the whole call's workspace only: never split."""
    lib = lm.load_library()
    n, _ = workspace_sizes(lm, q, k)
    in_place = q.dtype == torch.float16 and q.shape[-1] <= 128
    ws = None if in_place else torch.empty(n, dtype=torch.uint8, device=DEV)
    out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV)
    dq, dk, dv, do = (lm.desc(t) for t in (q, k, v, out))
    rc = lib.sia_attention_flash_fwd(ctypes.byref(dq), ctypes.byref(dk), ctypes.byref(dv), int(causal),
                                     ctypes.c_float(q.shape[-1] ** -0.5), ctypes.byref(do),
                                     None if ws is None else ctypes.c_void_p(ws.data_ptr()),
                                     0 if ws is None else n,
                                     ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert rc == 0, lib.sia_last_error_message()
    return out


def inputs(B, Hq, Hkv, Tq, Tk, D, dtype, layout, seed):
    """q, k, v (B, H, T, D): contiguous, or token-major views and padded rows of larger buffers."""
    g = torch.Generator(device=DEV).manual_seed(seed)

    def t(H, T):
        x = torch.randn(B, H, T, D, generator=g, device=DEV) * 0.5
        if layout == "token_major":
            return x.transpose(1, 2).contiguous().to(dtype).transpose(1, 2)
        if layout == "cache":       # a prefix view of a longer cache with padded rows
            big = torch.zeros(B, H, T + 37, D + 8, dtype=dtype, device=DEV)
            big[:, :, :T, :D] = x.to(dtype)
            return big[:, :, :T, :D]
        return x.to(dtype)

    return t(Hq, Tq), t(Hkv, Tk), t(Hkv, Tk)


def check_all(out, whole, q, k, v, causal, what):
    G = q.shape[1] // k.shape[1]
    qf, kf, vf = (f64(x) for x in (q, k, v))
    for b in range(q.shape[0]):
        for h in range(k.shape[1]):
            ref = O.flash_attention(qf[b:b + 1, h * G:(h + 1) * G], kf[b:b + 1, h:h + 1], vf[b:b + 1, h:h + 1],
                                    causal=causal)
            assert_close(out[b:b + 1, h * G:(h + 1) * G], ref, 2e-3, f"{what} b={b} kv head {h}")
    a, w = f64(out), f64(whole)
    assert (np.abs(a - w) <= 2 * allowed_error(w, out.dtype, 2e-3)).all(), f"{what}: split and whole call differ"


# (B, Hq, Hkv, Tq, Tk): one row; a ragged last block and row group; group sizes 1, 3, 4, 8; rows of a
# causal call that see no key (Tq > Tk); runs that end in a one-key block; a batch
SHAPES = [(1, 4, 1, 2, 1000), (1, 12, 4, 33, 1500), (2, 8, 1, 70, 2113), (1, 4, 4, 129, 900), (1, 2, 2, 700, 577),
          (3, 8, 2, 5, 4097)]


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("causal,layout", [(True, "plain"), (False, "token_major"), (True, "cache")])
def test_split_equals_whole_and_oracle(gpu_pkg, D, dtype, shape, causal, layout):
    lm = import_module("simple-inference-autoresearch_amd._lib")
    B, Hq, Hkv, Tq, Tk = shape
    announce(f"prefill split D={D} {dtype} {shape} causal={causal} {layout}")
    q, k, v = inputs(B, Hq, Hkv, Tq, Tk, D, dtype, layout, seed=D + Tk)
    n_whole, n_split = workspace_sizes(lm, q, k)
    rows = B * Hq * Tq
    assert n_split >= rows * 2 * (D + 2) * 4, "this shape is meant to be split"
    out = gpu_pkg.attention_flash_triton(q, k, v, causal=causal)
    check_all(out, whole_call(lm, q, k, v, causal), q, k, v, causal, f"D={D} {shape} {layout}")
    tm = gpu_pkg.attention_flash_triton(q, k, v, causal=causal, out_token_major=True)
    assert torch.equal(tm.transpose(1, 2), out)


def assert_eight_wave_runs(lm, q, k, runs):
    """These tensors are cut into `runs` runs on variant 4, which needs the V^T images as well as the partials (variant
    3, the 4-wave groups that convert V in LDS, needs the partials alone)."""
    B, Hq, Tq, D = q.shape
    n_whole, n_split = workspace_sizes(lm, q, k)
    assert n_split == n_whole + B * Hq * Tq * runs * (D + 2) * 4, (n_whole, n_split)


@pytest.mark.gpu
@pytest.mark.parametrize("Tq,Tk", [(512, 8192), (500, 6001)])
def test_split_eight_wave_groups(gpu_pkg, Tq, Tk):
    """A prompt chunk wide enough for the 8-wave groups (bf16, head_dim 128) over a long prefix."""
    lm = import_module("simple-inference-autoresearch_amd._lib")
    announce(f"prefill split 8 waves {Tq} {Tk}")
    q, k, v = inputs(1, 32, 8, Tq, Tk, 128, torch.bfloat16, "plain", seed=Tk)
    assert_eight_wave_runs(lm, q, k, 4)
    out = gpu_pkg.attention_flash_triton(q, k, v, causal=True)
    check_all(out, whole_call(lm, q, k, v, True), q, k, v, True, f"8 waves {Tq} {Tk}")


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("table", ["same", "fp32"])
def test_split_rotary_prologue(gpu_pkg, D, dtype, interleaved, table):
    """The split call with q rotated as it is read gives the bits of rope_triton, then the split call."""
    announce(f"prefill split rope D={D} {dtype} interleaved={interleaved} {table}")
    B, Hq, Hkv, T, start = 2, 8, 2, 19, 1480
    q, k, v = inputs(B, Hq, Hkv, T, start + T, D, dtype, "token_major", seed=D)
    rf = gpu_pkg.RopeFrequencies(D, start + T, device=torch.device(DEV))
    cos, sin = rf.get(start + T, dtype=dtype if table == "same" else torch.float32)
    out = gpu_pkg.rope_attention_flash_triton(q, k, v, cos, sin, causal=True, start_offset=start,
                                              interleaved=interleaved)
    qr, _ = gpu_pkg.rope_triton(q.transpose(1, 2), q.transpose(1, 2), cos[start:], sin[start:],
                                interleaved=interleaved)
    assert torch.equal(out, gpu_pkg.attention_flash_triton(qr.transpose(1, 2), k, v, causal=True))


@pytest.mark.gpu
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("table", ["same", "fp32"])
def test_split_eight_wave_rotary_prologue(gpu_pkg, interleaved, table):
    """The same at the prompt chunks and prefixes that run the 8-wave groups (bf16, head_dim 128)."""
    lm = import_module("simple-inference-autoresearch_amd._lib")
    announce(f"prefill split rope 8 waves interleaved={interleaved} {table}")
    T, start, D = 500, 6001, 128
    q, k, v = inputs(1, 32, 8, T, start + T, D, torch.bfloat16, "token_major", seed=start)
    assert_eight_wave_runs(lm, q, k, 4)
    rf = gpu_pkg.RopeFrequencies(D, start + T, device=torch.device(DEV))
    cos, sin = rf.get(start + T, dtype=torch.bfloat16 if table == "same" else torch.float32)
    out = gpu_pkg.rope_attention_flash_triton(q, k, v, cos, sin, causal=True, start_offset=start,
                                              interleaved=interleaved)
    qr, _ = gpu_pkg.rope_triton(q.transpose(1, 2), q.transpose(1, 2), cos[start:], sin[start:],
                                interleaved=interleaved)
    qr = qr.transpose(1, 2)
    check_all(out, whole_call(lm, qr, k, v, True), qr, k, v, True, f"8 waves rope {table}")
    assert torch.equal(out, gpu_pkg.attention_flash_triton(qr, k, v, causal=True))


@pytest.mark.gpu
def test_split_graph_replay(gpu_pkg):
    """Captured in a graph, with other inputs in place at each replay and eager calls between."""
    announce("prefill split graph replay")
    q, k, v = inputs(1, 32, 8, 40, 3000, 128, torch.bfloat16, "plain", seed=3)
    q0, k0, v0 = q.clone(), k.clone(), v.clone()
    gpu_pkg.attention_flash_triton(q0, k0, v0, causal=True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = gpu_pkg.attention_flash_triton(q0, k0, v0, causal=True)
    for i in range(3):
        a, b, c = inputs(1, 32, 8, 40, 3000, 128, torch.bfloat16, "plain", seed=10 + i)
        q0.copy_(a), k0.copy_(b), v0.copy_(c)
        graph.replay()
        ref = gpu_pkg.attention_flash_triton(a, b, c, causal=True)
        torch.cuda.synchronize()
        assert torch.equal(out, ref), i


def test_workspace_sizes_on_the_host():
    """The size function never asks for less than the whole call needs, and refuses what the call refuses."""
    import os
    from conftest import load_pkg
    if not os.path.exists(load_pkg().library_path()):
        pytest.skip("library not built")
    lm = import_module("simple-inference-autoresearch_amd._lib")
    lib = lm.load_library()

    def d(dtype, shape):
        t = lm.SiaTensor()
        t.data, t.dtype, t.ndim = 0x10000, dtype, 4
        for i in range(4):
            t.shape[i] = shape[i]
        return t

    n, m = ctypes.c_size_t(0), ctypes.c_size_t(0)
    for D in (16, 32, 64, 128, 256):
        for Tq, Tk in ((1, 1), (5, 8192), (512, 512), (0, 64), (200, 6200)):
            q, k = d(1, (2, 8, Tq, D)), d(1, (2, 2, Tk, D))
            assert lib.sia_attention_flash_fwd_workspace_size(ctypes.byref(q), ctypes.byref(k), ctypes.byref(n)) == 0
            assert lib.sia_prefill_workspace_size(2, 2, Tk, D, ctypes.byref(m)) == 0
            assert n.value >= m.value
    for dtype in (0, 2):   # float16 up to head_dim 128 and float32: no images
        q, k = d(dtype, (2, 8, 100, 128)), d(dtype, (2, 2, 100, 128))
        assert lib.sia_attention_flash_fwd_workspace_size(ctypes.byref(q), ctypes.byref(k), ctypes.byref(n)) == 0
        assert n.value == 0
    q, k = d(1, (2, 7, 100, 128)), d(1, (2, 2, 100, 128))
    assert lib.sia_attention_flash_fwd_workspace_size(ctypes.byref(q), ctypes.byref(k), ctypes.byref(n)) == -1
    q, k = d(1, (2, 8, 100, 48)), d(1, (2, 2, 100, 48))
    assert lib.sia_attention_flash_fwd_workspace_size(ctypes.byref(q), ctypes.byref(k), ctypes.byref(n)) == -2
