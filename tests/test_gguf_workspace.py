"""Scratch of the projections that read GGUF blocks: the queries cover every shorter call, and a call
whose tile kernel takes no scratch runs without a workspace."""
import ctypes

import numpy as np
import pytest
import torch

import airframe_amd
from airframe_amd import _lib, weights
from tests.gpu_util import Pair, dev, say
from tests.test_gpu_weights import random_blob


def proj_bytes(fmt, n_tok, attn_dim, dim):
    b = ctypes.c_uint64()
    assert airframe_amd.load().ts_attn_out_proj_gguf_workspace(fmt, n_tok, attn_dim, dim, ctypes.byref(b)) == _lib.TS_OK
    return b.value


@pytest.mark.parametrize("fmt", [weights.Q4_K, weights.Q5_0])
@pytest.mark.parametrize("attn_dim,dim", [(4096, 4096), (256, 9), (3072, 5120)])
def test_out_proj_query_covers_shorter_calls(fmt, attn_dim, dim):
    """Long prompts (256 tiles of 32 x 256 and more) need no scratch themselves, but a buffer sized
    for one has to serve the rows of a decode step too."""
    sizes = [proj_bytes(fmt, n, attn_dim, dim) for n in (1, 2, 31, 32, 33, 100, 500, 700, 2048, 9000, 50000)]
    assert sizes == sorted(sizes) and sizes[0] > 0
    # partials of fewer than 512 tiles of 32 x 256 f32, whatever the length
    assert sizes[-1] < 512 * 32 * 256 * 4


def call_proj(fmt, a, w, dim, act, ws):
    L = airframe_amd.load()
    p = ctypes.c_void_p
    return L.ts_attn_out_proj_gguf(p(a.data_ptr()), a.shape[0], a.shape[1], fmt, p(w.data_ptr()), dim,
                                   p(act.data_ptr()), None, p(ws.data_ptr()) if ws is not None else None,
                                   ws.numel() if ws is not None else 0, p(torch.cuda.current_stream().cuda_stream))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [weights.Q4_K, weights.Q8_0])
def test_out_proj_without_workspace(gpu, fmt):
    say(f"out_proj gguf without workspace fmt={fmt}")
    rng = np.random.default_rng(fmt)
    n_tok, attn_dim, dim = 900, 256, 2049  # 29 x 9 tiles
    a = dev(rng.standard_normal((n_tok, attn_dim)).astype(np.float32))
    w = dev(random_blob(rng, fmt, dim, attn_dim))
    ws = torch.empty(proj_bytes(fmt, n_tok, attn_dim, dim), dtype=torch.uint8, device="cuda")
    want, got = torch.zeros((n_tok, dim), device="cuda"), torch.zeros((n_tok, dim), device="cuda")
    assert call_proj(fmt, a, w, dim, want, ws) == _lib.TS_OK
    assert call_proj(fmt, a, w, dim, got, None) == _lib.TS_OK
    torch.cuda.synchronize()
    assert torch.equal(want, got)
    # the same buffer for a short call, which is refused without one
    act = torch.zeros((40, dim), device="cuda")
    assert call_proj(fmt, a[:40], w, dim, act, ws) == _lib.TS_OK
    assert call_proj(fmt, a[:40], w, dim, act, None) == _lib.TS_ERR_WORKSPACE


@pytest.mark.gpu
@pytest.mark.parametrize("hd", [64, 96])
def test_qkv_without_workspace(gpu, hd):
    say(f"qkv gguf without workspace hd={hd}")
    rng = np.random.default_rng(hd)
    fmt, n_seq, n_tok, dim, n_head, n_kv = weights.Q4_0, 70, 120, 256, 2, 1  # 70 x 5 x 2 tiles; hd 96: 263
    p = Pair(n_seq, n_kv, hd, 256, 1e6)
    L, vp = airframe_amd.load(), ctypes.c_void_p
    w = [dev(random_blob(rng, fmt, r, dim)) for r in (n_head * hd, n_kv * hd, n_kv * hd)]

    def need(n):
        b = ctypes.c_uint64()
        assert L.ts_qkv_gguf_workspace(p.gpu.handle, fmt, dim, n, n_head, ctypes.byref(b)) == _lib.TS_OK
        return b.value

    def call(n, ws):
        x = dev(rng.standard_normal((n_seq, n, dim)).astype(np.float32))
        q = torch.empty((n_seq, n, n_head, hd), device="cuda")
        k, v = torch.empty((n_seq, n, n_kv, hd), device="cuda"), torch.empty((n_seq, n, n_kv, hd), device="cuda")

        def run(ws, out):
            return L.ts_qkv_append_gguf(p.gpu.handle, 0, vp(x.data_ptr()), dim, n, fmt, *(vp(t.data_ptr()) for t in w),
                                        n_head, p.rope.handle, vp(out.data_ptr()), vp(k.data_ptr()), vp(v.data_ptr()),
                                        vp(ws.data_ptr()) if ws is not None else None, ws.numel() if ws is not None else 0,
                                        vp(torch.cuda.current_stream().cuda_stream))

        rc = run(ws, q)
        torch.cuda.synchronize()
        return rc, q, run

    sizes = [need(n) for n in (1, 2, 31, 32, 64, 120, 240)]
    assert sizes == sorted(sizes) and sizes[0] > 0
    ws = torch.empty(need(n_tok), dtype=torch.uint8, device="cuda")
    rc, q, run = call(n_tok, ws)
    assert rc == _lib.TS_OK
    q2 = torch.empty_like(q)
    assert run(None, q2) == _lib.TS_OK
    torch.cuda.synchronize()
    assert torch.equal(q, q2)
    for n in (1, 3):  # shorter chunks in the same buffer
        rc, _, run = call(n, ws)
        assert rc == _lib.TS_OK
    assert run(None, torch.empty((n_seq, 3, n_head, hd), device="cuda")) == (
        _lib.TS_OK if hd == 64 else _lib.TS_ERR_WORKSPACE)  # 280 tiles of hd 64; 7 x 1 of hd 96's rows
