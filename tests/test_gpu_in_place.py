"""Projections whose output shares memory with their input (a host that reuses the input's buffer):
one and two rows, where the vector-unit kernel would read x while other workgroups write, and GGUF
prompts of so many tiles that the tile kernel would.  Many more workgroups than run at once, so that
late ones would read what early ones wrote.  Against the oracle's f32 dot within
|err| <= 2e-3 + 1e-3*|ref|."""
import ctypes

import numpy as np
import pytest
import torch

import airframe_amd
from airframe_amd import _lib, weights
from airframe_amd.kv_cache import attn_out_proj, attn_out_proj_gguf
from oracle import oracle
from tests.gpu_util import Pair, assert_close, dev, say
from tests.test_gpu_weights import random_blob

pytestmark = pytest.mark.gpu

BLOCKS = {"q4_k": weights.Q4_K, "q5_0": weights.Q5_0}


def matrix(rng, form, rows, cols):
    if form in BLOCKS:
        blob = random_blob(rng, BLOCKS[form], rows, cols)
        return dev(blob), oracle.dequant(BLOCKS[form], blob, rows * cols).reshape(rows, cols)
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float16)
    return dev(w), w.astype(np.float32)


@pytest.mark.parametrize("form", ["f16", "q4_k", "q5_0"])
@pytest.mark.parametrize("n_tok", [1, 2])
def test_stash_over_input(gpu, form, n_tok):
    say(f"out_proj in place form={form} n_tok={n_tok}")
    rng = np.random.default_rng(n_tok)
    attn_dim, dim = 512, 32768
    w, wf = matrix(rng, form, dim, attn_dim)
    a = rng.standard_normal((n_tok, attn_dim)).astype(np.float32)
    act = torch.zeros((n_tok, dim), dtype=torch.float32, device="cuda")
    stash = torch.empty((n_tok, dim), dtype=torch.float32, device="cuda")
    attn = stash.view(-1)[:n_tok * attn_dim].view(n_tok, attn_dim)
    attn.copy_(dev(a))
    if form in BLOCKS:
        attn_out_proj_gguf(attn, BLOCKS[form], w, dim, act, stash=stash)
    else:
        attn_out_proj(attn, w, act, stash=stash)
    torch.cuda.synchronize()
    dot = oracle.project_f32(a, wf)
    assert_close(act.cpu().numpy(), dot, "act")
    assert_close(stash.cpu().numpy(), dot, "stash")


@pytest.mark.parametrize("form", ["f16", "q4_k"])
def test_q_over_input(gpu, form):
    say(f"qkv in place form={form}")
    rng = np.random.default_rng(3)
    dim, n_head, n_kv, hd = 512, 256, 1, 128
    p = Pair(1, n_kv, hd, 64, 1e6)
    (wq, fq), (wk, fk), (wv, fv) = (matrix(rng, form, r * hd, dim) for r in (n_head, n_kv, n_kv))
    x = rng.standard_normal((1, 1, dim)).astype(np.float32)
    q = torch.empty((1, 1, n_head, hd), dtype=torch.float32, device="cuda")
    k, v = (torch.empty((1, 1, n_kv, hd), dtype=torch.float32, device="cuda") for _ in range(2))
    xd = q.view(-1)[:dim].view(1, 1, dim)
    xd.copy_(dev(x))
    if form in BLOCKS:
        p.gpu.qkv_append_gguf(0, xd, BLOCKS[form], wq, wk, wv, p.rope, q_out=q, kv_out=(k, v))
    else:
        p.gpu.qkv_append(0, xd, wq, wk, wv, p.rope, q_out=q, kv_out=(k, v))
    torch.cuda.synchronize()
    for name, got, wf in (("q", q, fq), ("k", k, fk), ("v", v, fv)):
        assert_close(got.cpu().numpy().reshape(1, -1), oracle.project_f32(x[0], wf), name)


def test_prompt_stash_over_input(gpu):
    """From 256 tiles on the partials need 32 KB a tile; less is refused, nothing written."""
    say("out_proj in place, 514 tiles")
    rng = np.random.default_rng(4)
    fmt, n_tok, dim = weights.Q8_0, 8200, 512
    blob = random_blob(rng, fmt, dim, dim)
    w = dev(blob)
    a = rng.standard_normal((n_tok, dim)).astype(np.float32)
    buf = dev(a)
    act = torch.zeros((n_tok, dim), dtype=torch.float32, device="cuda")
    L, vp = airframe_amd.load(), ctypes.c_void_p

    def call(ws):
        return L.ts_attn_out_proj_gguf(vp(buf.data_ptr()), n_tok, dim, fmt, vp(w.data_ptr()), dim, vp(act.data_ptr()),
                                       vp(buf.data_ptr()), vp(ws.data_ptr()), ws.numel(),
                                       vp(torch.cuda.current_stream().cuda_stream))

    tiles = 257 * 2
    ws = torch.empty(tiles * 32768, dtype=torch.uint8, device="cuda")
    assert call(ws[:-16]) == _lib.TS_ERR_WORKSPACE
    assert call(ws) == _lib.TS_OK
    torch.cuda.synchronize()
    dot = oracle.project_f32(a[-500:], oracle.dequant(fmt, blob, dim * dim).reshape(dim, dim))
    assert_close(act[-500:].cpu().numpy(), dot, "act")
    assert torch.equal(act, buf)
