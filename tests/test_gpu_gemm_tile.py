"""The projections' tile kernels (64 rows over the whole reduction) where their tiling can go
wrong: reductions of one to a few 32-long chunks and every remainder of the loop's three
buffers, row counts around the 64-row tile, column counts around the 256-column tile, V blocks
of several ragged sequences inside one row tile (also more than 64 sequences, which the unit
search takes 64 at a time), and two weight planes.  Against the oracle's f32 dot within
|err| <= 2e-3 + 1e-3*|ref|; cache codes bit-exact with the append of the kernel's own K and V."""
import numpy as np
import pytest
import torch

from airframe_amd.kv_cache import attn_out_proj
from oracle import oracle
from tests.gpu_util import Pair, assert_close, dev, say
from tests.test_gpu_qkv import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_seq,n_tok,dim,n_head,n_kv,hd", [
    (5, 40, 64, 8, 2, 128),    # two chunks; units of ragged sequences share a tile
    (3, 33, 128, 4, 4, 64),    # four chunks, hd 64
    (2, 95, 192, 3, 1, 128),   # six chunks, half an empty q tile
    (70, 3, 320, 2, 1, 64),    # more than 64 sequences, ten chunks
    (65, 1, 448, 4, 2, 128),   # decode rows: one past a row tile, fourteen chunks
])
def test_qkv_tiles(gpu, n_seq, n_tok, dim, n_head, n_kv, hd):
    say(f"qkv tiles n_seq={n_seq} n_tok={n_tok} dim={dim} n_head={n_head} n_kv={n_kv} hd={hd}")
    rng = np.random.default_rng(dim + n_tok + n_seq)
    p = Pair(n_seq, n_kv, hd, 100 + 2 * n_tok, 1e6)
    p.set_lens(rng.integers(0, 97, size=n_seq).astype(np.int32))
    run_case(p, rng, n_tok, dim, n_head, x_scale=3.0)
    run_case(p, rng, n_tok, dim, n_head, x_scale=3.0)


@pytest.mark.parametrize("n_tok,attn_dim,dim,planes", [
    (1, 64, 8, 1), (63, 64, 255, 1), (64, 128, 256, 1), (65, 192, 257, 1), (130, 320, 300, 1),
    (70, 64, 260, 2), (65, 192, 40, 2),
])
def test_out_proj_tiles(gpu, n_tok, attn_dim, dim, planes):
    say(f"out_proj tiles n_tok={n_tok} attn_dim={attn_dim} dim={dim} planes={planes}")
    rng = np.random.default_rng(n_tok + attn_dim + dim)
    a = (rng.standard_normal((n_tok, attn_dim)) * 3).astype(np.float32)
    w = (rng.standard_normal((dim, attn_dim)) * 0.02).astype(np.float32)
    hi = w.astype(np.float16)
    lo = (w - hi.astype(np.float32)).astype(np.float16)
    wo = np.concatenate([hi, lo], 1) if planes == 2 else hi
    wf = hi.astype(np.float32) + (lo.astype(np.float32) if planes == 2 else 0)
    act = (rng.standard_normal((n_tok, dim)) * 4).astype(np.float32)
    act_d, stash_d = dev(act), torch.zeros((n_tok, dim), dtype=torch.float32, device="cuda")
    attn_out_proj(dev(a), dev(wo), act_d, stash=stash_d, planes=planes)
    torch.cuda.synchronize()
    dot = oracle.project_f32(a, wf)
    assert_close(stash_d.cpu().numpy(), dot, "projection")
    assert_close(act_d.cpu().numpy(), act + dot, "residual + projection")
