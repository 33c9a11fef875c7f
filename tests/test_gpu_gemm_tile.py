"""The projections' tile kernels (64 rows over the whole reduction) where their tiling can go
wrong: reductions of one to a few 32-long chunks and every remainder of the loop's three
buffers, row counts around the 64-row tile, column counts around the 256-column tile, V blocks
of several ragged sequences inside one row tile (also more than 64 sequences, which the unit
search takes 64 at a time), two weight planes, and GGUF blocks with so many tiles that the tile
kernel takes them (one to three super-blocks).  Against the oracle's f32 dot within
|err| <= 2e-3 + 1e-3*|ref|; cache codes bit-exact with the append of the kernel's own K and V."""
import numpy as np
import pytest
import torch

from airframe_amd import weights
from airframe_amd.kv_cache import attn_out_proj, attn_out_proj_gguf
from oracle import oracle
from tests.gpu_util import Pair, assert_close, dev, say
from tests.test_gpu_qkv import run_case
from tests.test_gpu_weights import random_blob

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


@pytest.mark.parametrize("fmt,n_seq,n_tok,dim,n_head,n_kv,hd", [
    (weights.Q4_K, 70, 3, 256, 2, 1, 64),
    (weights.Q5_K, 65, 3, 768, 2, 1, 64),
    (weights.Q8_0, 70, 35, 512, 2, 1, 64),
    (weights.Q4_0, 33, 100, 256, 4, 2, 128),
    (weights.Q5_0, 70, 5, 512, 3, 1, 128),
    (weights.Q4_K, 420, 1, 512, 64, 8, 64),    # decode rows: the last tile of 4 sequences
    (weights.Q8_0, 550, 1, 256, 32, 8, 128),   # ... of half a tile's units
])
def test_qkv_block_tiles(gpu, fmt, n_seq, n_tok, dim, n_head, n_kv, hd):
    say(f"qkv block tiles fmt={fmt} n_seq={n_seq} n_tok={n_tok} dim={dim} n_head={n_head} n_kv={n_kv} hd={hd}")
    # (more than 256 tiles of 32 rows x 256 columns: the tile kernel takes them)
    rows32 = -(-n_seq // 32) if n_tok == 1 else n_seq * (n_tok // 32 + 2)
    assert rows32 * (-(-n_head * hd // 256) + -(-n_kv * hd // 128)) > 256
    rng = np.random.default_rng(fmt + dim + n_tok)
    p = Pair(n_seq, n_kv, hd, 100 + n_tok, 1e6)
    p.set_lens(rng.integers(0, 97, size=n_seq).astype(np.int32))
    rows = (n_head * hd, n_kv * hd, n_kv * hd)
    blobs = [random_blob(rng, fmt, r, dim) for r in rows]
    x = rng.standard_normal((n_seq, n_tok, dim)).astype(np.float32)
    k_out = torch.empty((n_seq, n_tok, n_kv, hd), dtype=torch.float32, device="cuda")
    v_out = torch.empty_like(k_out)
    q = p.gpu.qkv_append_gguf(0, dev(x), fmt, *(dev(b) for b in blobs), p.rope, kv_out=(k_out, v_out))
    torch.cuda.synchronize()
    q, k_out, v_out = q.cpu().numpy(), k_out.cpu().numpy(), v_out.cpu().numpy()
    xf = x.reshape(-1, dim)
    for name, got, blob, r in (("q", q, blobs[0], rows[0]), ("k", k_out, blobs[1], rows[1]), ("v", v_out, blobs[2], rows[2])):
        ref = oracle.project_f32(xf, oracle.dequant(fmt, blob, r * dim).reshape(r, dim))
        assert_close(got.reshape(n_seq * n_tok, -1), ref, name)
    p.ora.append(k_out, v_out)
    p.advance(n_tok)
    p.check_codes()


@pytest.mark.parametrize("fmt,n_seq,n_tok,hd", [(weights.Q4_K, 70, 35, 64), (weights.Q5_0, 70, 35, 128), (weights.Q8_0, 550, 1, 128)])
def test_qkv_block_tiles_norm(gpu, fmt, n_seq, n_tok, hd):
    """With the QK norm; and without the raw K and V: the same q and cache bits."""
    say(f"qkv block tiles with norm fmt={fmt} n_seq={n_seq} n_tok={n_tok} hd={hd}")
    rng = np.random.default_rng(fmt + hd)
    dim, n_kv = 256, 2 if n_tok > 1 else 8
    n_head = 2 * n_kv
    lens = rng.integers(0, 97, size=n_seq).astype(np.int32)
    norms = [(rng.standard_normal(hd) * 0.4 + 1.0).astype(np.float32) for _ in range(2)]
    w = [dev(random_blob(rng, fmt, r * hd, dim)) for r in (n_head, n_kv, n_kv)]
    x = dev(rng.standard_normal((n_seq, n_tok, dim)).astype(np.float32))
    caches = [Pair(n_seq, n_kv, hd, 100 + n_tok, 1e6) for _ in range(2)]
    for p in caches:
        p.set_lens(lens)
        p.gpu.set_qk_norm(0, dev(norms[0]), dev(norms[1]), 1e-6)
    k_out = torch.empty((n_seq, n_tok, n_kv, hd), dtype=torch.float32, device="cuda")
    v_out = torch.empty_like(k_out)
    q = caches[0].gpu.qkv_append_gguf(0, x, fmt, *w, caches[0].rope, kv_out=(k_out, v_out))
    q2 = caches[1].gpu.qkv_append_gguf(0, x, fmt, *w, caches[1].rope)
    torch.cuda.synchronize()
    assert torch.equal(q, q2)
    ora = caches[0].ora
    ora.q_norm, ora.k_norm, ora.norm_eps = norms[0], norms[1], 1e-6
    ora.append(k_out.cpu().numpy(), v_out.cpu().numpy())
    caches[1].ora = ora
    for p in caches:
        p.gpu.increment(n_tok)
    ora.advance(n_tok)
    for p in caches:
        p.check_codes()


@pytest.mark.parametrize("fmt,n_tok,attn_dim,dim", [
    (weights.Q4_K, 900, 256, 2049), (weights.Q5_K, 8195, 256, 8), (weights.Q8_0, 1030, 512, 1800),
    (weights.Q4_0, 900, 768, 2300), (weights.Q5_0, 830, 256, 2500),
])
def test_out_proj_block_tiles(gpu, fmt, n_tok, attn_dim, dim):
    say(f"out_proj block tiles fmt={fmt} n_tok={n_tok} attn_dim={attn_dim} dim={dim}")
    assert -(-n_tok // 32) * -(-dim // 256) > 256  # the tile kernel takes them
    rng = np.random.default_rng(fmt + n_tok + dim)
    blob = random_blob(rng, fmt, dim, attn_dim)
    a = rng.standard_normal((n_tok, attn_dim)).astype(np.float32)
    act = (rng.standard_normal((n_tok, dim)) * 4).astype(np.float32)
    act_d, stash_d = dev(act), torch.zeros((n_tok, dim), dtype=torch.float32, device="cuda")
    attn_out_proj_gguf(dev(a), fmt, dev(blob), dim, act_d, stash=stash_d)
    torch.cuda.synchronize()
    dot = oracle.project_f32(a, oracle.dequant(fmt, blob, dim * attn_dim).reshape(dim, attn_dim))
    assert_close(stash_d.cpu().numpy(), dot, "projection")
    assert_close(act_d.cpu().numpy(), act + dot, "residual + projection")
