"""Projections of one and two rows (decode of one or two sequences), whose kernels give eight lanes
to a weight row: every weight form, reductions of one 256, of fewer and more 256s than the four
waves keep in flight, and longer than the x that LDS holds at a time; row counts that are no
multiple of a workgroup's.  Against the oracle's f32 dot within |err| <= 2e-3 + 1e-3*|ref|; cache
codes bit-exact with the append of the kernel's own K and V."""
import numpy as np
import pytest
import torch

from airframe_amd import weights
from airframe_amd.kv_cache import attn_out_proj, attn_out_proj_gguf
from oracle import oracle
from tests.gpu_util import Pair, assert_close, dev, say
from tests.test_gpu_weights import random_blob

pytestmark = pytest.mark.gpu

PLANES = {"f16": 1, "f16x2": 2}
BLOCKS = {"q4_k": weights.Q4_K, "q5_k": weights.Q5_K, "q8_0": weights.Q8_0, "q4_0": weights.Q4_0, "q5_0": weights.Q5_0}
FORMS = [*PLANES, *BLOCKS]


def matrix(rng, form, rows, cols):
    """(device tensor, f32 values) of a weight matrix."""
    if form in PLANES:
        w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
        hi = w.astype(np.float16)
        if form == "f16":
            return dev(hi), hi.astype(np.float32)
        lo = (w - hi.astype(np.float32)).astype(np.float16)
        return dev(np.concatenate([hi, lo], 1)), hi.astype(np.float32) + lo.astype(np.float32)
    blob = random_blob(rng, BLOCKS[form], rows, cols)
    return dev(blob), oracle.dequant(BLOCKS[form], blob, rows * cols).reshape(rows, cols)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("n_tok,attn_dim,dim", [(1, 256, 9), (1, 1280, 200), (2, 512, 33), (1, 8448, 24), (2, 8448, 17)])
def test_out_proj_rows(gpu, form, n_tok, attn_dim, dim):
    say(f"out_proj rows form={form} n_tok={n_tok} attn_dim={attn_dim} dim={dim}")
    rng = np.random.default_rng(FORMS.index(form) * 7 + attn_dim + dim)
    w, wf = matrix(rng, form, dim, attn_dim)
    a = rng.standard_normal((n_tok, attn_dim)).astype(np.float32)
    act = (rng.standard_normal((n_tok, dim)) * 4).astype(np.float32)
    act_d, stash_d = dev(act), torch.zeros((n_tok, dim), dtype=torch.float32, device="cuda")
    if form in PLANES:
        attn_out_proj(dev(a), w, act_d, stash=stash_d, planes=PLANES[form])
    else:
        attn_out_proj_gguf(dev(a), BLOCKS[form], w, dim, act_d, stash=stash_d)
    torch.cuda.synchronize()
    dot = oracle.project_f32(a, wf)
    assert_close(stash_d.cpu().numpy(), dot, "projection")
    assert_close(act_d.cpu().numpy(), act + dot, "residual + projection")


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("n_seq,dim,n_head,n_kv,hd", [(1, 768, 3, 1, 128), (2, 1280, 4, 2, 64), (1, 512, 2, 1, 96)])
def test_qkv_rows(gpu, form, n_seq, dim, n_head, n_kv, hd):
    say(f"qkv rows form={form} n_seq={n_seq} dim={dim} n_head={n_head} n_kv={n_kv} hd={hd}")
    rng = np.random.default_rng(FORMS.index(form) * 11 + dim)
    p = Pair(n_seq, n_kv, hd, 70, 1e6)
    for start in (0, 31, 62):  # the first, the last and a middle position of a V block
        p.set_lens(np.full(n_seq, start, np.int32))
        (wq, fq), (wk, fk), (wv, fv) = (matrix(rng, form, r, dim) for r in (n_head * hd, n_kv * hd, n_kv * hd))
        x = rng.standard_normal((n_seq, 1, dim)).astype(np.float32)
        k_out = torch.empty((n_seq, 1, n_kv, hd), dtype=torch.float32, device="cuda")
        v_out = torch.empty_like(k_out)
        args = (wq, wk, wv, p.rope)
        if form in PLANES:
            q = p.gpu.qkv_append(0, dev(x), *args, kv_out=(k_out, v_out), planes=PLANES[form])
            q2 = p.gpu.qkv_append(0, dev(x), *args, planes=PLANES[form])  # K and V through the workspace
        else:
            q = p.gpu.qkv_append_gguf(0, dev(x), BLOCKS[form], *args, kv_out=(k_out, v_out))
            q2 = p.gpu.qkv_append_gguf(0, dev(x), BLOCKS[form], *args)
        torch.cuda.synchronize()
        assert torch.equal(q, q2)
        q, k_out, v_out = q.cpu().numpy(), k_out.cpu().numpy(), v_out.cpu().numpy()
        for name, got, wf in (("q", q, fq), ("k", k_out, fk), ("v", v_out, fv)):
            assert_close(got.reshape(n_seq, -1), oracle.project_f32(x[:, 0], wf), name)
        p.ora.append(k_out, v_out)
        p.check_codes(upto=[start + 1] * n_seq)
