"""GGUF projections of exactly 256 tiles of 32 rows x 256 columns, where a long Q4_K reduction keeps
the slices (one each, no split) and every other case takes the tile kernel, and one row tile less
and more.  Against the oracle's f32 dot within |err| <= 2e-3 + 1e-3*|ref|."""
import numpy as np
import pytest
import torch

from airframe_amd import weights
from airframe_amd.kv_cache import attn_out_proj_gguf
from oracle import oracle
from tests.gpu_util import assert_close, dev, say
from tests.test_gpu_weights import random_blob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,attn_dim", [(weights.Q4_K, 2304), (weights.Q4_K, 256), (weights.Q5_K, 2304)])
@pytest.mark.parametrize("n_tok", [8160, 8191, 8193])
def test_out_proj_one_round(gpu, fmt, attn_dim, n_tok):
    say(f"out_proj one round fmt={fmt} attn_dim={attn_dim} n_tok={n_tok}")
    rng = np.random.default_rng(attn_dim + n_tok)
    dim = 9
    blob = random_blob(rng, fmt, dim, attn_dim)
    a = rng.standard_normal((n_tok, attn_dim)).astype(np.float32)
    act_d = torch.zeros((n_tok, dim), dtype=torch.float32, device="cuda")
    attn_out_proj_gguf(dev(a), fmt, dev(blob), dim, act_d)
    torch.cuda.synchronize()
    # the first and last tiles
    pick = np.r_[0:70, n_tok - 70:n_tok]
    dot = oracle.project_f32(a[pick], oracle.dequant(fmt, blob, dim * attn_dim).reshape(dim, attn_dim))
    assert_close(act_d.cpu().numpy()[pick], dot, "projection")
