"""Decode under the plans that weigh kernels and split lengths against each other: ragged batches of
about as many streams as compute units without a split, the integer kernel in splits of fewer
than four rounds (256-dim rows), long contexts of one sequence, an empty sequence among others.
Fused append + decode against the oracle within |err| <= 2e-3 + 1e-3*|ref|, two steps in a row;
codes bit-exact."""
import numpy as np
import pytest
import torch

from airframe_amd import synth
from tests.gpu_util import Pair, assert_close, dev, say
from tests.test_gpu_decode import prefill_cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_seq,n_kv,G,hd,lo,hi", [
    (30, 8, 4, 128, 90, 400),      # nearly as many streams as compute units: no split
    (32, 8, 8, 64, 0, 700),        # an empty sequence beside splits' ends, no split
    (8, 8, 2, 256, 300, 1100),     # short integer splits on 256-dim rows
    (4, 8, 4, 128, 1500, 3001),
    (1, 8, 3, 128, 9000, 9000),    # one long sequence in integer splits
    (2, 8, 8, 96, 30, 2500),       # padded rows, very different lengths
])
def test_weighed_plans(gpu, n_seq, n_kv, G, hd, lo, hi):
    say(f"decode plans n_seq={n_seq} n_kv={n_kv} G={G} hd={hd} lo={lo} hi={hi}")
    rng = np.random.default_rng(n_seq + hd + hi)
    p = Pair(n_seq, n_kv, hd, hi + 4, 500000.0)
    prefill_cache(p, rng, hi)
    lens = np.linspace(lo, hi, n_seq).round().astype(np.int32)[rng.permutation(n_seq)]
    p.set_lens(lens)
    for step in range(2):
        k = synth.normal(rng, (n_seq, 1, n_kv, hd))
        v = synth.normal(rng, (n_seq, 1, n_kv, hd))
        q = synth.normal(rng, (n_seq, n_kv * G, hd))
        out = p.gpu.attn_decode_append(0, dev(k), dev(v), dev(q), p.rope)
        torch.cuda.synchronize()
        p.ora.append(k, v)
        ref = p.ora.attend(q[:, None], 1, threads=8)[:, 0]
        p.advance(1)
        assert_close(out.cpu().numpy(), ref, f"step {step}")
    p.check_codes()
