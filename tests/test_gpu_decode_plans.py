"""Decode under the plans that weigh kernels and split lengths against each other, each shape with the
plan that it is here for: ragged batches of about as many streams as compute units without a
split, an empty sequence among others, short integer splits, longer splits of the 16x16 kernel.
Fused append + decode against the oracle within |err| <= 2e-3 + 1e-3*|ref|, two steps in a row;
codes bit-exact."""
import numpy as np
import pytest
import torch

from airframe_amd import synth
from airframe_amd.kv_cache import decode_plan
from tests.gpu_util import Pair, assert_close, dev, say
from tests.test_gpu_decode import prefill_cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_seq,n_kv,G,hd,lo,hi,want", [
    (32, 8, 4, 128, 700, 1531, ("integer", 1536, 1)),  # spread evenly: two splits for some
    (32, 8, 4, 64, 1000, 3000, ("integer", 3008, 1)),
    (32, 8, 8, 64, 0, 1100, ("integer", 1152, 1)),     # an empty sequence, no split
    (32, 8, 8, 64, 0, 700, ("16x16", 704, 1)),         # ... in a wide workgroup each
    (30, 8, 4, 128, 90, 400, ("16x16", 448, 1)),
    (8, 8, 2, 256, 1000, 4000, ("integer", 1024, 4)),  # the 16x16 kernel's splits before
    (8, 8, 2, 256, 300, 1100, ("16x16", 256, 5)),      # the even plan
    (4, 8, 4, 128, 1500, 3001, ("integer", 512, 6)),
    (1, 8, 3, 128, 9000, 9000, ("integer", 512, 18)),
    (5, 8, 2, 256, 1779, 1779, ("16x16", 512, 4)),     # longer splits of the 16x16 kernel
    (10, 8, 5, 128, 1265, 1265, ("16x16", 448, 3)),
    (2, 8, 8, 96, 30, 2500, ("16x16", 256, 10)),       # the even plan: padded rows, very different lengths
])
def test_weighed_plans(gpu, n_seq, n_kv, G, hd, lo, hi, want):
    say(f"decode plans n_seq={n_seq} n_kv={n_kv} G={G} hd={hd} lo={lo} hi={hi}")
    rng = np.random.default_rng(n_seq + hd + hi)
    p = Pair(n_seq, n_kv, hd, hi + 4, 500000.0)
    prefill_cache(p, rng, hi)
    lens = np.linspace(lo, hi, n_seq).round().astype(np.int32)[rng.permutation(n_seq)]
    p.set_lens(lens)
    n_cu = torch.cuda.get_device_properties(0).multi_processor_count
    plan = decode_plan([int(n) + 1 for n in lens], n_kv, n_kv * G, hd, n_cu)
    assert n_cu != 256 or ("integer" if plan["integer"] else "16x16", plan["chunk"], plan["splits"]) == want
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
