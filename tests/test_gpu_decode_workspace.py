"""Which decode calls have to bring a workspace: those whose context, spread evenly, is split, whatever
plan is taken in the end; and batches whose plan has more partials than there is room for."""
import ctypes

import numpy as np
import pytest
import torch

import airframe_amd
from airframe_amd import _lib, synth
from airframe_amd.kv_cache import decode_plan
from tests.gpu_util import Pair, assert_close, dev, say
from tests.test_gpu_decode import prefill_cache

pytestmark = pytest.mark.gpu


def batch(n_seq, n_kv, hd, lens, seed):
    rng = np.random.default_rng(seed)
    p = Pair(n_seq, n_kv, hd, max(lens) + 4, 500000.0)
    # (positions past the first 600 or 100 keep the zeros of a new cache: keys and values of 0 on either side)
    prefill_cache(p, rng, min(600 if n_seq < 100 else 100, max(lens)))
    p.set_lens(np.asarray(lens, np.int32))
    return rng, p


def call(p, fn, q, k, v, n_head, out, ws, nbytes):
    L, vp = airframe_amd.load(), ctypes.c_void_p
    st = vp(torch.cuda.current_stream().cuda_stream)
    tail = (vp(out.data_ptr()), vp(ws), nbytes, st) if fn == "ts_attn_decode_append" else (vp(out.data_ptr()), st)
    return getattr(L, fn)(p.gpu.handle, 0, vp(k.data_ptr()), vp(v.data_ptr()), vp(q.data_ptr()), n_head, p.rope.handle,
                          0.0, *tail)


def step(p, rng, n_kv, G, hd, fn, ws=None, nbytes=0):
    """(status, output, the oracle's output) of one step; the lengths stay."""
    n_seq = p.n_seq
    k, v = synth.normal(rng, (n_seq, 1, n_kv, hd)), synth.normal(rng, (n_seq, 1, n_kv, hd))
    q = synth.normal(rng, (n_seq, n_kv * G, hd))
    out = torch.empty((n_seq, n_kv * G, hd), device="cuda")
    rc = call(p, fn, dev(q), dev(k), dev(v), n_kv * G, out, ws, nbytes)
    torch.cuda.synchronize()
    if rc != _lib.TS_OK:
        return rc, None, None
    p.ora.append(k, v)
    return rc, out.cpu().numpy(), p.ora.attend(q[:, None], 1, threads=8)[:, 0]


def test_split_context_needs_a_workspace(gpu):
    """Streams for every compute unit, some longer than an even share: refused without a workspace also
    where the plan that is taken has no split."""
    say("decode without a workspace: refused")
    lens = np.linspace(700, 1531, 32).astype(int)
    rng, p = batch(32, 8, 128, lens, 1)
    ws = p.gpu.workspace(32)
    assert step(p, rng, 8, 4, 128, "ts_attn_decode_append")[0] == _lib.TS_ERR_WORKSPACE
    assert step(p, rng, 8, 4, 128, "ts_attn_decode_append", ws.data_ptr(), ws.numel() - 16)[0] == _lib.TS_ERR_WORKSPACE
    assert step(p, rng, 8, 4, 128, "ts_attn_decode_append", ws.data_ptr() + 4, ws.numel())[0] == _lib.TS_ERR_INVALID
    rc, out, ref = step(p, rng, 8, 4, 128, "ts_attn_decode_append", ws.data_ptr(), ws.numel())
    assert rc == _lib.TS_OK
    assert_close(out, ref, "with a workspace")


def test_split_context_beyond_the_scratch(gpu):
    """... and refused without allocation where its partials exceed the library's scratch, whatever plan
    a caller's workspace gets."""
    say("noalloc decode beyond the scratch: refused")
    lens = np.linspace(150, 301, 65).astype(int)
    n_cu = torch.cuda.get_device_properties(0).multi_processor_count
    assert n_cu != 256 or decode_plan([int(n) + 1 for n in lens], 8, 64, 256, n_cu)["splits"] == 1
    rng, p = batch(65, 8, 256, lens, 2)
    assert step(p, rng, 8, 8, 256, "ts_attn_decode_append_noalloc")[0] == _lib.TS_ERR_WORKSPACE
    ws = p.gpu.workspace(64)
    rc, out, ref = step(p, rng, 8, 8, 256, "ts_attn_decode_append", ws.data_ptr(), ws.numel())
    assert rc == _lib.TS_OK
    assert_close(out, ref, "with a workspace")


@pytest.mark.parametrize("n_seq,n_kv,G,hd,lo,hi", [
    (16, 8, 4, 128, 4200, 4200),   # equal lengths: one split each, spread evenly
    (104, 16, 8, 256, 215, 264),   # one of 791 among them
    (58, 2, 5, 256, 2376, 2376),   # one split each, spread evenly; the plan has two
    (8, 32, 16, 256, 4071, 4135),  # ... with more partials than the library's scratch holds
])
@pytest.mark.parametrize("fn", ["ts_attn_decode_append", "ts_attn_decode_append_noalloc"])
def test_unsplit_context_needs_none(gpu, fn, n_seq, n_kv, G, hd, lo, hi):
    say(f"{fn} without a workspace n_seq={n_seq} hd={hd}")
    lens = np.linspace(lo, hi, n_seq).round().astype(int)
    if n_seq == 104:
        lens[0] = 791
    n_cu = torch.cuda.get_device_properties(0).multi_processor_count
    splits = decode_plan([int(n) + 1 for n in lens], n_kv, n_kv * G, hd, n_cu)["splits"]
    assert n_cu != 256 or splits == (2 if n_seq in (58, 8) else 1)
    assert n_seq != 8 or splits * n_seq * n_kv * G * (hd + 2) * 4 > 8 << 20
    rng, p = batch(n_seq, n_kv, hd, lens, n_seq)
    rc, out, ref = step(p, rng, n_kv, G, hd, fn)
    assert rc == _lib.TS_OK
    assert_close(out, ref, fn)
