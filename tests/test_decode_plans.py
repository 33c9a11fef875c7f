"""The plan of a decode call (kernel, positions per split, splits) through the library's host-only query:
which shapes the weighed plan changes, and to what."""
import ctypes
import time

import pytest

import airframe_amd
from airframe_amd import _lib
from airframe_amd.kv_cache import decode_plan

N_CU = 256


def lens(n_seq, lo, hi):
    """Keys of n_seq sequences spread evenly from lo to hi."""
    return [lo + (hi - lo) * s // max(1, n_seq - 1) for s in range(n_seq)]


def plan(n_seq, n_kv, G, hd, lo, hi):
    p = decode_plan(lens(n_seq, lo, hi), n_kv, n_kv * G, hd, N_CU)
    return ("integer" if p["integer"] else "16x16", p["waves"], p["chunk"], p["splits"])


@pytest.mark.parametrize("shape,want", [
    ((1, 8, 4, 64, 513, 513), ("16x16", 8, 576, 1)),         # a wide workgroup per stream
    ((1, 8, 3, 128, 4172, 4172), ("16x16", 4, 256, 17)),     # short splits, two workgroups a CU
    ((32, 8, 4, 128, 8193, 8193), ("integer", 4, 8256, 1)),  # a workgroup per stream and CU
    ((32, 8, 4, 128, 701, 1532), ("integer", 4, 1536, 1)),   # ragged, about as many streams as CUs: no split
    ((32, 8, 4, 64, 1000, 3000), ("integer", 4, 3008, 1)),
    ((8, 8, 2, 256, 1000, 4000), ("integer", 4, 1024, 4)),
    ((2, 8, 4, 128, 6369, 6369), ("integer", 4, 448, 15)),   # integer splits of less than four rounds
    ((60, 2, 40, 128, 90, 90), ("16x16", 4, 256, 1)),        # more query heads than the integer kernel takes
])
def test_plan(shape, want):
    assert plan(*shape) == want


@pytest.mark.parametrize("n_seq,n_kv,G", [(32, 8, 1), (17, 8, 4), (28, 8, 8), (8, 32, 1), (64, 4, 4), (26, 8, 8)])
@pytest.mark.parametrize("ctx", [961, 1000, 1024])
def test_integer_kernel_keeps_unsplit_streams(n_seq, n_kv, G, ctx):
    """About as many streams as CUs of one round of the integer kernel: the wide workgroups of the 16x16
    kernel take a third longer there."""
    assert plan(n_seq, n_kv, G, 64, ctx, ctx) == ("integer", 4, 1024, 1)


@pytest.mark.parametrize("shape,want", [
    ((16, 8, 4, 64, 3516, 3516), ("integer", 4, 3520, 1)),     # two integer splits for one: 15.2 us, 12.0
    ((10, 8, 8, 64, 1629, 1629), ("integer", 4, 1664, 1)),
    ((6, 2, 16, 128, 18562, 18562), ("integer", 4, 1088, 18)),
    ((8, 8, 4, 64, 11833, 11833), ("integer", 4, 3968, 3)),
    ((2, 8, 4, 128, 2, 7672), ("integer", 4, 704, 11)),        # not in a grid of idle workgroups: 16.0, 13.3
    ((7, 8, 8, 128, 2091, 4182), ("16x16", 4, 384, 11)),       # 22.4, 20.0
    ((6, 4, 12, 128, 2, 9471), ("16x16", 4, 512, 19)),         # 23.5, 20.3
    ((24, 2, 6, 64, 2, 7583), ("16x16", 4, 384, 20)),          # 22.4, 18.3
    ((3, 4, 12, 128, 10409, 10409), ("16x16", 4, 512, 21)),
    ((1, 8, 4, 128, 801, 801), ("16x16", 4, 256, 4)),
])
def test_estimates_too_close_to_decide(shape, want):
    """Shapes that an estimate a little lower had moved to a slower plan."""
    assert plan(*shape) == want


@pytest.mark.parametrize("shape", [(52, 8, 8, 128, 722, 1444), (43, 8, 5, 128, 1322, 1322), (20, 2, 16, 128, 4836, 4836),
                                   (2, 32, 1, 128, 2964, 2964), (14, 1, 8, 128, 15698, 15698)])
def test_integer_kernel_is_not_replaced(shape):
    """The integer kernel's scores are exact before one rounding: where the evenly spread context is its, the 16x16
    kernel (a tenth more error) does not take over."""
    assert plan(*shape)[0] == "integer"


def test_planning_a_large_batch_of_short_sequences_is_cheap():
    """The host sets the pace of such calls, and every layer of a step plans again."""
    L = airframe_amd.load()

    def best(n_seq):
        ctx, out = (ctypes.c_int32 * n_seq)(*[91] * n_seq), (ctypes.c_int32 * 4)()
        times = []
        for _ in range(30):
            t = time.perf_counter()
            for _ in range(50):
                L.ts_attn_decode_plan(ctx, n_seq, 2, 8, 64, N_CU, 1, out)
            times.append(time.perf_counter() - t)
        return min(times)

    # 1.0 and 1.9 us with the call itself; walking the sequences for every candidate 10.4
    assert best(1024) < 4 * best(1)


def test_query_refuses_bad_arguments():
    L = airframe_amd.load()
    i32 = ctypes.c_int32
    ctx, out = (i32 * 2)(5, 9), (i32 * 4)()
    assert L.ts_attn_decode_plan(ctx, 2, 8, 32, 128, N_CU, 1, out) == _lib.TS_OK
    for bad in ((None, 2, 8, 32, 128, N_CU, 1, out), (ctx, 0, 8, 32, 128, N_CU, 1, out), (ctx, 2, 0, 32, 128, N_CU, 1, out),
                (ctx, 2, 8, 31, 128, N_CU, 1, out), (ctx, 2, 8, 32, 260, N_CU, 1, out), (ctx, 2, 8, 32, 60, N_CU, 1, out),
                (ctx, 2, 8, 32, 128, 0, 1, out), (ctx, 2, 8, 32, 128, N_CU, 1, None),
                ((i32 * 2)(0, 9), 2, 8, 32, 128, N_CU, 1, out)):
        assert L.ts_attn_decode_plan(*bad) == _lib.TS_ERR_INVALID
