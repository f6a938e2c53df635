"""Rules of the work splits, on the host."""
import ctypes as C
import os

import pytest

import fixtures as fx

_HOST = os.path.join(fx.ROOT, "tests", "native", "liblba_math_host.so")


def _lib():
    L = C.CDLL(_HOST)
    L.host_iteration_us.restype = C.c_double
    for f in (L.host_iteration_us, L.host_waits_fit):
        f.argtypes = [C.c_int64] + [C.c_int] * 5
    return L


# trials, accumulators, FP64, chain groups, chains per item, ring; whether
# workgroups may wait for one iteration of it (50 ms, an eighth of the bound)
@pytest.mark.parametrize("case,fits", [
    ((768, 2, 0, 2, 1, 0), True),
    ((2048, 4, 0, 2, 17, 0), True),          # a chain group per item: 1.1 ms
    ((16384, 2, 1, 39, 1, 0), True),         # every chain a group: 15 ms
    ((300_000, 2, 0, 2, 1, 0), True),        # 4.7 ms,
    ((300_000, 2, 0, 39, 1, 0), False),      # and with 39 groups in a row 91 ms
    ((300_000, 2, 0, 2, 20, 0), False),      # or 20 chains per item
    ((16384, 2, 1, 2, 1, 39), True),         # a ring of 39 steps: 15 ms
    ((100_608, 4, 1, 2, 1, 33), False),      # 156 ms
])
def test_waits_are_bounded_by_one_iteration(case, fits):
    L = _lib()
    assert bool(L.host_waits_fit(*case)) == fits
    trials, acc, fp64, G, k, ring = case
    rounds = -(-trials // 512)
    want = rounds * 2.0 * acc * (3 if fp64 else 1) * max(G * k, ring)
    assert L.host_iteration_us(*case) == want
    assert fits == (want < 50_000)


def _shape(n, nj, cus=256, may_split=True):
    out = (C.c_int * 4)()
    L = _lib()
    L.host_loglike_shape.argtypes = [C.c_int64, C.c_int, C.c_int64, C.c_int, C.POINTER(C.c_int)]
    L.host_loglike_shape(n, nj, cus, int(may_split), out)
    return list(out)


@pytest.mark.parametrize("n", [1, 3, 33, 64, 130, 200, 256, 257, 400, 511, 512, 520, 8190])
def test_a_split_vector_gives_every_wave_a_chunk(n):
    # off-multiple chunk counts too: 9 or 13 chunks had been split into
    # workgroups of one chunk with three idle waves, 17 into 16 and 1
    for nj in list(range(1, 120)) + [786, 5000]:
        k, threads, jper, stage = _shape(n, nj)
        parts = -(-nj // jper)
        if parts > 1:
            assert k == 1
            if stage:
                assert (threads, jper) == (512, 8) and n * -(-nj // 8) <= 256
            else:
                assert threads == 256 and n < 512 and nj >= 7
                assert 3 <= jper <= 16
                assert jper == -(-nj // parts)      # evenly
        # may not split: whole vectors
        assert -(-nj // _shape(n, nj, may_split=False)[2]) == 1


@pytest.mark.parametrize("n,nj,jper", [(200, 9, 3), (200, 13, 4), (400, 5, 5), (400, 6, 6), (400, 8, 4),
                                       (400, 10, 5), (500, 17, 9), (300, 17, 6), (33, 786, 16), (4, 786, 4),
                                       (511, 33, 11)])
def test_chunks_per_workgroup(n, nj, jper):
    assert _shape(n, nj)[2] == jper
