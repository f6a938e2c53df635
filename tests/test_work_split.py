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
