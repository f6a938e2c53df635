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


def _stuck(phi_wgs, subjects, ranges, slots, launches=4):
    """Whether `launches` equal launches, given slots in turn, come to hold them
    all without one subject's items together: segment order is phi_wgs population
    workgroups, then the items, subjects in turn by workgroup id mod 8."""
    left = {x: ranges for x in range(subjects)}
    order = [None] * phi_wgs
    while any(left.values()):
        want = len(order) % 8
        x = next(b for d in range(8) for b in sorted(left) if b % 8 == (want + d) % 8 and left[b])
        left[x] -= 1
        order.append(x)
    held = min(len(order), slots // launches)
    seen = [order[:held].count(x) for x in range(subjects)]
    return held < len(order) and max(seen) < ranges


@pytest.mark.parametrize("phi_wgs,subjects,ranges", [(0, 1, 9), (0, 1, 20), (0, 1, 128), (0, 3, 20), (0, 8, 16),
                                                     (18, 1, 9), (18, 5, 9), (39, 1, 20), (39, 2, 20), (39, 3, 20),
                                                     (39, 4, 20), (33, 5, 17), (7, 12, 4), (48, 1, 24)])
def test_spanning_items_of_several_launches_cannot_stop_each_other(phi_wgs, subjects, ranges):
    L = _lib()
    L.host_span_beside_others.argtypes = [C.c_int64] * 4
    ok = bool(L.host_span_beside_others(phi_wgs, subjects, ranges, 256))
    assert ok == (4 * (phi_wgs + min(8, subjects) * ranges) <= 256)
    if ok:
        assert not any(_stuck(phi_wgs, subjects, ranges, 256, n) for n in (1, 2, 3, 4))


def test_four_small_hierarchical_launches_of_eight_waves_would():
    # what the rule is there for: 3 subjects x 20 ranges, 39 population workgroups
    assert _stuck(39, 3, 20, 256) and not _lib().host_span_beside_others(39, 3, 20, 256)


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
