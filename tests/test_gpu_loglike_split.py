"""The work splits of a likelihood call (one workgroup per vector, several
vectors per workgroup, a long subject over many workgroups) give the same bits,
those of the sampler's canonical sums, at the edges of chunks and splits."""
import numpy as np
import pytest

import fixtures as fx

pytestmark = pytest.mark.gpu


def _data(gpu, fix, ntrial):
    """ntrial trials of the fixture's subject, repeated cell by cell."""
    d = fix.sub_data
    cells = [d.rt[d.cell_off[c]:d.cell_off[c + 1]] for c in range(len(d.cell_off) - 1)]
    full = [c for c in range(len(cells)) if len(cells[c])]
    out = [c[:0] for c in cells]
    for i, c in enumerate(full):
        n = ntrial // len(full) + (i < ntrial % len(full))
        out[c] = np.resize(cells[c], n)
    return gpu.SubjectData.from_cells(out)


@pytest.mark.parametrize("precision", ["MIXED_BATCHED", "FP64_PLAIN"])
@pytest.mark.parametrize("ntrial", [1, 127, 129, 1024, 1025, 5000, 35000])
def test_every_split_gives_the_same_bits(gpu, ntrial, precision):
    prec = getattr(gpu, precision)
    fix = fx.load("lba_data6")
    data = _data(gpu, fix, ntrial)
    base = fx.near_thetas(fix, 7, seed=ntrial)
    one = np.array([gpu.loglike(fix.model, data, x[None], prec)[0] for x in base])
    # 300 vectors take another split than one (3 and 31 of up to 5000 trials the
    # same: 8 chunks a workgroup; 31 of 35000 another); 2700 share workgroups
    for n in (3, 31, 300, 2700) if ntrial <= 1025 else (3, 31, 300):
        idx = np.arange(n) % 7
        got = gpu.loglike(fix.model, data, base[idx], prec)
        assert np.array_equal(got, one[idx]), n
        if n <= 300:
            assert np.array_equal(gpu.loglike(fix.model, data, base[idx], prec, noalloc=True), one[idx]), n


def test_fixed_staging_takes_what_it_took_before_the_split(gpu):
    # 16 MiB hold these trials and vectors, but not chunk sums beside them: the
    # call falls back to whole vectors instead of being refused
    fix = fx.load("lba_data6")
    data = _data(gpu, fix, 1_670_000)
    th = fx.near_thetas(fix, 40, seed=1)
    got = gpu.loglike(fix.model, data, th, gpu.MIXED_BATCHED, noalloc=True)
    assert np.array_equal(got, gpu.loglike(fix.model, data, th, gpu.MIXED_BATCHED))


@pytest.mark.parametrize("precision", ["MIXED_BATCHED", "FP64_PLAIN"])
@pytest.mark.parametrize("n,ntrial", [(200, 1100), (200, 1634), (400, 640), (400, 1250), (300, 1793), (500, 2146)])
def test_uneven_splits_give_the_same_bits(gpu, n, ntrial, precision):
    # 9, 13, 10, 15 and 17 chunks over 3, 4, 2, 4 and 2 workgroups, the last of
    # most short of the others; 5 chunks in one
    prec = getattr(gpu, precision)
    fix = fx.load("lba_data6")
    data = _data(gpu, fix, ntrial)
    base = fx.near_thetas(fix, 5, seed=ntrial)
    one = np.array([gpu.loglike(fix.model, data, x[None], prec)[0] for x in base])
    idx = np.arange(n) % 5
    assert np.array_equal(gpu.loglike(fix.model, data, base[idx], prec), one[idx])
    assert np.array_equal(gpu.loglike(fix.model, data, base[idx], prec, noalloc=True), one[idx])
