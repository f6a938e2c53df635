"""The batched path's trial arithmetic where its quick forms hand over: constants
outside their range, times before t0, and pairs of trials sharing a lane."""
import numpy as np
import pytest

import oracle_lib as O
from ggdmc_amd import workloads as W
from ggdmc_amd.model import build_model
from ggdmc_amd.simulate import simulate_subject

pytestmark = pytest.mark.gpu

# the FP32 logarithm contributes up to 1e-8 per trial, a kept evaluation up to
# 1e-5 (the error model's bound); the terms below are of order 1 and more
RTOL = 1e-6


@pytest.mark.parametrize("spec,truth", [(W.C1_SPEC, W.C1_TRUE), (W.C5_SPEC, W.C5_MEAN)])
@pytest.mark.parametrize("ntrial", [1, 63, 64, 65, 127, 128, 129, 300])
def test_mixed_matches_fp64_off_its_quick_range(gpu, spec, truth, ntrial):
    m = build_model(**spec)
    x = np.array([truth[p] for p in m.pnames])
    rng = np.random.default_rng(ntrial)
    full = simulate_subject(m, x, 300, rng)
    keep = np.sort(rng.choice(len(full.rt), ntrial, replace=False))
    off = np.searchsorted(keep, full.cell_off)
    data = gpu.SubjectData(full.rt[keep], off.astype(np.int64))
    th = [x]
    # (a start-point range of 1e-40 is left out: the reference's own quotient by
    # A is rounding noise there)
    for name, v in (("A", -0.3), ("B", -0.5), ("mean_v.true", 0.0), ("mean_v.true", -4.0), ("mean_v.true", 1e31),
                    ("sd_v.true", -0.4), ("sd_v.true", 1e-40)):
        for k, p in enumerate(m.pnames):
            if p.startswith(name):
                y = x.copy()
                y[k] = v
                th.append(y)
    t0 = [k for k, p in enumerate(m.pnames) if p.startswith("t0")]
    for v in (np.median(data.rt), data.rt.min(), 50.0):      # some, one, all trials at t <= 0
        y = x.copy()
        y[t0] = v
        th.append(y)
    th = np.array(th)
    ref = gpu.loglike(m, data, th, gpu.FP64_PLAIN)
    got = gpu.loglike(m, data, th, gpu.MIXED_BATCHED)
    assert np.array_equal(np.isnan(ref), np.isnan(got))
    ok = ~np.isnan(ref)
    assert ok.sum() >= 8
    assert np.allclose(got[ok], ref[ok], rtol=RTOL, atol=RTOL * ntrial)
    # the FP64 form itself: its shared quotients and cut tails against the
    # oracle's (a branch taken wrongly is off by whole units; 1e-9 leaves room
    # for survivors a few ulps of 1 from 0)
    om = O.Model(m.winner, m.par_src, m.par_const, m.npar)
    want = np.array([O.lba_loglike(om, data.rt, data.cell_off, y) for y in th])
    assert np.array_equal(np.isnan(want), np.isnan(ref))
    assert np.allclose(ref[ok], want[ok], rtol=1e-9, atol=1e-9)
