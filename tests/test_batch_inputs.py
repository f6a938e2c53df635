"""How the arrays of a batch reach the C structures, without a GPU."""
import numpy as np
import pytest

import fixtures as fx
from ggdmc_amd import _lib
from ggdmc_amd.runs import JobSpec, _Batch, make_config


def _job(fix, starts):
    n = 4
    phi = (np.ones((2 * fix.P, n)), np.zeros(n), np.zeros(n))
    return JobSpec(_lib.KIND_HIER, 1, fix.pop_prior, h_prior=fix.hyper_prior, phi_start=phi,
                   subjects=[fix.pop_data(0), fix.pop_data(1)], subject_starts=starts)


def test_start_states_may_come_from_any_iterable():
    fix = fx.load("lba_data6")
    states = [(np.arange(fix.P * 4.0).reshape(fix.P, 4) + s, np.full(4, 0.5 + s), np.full(4, -1.0 - s))
              for s in range(2)]
    for starts in (states, tuple(states), iter(states), zip(*zip(*states))):
        b = _Batch(make_config(3, 4), fix.model, [_job(fix, starts)])
        assert b.cjobs[0].nsubject == 2
        for s, (th, lp, ll) in enumerate(states):
            st = b.cjobs[0].subject_starts[s]
            assert np.array_equal(np.ctypeslib.as_array(st.theta, (4, fix.P)), th.T)
            assert np.array_equal(np.ctypeslib.as_array(st.lp, (4,)), lp)
            assert np.array_equal(np.ctypeslib.as_array(st.ll, (4,)), ll)
    for k in (1, 3):
        with pytest.raises(ValueError):
            _Batch(make_config(3, 4), fix.model, [_job(fix, (states * 2)[:k])])
