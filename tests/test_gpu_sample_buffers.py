"""A null sample buffer is refused with an error, before anything is written."""
import ctypes as C

import numpy as np
import pytest

from ggdmc_amd import _lib
from ggdmc_amd import runs
from ggdmc_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("field", ["theta", "lp", "ll"])
@pytest.mark.parametrize("level", ["phi", "subject"])
def test_null_sample_buffer_is_refused(gpu, field, level):
    w = W.make("c3", scale=0.1)
    cfg = gpu.make_config(3, w.nchain)
    s = gpu.Session(cfg, w.model, w.jobs)
    s.advance(s.total_iters)
    job = s.batch.cjobs[0]
    # the last of several subjects: their buffers are filled from one transfer
    out = job.phi_out[0] if level == "phi" else job.subject_outs[job.nsubject - 1]
    kept = C.cast(getattr(out, field), C.c_void_p).value
    setattr(out, field, None)
    with pytest.raises(gpu.GgdmcError, match="sample buffer missing"):
        s.download()
    setattr(out, field, C.cast(C.c_void_p(kept), C.POINTER(C.c_double)))
    want = s.download()
    s.close()

    b = runs._Batch(cfg, w.model, w.jobs)
    job = b.cjobs[0]
    out = job.phi_out[0] if level == "phi" else job.subject_outs[job.nsubject - 1]
    kept = C.cast(getattr(out, field), C.c_void_p).value
    setattr(out, field, None)
    with pytest.raises(gpu.GgdmcError, match="sample buffer missing"):
        _lib.check(_lib.lib().ggdmc_run_batch(*b.args()))
    setattr(out, field, C.cast(C.c_void_p(kept), C.POINTER(C.c_double)))
    _lib.check(_lib.lib().ggdmc_run_batch(*b.args()))
    for p, q in zip([want[0]["phi"]] + want[0]["subjects"], [b.results()[0]["phi"]] + b.results()[0]["subjects"]):
        assert np.array_equal(p.theta, q.theta)
        assert np.array_equal(p.summed_log_prior, q.summed_log_prior)
        assert np.array_equal(p.log_likelihoods, q.log_likelihoods)
