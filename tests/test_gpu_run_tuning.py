"""A one-shot run changes its work decomposition while it runs; its samples are
those of a session that keeps one decomposition throughout, bit for bit."""
import numpy as np
import pytest

from ggdmc_amd import workloads as W

pytestmark = pytest.mark.gpu


def _same(a, b):
    for x, y in zip(a, b):
        posts = [(x["phi"], y["phi"])] if x["phi"] is not None else []
        for p, q in posts + list(zip(x["subjects"], y["subjects"])):
            assert np.array_equal(p.theta, q.theta)
            assert np.array_equal(p.summed_log_prior, q.summed_log_prior)
            assert np.array_equal(p.log_likelihoods, q.log_likelihoods)


# iterations: below a launch, the longest run that is not timed, one that times
# some candidates, one that times them all and ends in part of a launch
@pytest.mark.parametrize("nmc,thin", [(12, 1), (96, 2), (100, 3), (211, 5)])
@pytest.mark.parametrize("kw", [{}, {"sweep_groups": 3}, {"sub_migration_prob": 0.1, "pop_migration_prob": 0.1},
                                {"is_pblocked": True}, {"launch_mode": 1}])
def test_one_shot_run_equals_a_fixed_decomposition(gpu, nmc, thin, kw):
    w = W.make("c3", scale=0.1)
    cfg = dict(nmc=nmc, thin=thin, nchain=w.nchain, sweep_groups=2)
    cfg.update(kw)
    got = gpu.run_batch(gpu.make_config(**cfg), w.model, w.jobs)
    cfg.update(launch_mode=1, chains_per_item=4)
    s = gpu.Session(gpu.make_config(**cfg), w.model, w.jobs)
    s.advance(s.total_iters)
    _same(got, s.download())
    s.close()


def test_one_shot_run_of_one_long_subject(gpu):
    # trial tiles are among its candidates
    w = W.make("c1")
    j = w.jobs[0]
    data = gpu.SubjectData.from_cells([np.resize(j.subject.rt[a:b], 4 * (b - a)) for a, b in
                                       zip(j.subject.cell_off[:-1], j.subject.cell_off[1:])])
    job = gpu.JobSpec(gpu.KIND_SUBJECT, 5, j.p_prior, start=j.start, subject=data)
    got = gpu.run_batch(gpu.make_config(600, 18), w.model, [job])
    s = gpu.Session(gpu.make_config(600, 18, launch_mode=1, chains_per_item=9), w.model, [job])
    s.advance(s.total_iters)
    _same(got, s.download())
    s.close()


def test_stored_samples_reach_their_buffers(gpu):
    # transfers of 499 KB a subject go straight to its buffer, of 25 KB through
    # the shared host buffer; 300 fits of 55 KB fill that buffer more than once
    w = W.make("c3", scale=0.1)
    few = gpu.run_batch(gpu.make_config(20, w.nchain), w.model, w.jobs)[0]
    many = gpu.run_batch(gpu.make_config(123, w.nchain), w.model, w.jobs)[0]
    for p, q in zip(few["subjects"] + [few["phi"]], many["subjects"] + [many["phi"]]):
        assert np.array_equal(p.theta, q.theta[:, :, :20])
        assert np.array_equal(p.summed_log_prior, q.summed_log_prior[:, :20])
        assert np.array_equal(p.log_likelihoods, q.log_likelihoods[:, :20])
    w = W.make("c1")
    j = w.jobs[0]
    jobs = [gpu.JobSpec(gpu.KIND_SUBJECT, 100 + r, j.p_prior, start=j.start, subject=j.subject) for r in range(300)]
    cfg = gpu.make_config(64, 18)
    a, b = gpu.run_batch(cfg, w.model, jobs), gpu.run_batch(cfg, w.model, jobs[280:])
    _same(a[280:], b)
    assert len({x["subjects"][0].theta[0, 0, -1] for x in a}) > 100
