"""Work decompositions at the edges of what fits: a candidate that does not fit
is passed over, and no decomposition changes a bit."""
import threading

import numpy as np
import pytest

import fixtures as fx
from ggdmc_amd import priors, workloads
from ggdmc_amd.model import build_model
from ggdmc_amd.simulate import simulate_subject

pytestmark = pytest.mark.gpu


def _thresholds_job(gpu, levels, nchain, per_level, seed=3):
    """Model and single-subject job with one threshold per stimulus: levels + 4
    parameters, levels x 2 condition x accumulator pairs."""
    stim = ["s%d" % i for i in range(levels)]
    m = build_model(p_map={"A": ["1"], "B": ["S"], "t0": ["1"], "mean_v": ["M"], "sd_v": ["1"], "st0": ["1"]},
                    match_map={"M": {s: ("r1", "r2")[i % 2] for i, s in enumerate(stim)}},
                    factors={"S": stim}, constants={"st0": 0.0, "sd_v": 1.0}, accumulators=["r1", "r2"])
    rng = np.random.default_rng(seed)
    x = np.array([{"A": 0.4, "t0": 0.1, "mean_v.true": 3.0, "mean_v.false": 1.0}.get(p, 1.2) for p in m.pnames])
    data = simulate_subject(m, x, per_level, rng)
    prior = gpu.PriorSpec.uniform(m.npar, 0.0, 10.0, m.pnames)
    th = x[:, None] * np.exp(rng.normal(0, 0.03, (m.npar, nchain)))
    lp = np.array([priors.sumlogprior(prior, th[:, c]) for c in range(nchain)])
    ll = gpu.loglike(m, data, th.T.copy(), gpu.FP64_PLAIN)
    return m, gpu.JobSpec(gpu.KIND_SUBJECT, seed, prior, start=(th, lp, ll), subject=data)


def _session(gpu, cfg, m, jobs):
    s = gpu.Session(gpu.make_config(**cfg), m, jobs)
    s.advance(s.total_iters)
    res = s.download()
    s.close()
    return res


def _same(a, b):
    for x, y in zip(a, b):
        for p, q in zip(x["subjects"], y["subjects"]):
            assert np.array_equal(p.theta, q.theta)
            assert np.array_equal(p.summed_log_prior, q.summed_log_prior)
            assert np.array_equal(p.log_likelihoods, q.log_likelihoods)


@pytest.mark.parametrize("precision", ["MIXED_BATCHED", "FP64_BATCHED"])
def test_a_candidate_too_large_for_lds_is_passed_over(gpu, precision):
    # 30 parameters, 90 chains: an item of a whole chain group takes 97 KB of
    # LDS, one chain 26 KB; blocked sweeps rank the former among the candidates
    m, job = _thresholds_job(gpu, 26, 90, 2)
    assert m.npar == 30
    cfg = dict(nmc=67, nchain=90, is_pblocked=True, precision=getattr(gpu, precision))
    got = gpu.run_batch(gpu.make_config(**cfg), m, [job])
    s = gpu.Session(gpu.make_config(**cfg), m, [job])
    assert s.decomposition()[0] != -1
    s.advance(s.total_iters)
    _same(got, s.download())
    s.close()
    _same(got, _session(gpu, dict(cfg, launch_mode=1, chains_per_item=2), m, [job]))


def test_a_launch_may_take_longer_than_the_bound_of_a_wait(gpu):
    # 32 iterations of about 20 ms in one launch: its last segment's workgroup
    # is resident, and waiting, from the start, and the bound of a wait (about
    # 0.4 s) counts from the awaited subject's last iteration
    fix = fx.load("lba_data6")
    cells = [np.resize(fix.sub_data.rt[a:b], 60000 * (b - a) // len(fix.sub_data.rt))
             for a, b in zip(fix.sub_data.cell_off[:-1], fix.sub_data.cell_off[1:])]
    data = gpu.SubjectData.from_cells(cells)
    rng = np.random.default_rng(2)
    th = fx.truth_vector(fix)[:, None] * np.exp(rng.normal(0, 0.02, (fix.P, 39)))
    lp = np.array([priors.sumlogprior(fix.sub_prior, th[:, c]) for c in range(39)])
    job = gpu.JobSpec(gpu.KIND_SUBJECT, 11, fix.sub_prior, subject=data,
                      start=(th, lp, gpu.loglike(fix.model, data, th.T.copy(), gpu.FP64_PLAIN)))
    cfg = dict(nmc=34, nchain=39, sweep_groups=39, precision=gpu.FP64_BATCHED, chains_per_item=1)
    _same(_session(gpu, dict(cfg, launch_mode=4), fix.model, [job]),
          _session(gpu, dict(cfg, launch_mode=1), fix.model, [job]))


@pytest.mark.parametrize("precision", ["MIXED_BATCHED", "FP64_BATCHED"])
@pytest.mark.parametrize("mig", [0.0, 0.2])     # the build for plain crossovers, the general one
def test_the_eight_wave_build_can_be_asked_for(gpu, mig, precision):
    # one subject's fit: the library takes this build by itself, and the
    # decomposition and build a session reports are the ones that give it again
    fix = fx.load("lba_data6")
    th, lp, ll = fx.near_start(fix, 39, seed=8, scale=0.02)
    job = gpu.JobSpec(gpu.KIND_SUBJECT, 3, fix.sub_prior, start=(th, lp, ll), subject=fix.sub_data)
    cfg = dict(nmc=40, nchain=39, sub_migration_prob=mig, precision=getattr(gpu, precision))
    want = _session(gpu, dict(cfg, launch_mode=1, chains_per_item=1), fix.model, [job])
    for k, tpt, mode, w in ((1, 0, 4, 2), (1, 0, 3, 2), (20, 0, 4, 2), (4, 128, 3, 2)):
        s = gpu.Session(gpu.make_config(**cfg, chains_per_item=k, trials_per_tile=tpt, launch_mode=mode,
                                        waves_per_simd=w), fix.model, [job])
        assert s.decomposition()[:2] == (k, tpt) and s.decomposition()[3] == mode
        assert s.waves_per_simd() == 2
        s.advance(s.total_iters)
        _same(want, s.download())
        s.close()
    with pytest.raises(gpu.GgdmcError, match="waves_per_simd"):
        gpu.Session(gpu.make_config(**cfg, chains_per_item=1, launch_mode=2, waves_per_simd=2), fix.model, [job])


def test_the_eight_wave_build_in_a_hierarchical_run(gpu):
    w = workloads.make("c3", scale=0.1)
    for kw in ({}, {"pop_migration_prob": 0.2, "sub_migration_prob": 0.2}, {"is_hblocked": True}):
        cfg = dict(nmc=35, nchain=w.nchain, **kw)
        want = _session(gpu, dict(cfg, launch_mode=1, chains_per_item=4), w.model, w.jobs)
        got = _session(gpu, dict(cfg, launch_mode=4, chains_per_item=1, waves_per_simd=2), w.model, w.jobs)
        _same(want, got)
        assert np.array_equal(want[0]["phi"].theta, got[0]["phi"].theta)
        assert np.array_equal(want[0]["phi"].log_likelihoods, got[0]["phi"].log_likelihoods)


@pytest.mark.parametrize("precision", ["MIXED_BATCHED", "FP64_BATCHED"])
def test_migration_rings_of_tiled_subjects(gpu, precision):
    # 71 chunks: a ring's likelihood takes more chunks at once than a tile has,
    # in two rounds
    fix = fx.load("lba_data6")
    cells = [np.resize(fix.sub_data.rt[a:b], 9000 * (b - a) // len(fix.sub_data.rt))
             for a, b in zip(fix.sub_data.cell_off[:-1], fix.sub_data.cell_off[1:])]
    data = gpu.SubjectData.from_cells(cells)
    assert 64 * 128 < len(data.rt)
    rng = np.random.default_rng(4)
    th = fx.truth_vector(fix)[:, None] * np.exp(rng.normal(0, 0.02, (fix.P, 12)))
    lp = np.array([priors.sumlogprior(fix.sub_prior, th[:, c]) for c in range(12)])
    start = (th, lp, gpu.loglike(fix.model, data, th.T.copy(), gpu.FP64_PLAIN))
    jobs = [gpu.JobSpec(gpu.KIND_SUBJECT, 11 + s, fix.sub_prior, subject=data, start=start) for s in range(2)]
    cfg = dict(nmc=12, nchain=12, sub_migration_prob=0.4, precision=getattr(gpu, precision))
    want = _session(gpu, dict(cfg, launch_mode=1, chains_per_item=2), fix.model, jobs)
    for k, tpt, mode in ((1, 128, 1), (2, 256, 2), (0, 256, 2), (4, 1024, 2), (2, 256, 3)):
        _same(want, _session(gpu, dict(cfg, launch_mode=mode, chains_per_item=k, trials_per_tile=tpt), fix.model, jobs))


def _wide_design(gpu, P, ntrial, seed):
    """256 condition x accumulator pairs and P parameters: thresholds (and
    onsets) by condition, 8 accumulators."""
    nq, na = 32, 8
    src = np.full((nq, na, na, 6), -1, np.int32)       # condition, response, accumulator, family
    cst = np.zeros(src.shape)
    q = np.arange(nq)[:, None, None]
    nb = min(32, P - 4)                                # thresholds; the rest are onsets
    src[..., 0] = 0
    src[..., 1] = 1 + q % nb
    match = (np.arange(nq) % na)[:, None, None] == np.arange(na)[None, None, :]
    src[..., 2] = np.where(match, 1 + nb, 2 + nb)
    cst[..., 3] = 1.0
    src[..., 5] = 3 + nb + q % (P - 3 - nb)
    # (conditions that share every parameter would merge: sd_v tells them apart)
    cst[..., 3] += 1e-3 * q
    m = gpu.LBAModel(np.tile(np.arange(na), nq).astype(np.int32), src.reshape(nq * na, na, 6),
                     cst.reshape(nq * na, na, 6), ["p%d" % i for i in range(P)])
    x = np.full(P, 1.2)
    x[0], x[1 + nb], x[2 + nb] = 0.4, 3.0, 1.0
    x[3 + nb:] = 0.1
    rng = np.random.default_rng(seed)
    data = gpu.SubjectData.from_cells([rng.uniform(0.4, 1.5, ntrial) for _ in range(nq * na)])
    return m, x, data


@pytest.mark.parametrize("P,nchain", [(64, 44), (40, 75), (20, 150)])
def test_the_largest_designs_that_lds_holds(gpu, P, nchain):
    m, x, data = _wide_design(gpu, P, 1, P)
    rng = np.random.default_rng(1)
    prior = gpu.PriorSpec.uniform(P, 0.0, 10.0)

    def job(n):
        th = x[:, None] * np.exp(rng.normal(0, 0.02, (P, n)))
        lp = np.array([priors.sumlogprior(prior, th[:, c]) for c in range(n)])
        return gpu.JobSpec(gpu.KIND_SUBJECT, 7, prior, subject=data,
                           start=(th, lp, gpu.loglike(m, data, th.T.copy(), gpu.FP64_PLAIN)))

    most = job(nchain)
    # (the stored likelihoods are the ones that loglike gives, bit for bit)
    for prec, ll_prec in ((gpu.MIXED_BATCHED, gpu.MIXED_BATCHED), (gpu.FP64_BATCHED, gpu.FP64_PLAIN)):
        cfg = dict(nmc=40, nchain=nchain, precision=prec)
        got = gpu.run_batch(gpu.make_config(**cfg), m, [most])
        _same(got, _session(gpu, dict(cfg, chains_per_item=1, launch_mode=3), m, [most]))
        p = got[0]["subjects"][0]
        moved = np.any(p.theta[:, :, -1] != p.theta[:, :, 0], axis=0)
        assert moved.any()
        ll = gpu.loglike(m, data, p.theta[:, moved, -1].T.copy(), ll_prec)
        assert np.array_equal(ll, p.log_likelihoods[moved, -1])
    plain = gpu.run_batch(gpu.make_config(3, nchain, precision=gpu.FP64_PLAIN), m, [most])[0]["subjects"][0]
    assert np.isfinite(plain.log_likelihoods).all()
    with pytest.raises(gpu.GgdmcError, match="too large for LDS"):
        gpu.run_batch(gpu.make_config(3, nchain + 1), m, [job(nchain + 1)])


def test_sessions_of_several_threads_run_beside_each_other(gpu):
    # four small hierarchical runs at once take the 8-wave build, one workgroup a
    # CU: together more workgroups than the chip holds
    w = workloads.make("c3", scale=0.1)
    assert len(w.jobs[0].subjects) == 3
    jobs = [gpu.JobSpec(j.kind, j.seed + r, j.p_prior, h_prior=j.h_prior, phi_start=j.phi_start, subjects=j.subjects,
                        subject_starts=j.subject_starts, nparameter_de=j.nparameter_de)
            for j in w.jobs for r in range(4)]
    cfg = gpu.make_config(500, w.nchain)
    alone = [gpu.run_batch(cfg, w.model, [j]) for j in jobs]
    got = [None] * 4

    def run(r):
        got[r] = gpu.run_batch(cfg, w.model, [jobs[r]])

    ts = [threading.Thread(target=run, args=(r,)) for r in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for a, b in zip(alone, got):
        _same(a, b)
        assert np.array_equal(a[0]["phi"].theta, b[0]["phi"].theta)
    s = gpu.Session(cfg, w.model, jobs[:1])
    assert not (s.waves_per_simd() == 2 and s.decomposition()[3] == 4)
    s.close()
