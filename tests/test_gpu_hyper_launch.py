"""Hyper-only runs keep their state in LDS for a launch of up to 256 iterations:
launch boundaries, uneven advances and thinning do not change a bit."""
import numpy as np
import pytest

import fixtures as fx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [{}, {"sub_migration_prob": 0.2}, {"is_pblocked": True}, {"sweep_groups": 9}])
def test_hyper_run_in_pieces_equals_one_run(gpu, kw):
    fix = fx.load("lba_data6")
    P = fix.P
    rng = np.random.default_rng(3)
    X = fx.truth_vector(fix) * np.exp(rng.normal(0, 0.1, (11, P)))
    n = 9
    pp = gpu.PriorSpec.tnorm(np.zeros(P), 10.0)
    hp = gpu.PriorSpec.uniform(2 * P, 0.0, 10.0)
    phi = np.concatenate([X.mean(0), X.std(0) + 0.05])[:, None] * np.exp(rng.normal(0, 0.05, (2 * P, n)))
    from ggdmc_amd import priors
    lp = np.array([priors.sumlogprior(hp, phi[:, c]) for c in range(n)])
    ll = np.array([priors.sumloghlike(pp, phi[:, c], X) for c in range(n)])
    nmc, thin = (300, 2) if not kw.get("is_pblocked") else (140, 2)
    cfg = gpu.make_config(nmc, n, thin=thin, **kw)
    job = [gpu.JobSpec(gpu.KIND_HYPER, 17 + r, pp, h_prior=hp, phi_start=(phi, lp, ll), hyper_data=X)
           for r in range(2)]
    one = gpu.run_batch(cfg, None, job)
    s = gpu.Session(cfg, None, job)
    for k in (1, 2, 255, 256, 257, 1000):
        s.advance(k)
    two = s.download()
    s.close()
    for a, b in zip(one, two):
        assert np.array_equal(a["phi"].theta, b["phi"].theta)
        assert np.array_equal(a["phi"].summed_log_prior, b["phi"].summed_log_prior)
        assert np.array_equal(a["phi"].log_likelihoods, b["phi"].log_likelihoods)
        assert np.unique(a["phi"].theta[0]).size > 10      # the chains move
