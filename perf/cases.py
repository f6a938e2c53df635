"""Timed cases of the engine: calls a program makes through the package's public
entry points, over the range of sizes, designs and options it is used with.

Kinds
  loglike  ggdmc_amd.loglike: summed log-likelihoods of parameter vectors
  fit      ggdmc_amd.run_subject: one single-subject fit, start to stored samples
  hyper    ggdmc_amd.run_hyper: population parameters of fixed subject vectors
  hier     ggdmc_amd.run_batch: one hierarchical run, with `fits` independent
           single-subject fits beside it in the same batch

Designs (ggdmc_amd.workloads): "one" 2 accumulators, 6 parameters, one condition
per stimulus; "bv" 2 accumulators, 13 parameters, 12 conditions; "four"
4 accumulators, 11 parameters, 4 conditions.

Data are simulated from the LBA rule at parameters drawn for the case's seed,
starts lie near them, and start densities are evaluated here in plain FP64.
"""
import math

import numpy as np
import torch

import ggdmc_amd as g
from ggdmc_amd import workloads as W
from ggdmc_amd.model import build_model

PRECISIONS = {"plain": g.FP64_PLAIN, "mixed": g.MIXED_BATCHED, "fp64": g.FP64_BATCHED}
DESIGNS = {"one": (W.C1_SPEC, W.C1_TRUE, None), "bv": (W.BV_SPEC, W.BV_MEAN, W.BV_SCALE),
           "four": (W.C5_SPEC, W.C5_MEAN, W.C5_SCALE)}
NPAR = {"one": 6, "bv": 13, "four": 11}
NACC = {"one": 2, "bv": 2, "four": 4}


def listed():
    return [
        # one likelihood of one subject: a check, an objective inside an optimiser; the smallest call
        {"name": "loglike 1 x 768", "kind": "loglike", "design": "bv", "thetas": 1, "trials": 768,
         "precision": "mixed", "draws": "near"},
        # what initialise_theta asks per round: 16 prior draws for each of 39 chains, reference arithmetic
        {"name": "loglike init 624 x 768", "kind": "loglike", "design": "bv", "thetas": 624, "trials": 768,
         "precision": "plain", "draws": "prior"},
        # the stored draws of one fit scored again (39 chains x 210 columns)
        {"name": "loglike draws 8190 x 768", "kind": "loglike", "design": "bv", "thetas": 8190,
         "trials": 768, "precision": "mixed", "draws": "near"},
        # every chain's vector on one very long data set, 4 accumulators
        {"name": "loglike long 33 x 100608", "kind": "loglike", "design": "four", "thetas": 33,
         "trials": 100608, "precision": "mixed", "draws": "near"},
        # an FP64 audit of a subject's draws, a trial count off every tile
        {"name": "loglike audit 1000 x 2047", "kind": "loglike", "design": "four", "thetas": 1000,
         "trials": 2047, "precision": "plain", "draws": "near"},
        # the plain single-subject fit: 6 parameters, 18 chains, 500 iterations
        {"name": "fit one 18 chains", "kind": "fit", "design": "one", "chains": 18, "trials": 768,
         "nmc": 500, "thin": 1, "migration": 0.0, "precision": "mixed"},
        # burn-in of the 13-parameter fit, with migration, FP64 arithmetic
        {"name": "fit bv burn-in fp64", "kind": "fit", "design": "bv", "chains": 39, "trials": 768,
         "nmc": 250, "thin": 2, "migration": 0.06, "precision": "fp64"},
        # the reference's own arithmetic and chain order
        {"name": "fit one reference order", "kind": "fit", "design": "one", "chains": 18, "trials": 768,
         "nmc": 64, "thin": 1, "migration": 0.0, "precision": "plain"},
        # population parameters of 32 fitted subjects
        {"name": "hyper 32 subjects", "kind": "hyper", "design": "bv", "chains": 39, "subjects": 32,
         "nmc": 500, "thin": 1},
        # the hierarchical benchmark design: 32 subjects x 768 trials
        {"name": "hier 32 x 768", "kind": "hier", "design": "bv", "chains": 39, "subjects": 32,
         "trials_lo": 768, "trials_hi": 768, "fits": 0, "nmc": 125, "thin": 4, "precision": "mixed"},
        # many ragged subjects and independent recovery fits in one batch
        {"name": "hier 256 ragged + 64 fits", "kind": "hier", "design": "bv", "chains": 39, "subjects": 256,
         "trials_lo": 96, "trials_hi": 2048, "fits": 64, "nmc": 19, "thin": 5, "precision": "mixed"},
        # a short run of the largest design: 1024 subjects x 2048 trials, 4 accumulators
        {"name": "hier 1024 x 2048", "kind": "hier", "design": "four", "chains": 33, "subjects": 1024,
         "trials_lo": 2048, "trials_hi": 2048, "fits": 0, "nmc": 3, "thin": 21, "precision": "mixed"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["loglike", "loglike", "loglike", "fit", "fit", "hyper", "hier"])
    design = rng.choice(["one", "bv", "four"])
    if kind == "loglike":
        trials = _log_int(rng, 64, 100608)
        most = max(1, min(8190, 13_000_000 // (trials * NACC[design])))
        return {"kind": kind, "design": design, "thetas": _log_int(rng, 1, most), "trials": trials,
                "precision": rng.choice(["mixed", "mixed", "plain"]),
                "draws": rng.choice(["near", "near", "prior"])}
    chains = rng.choice([3 * NPAR[design], rng.randint(7, 48)])
    if kind == "fit":
        precision = rng.choice(["mixed", "mixed", "fp64", "plain"])
        return {"kind": kind, "design": design, "chains": chains, "trials": _log_int(rng, 64, 4096),
                "nmc": rng.randint(8, 40) if precision == "plain" else _log_int(rng, 16, 400),
                "thin": 1 if precision == "plain" else rng.randint(1, 3),
                "migration": rng.choice([0.0, 0.0, 0.06]), "precision": precision}
    if kind == "hyper":
        return {"kind": kind, "design": design, "chains": chains, "subjects": _log_int(rng, 5, 300),
                "nmc": _log_int(rng, 16, 500), "thin": rng.randint(1, 3)}
    subjects = _log_int(rng, 4, 160)
    precision = rng.choice(["mixed", "mixed", "fp64"])
    most = min(2048, (160_000 if precision == "fp64" else 400_000) // (subjects * NACC[design]))
    lo = _log_int(rng, 96, most)
    return {"kind": kind, "design": design, "chains": chains, "subjects": subjects,
            "trials_lo": lo, "trials_hi": rng.randint(lo, most), "fits": rng.choice([0, 0, 9]),
            "nmc": rng.randint(2, 12), "thin": rng.randint(3, 12), "precision": precision}


# ---------------------------------------------------------------- FP64 densities
def _model(design):
    spec, mean, scale = DESIGNS[design]
    m = build_model(**spec)
    mean = np.array([mean[p] for p in m.pnames])
    scale = np.array([scale[p] for p in m.pnames]) if scale else 0.1 * mean
    return m, mean, scale


def _conditions(m):
    """Stimulus condition of every cell (cell names are '<levels>.<response>')
    and one cell of every condition."""
    names = [c.rsplit(".", 1)[0] for c in m.cell_names]
    order = sorted(set(names))
    return np.array([order.index(x) for x in names]), [names.index(x) for x in order]


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


def _params(m, theta):
    """[..., P] -> [..., condition, accumulator, 6]."""
    _, first = _conditions(m)
    src, cst = _dev(m.par_src[first].astype(np.int64)), _dev(m.par_const[first])
    return torch.where(src >= 0, theta[..., src.clamp(min=0)], cst)


def _ll64(m, theta, rt, cond, win, have):
    """Summed log-likelihoods [S, n] of theta [S, n, P] for subjects' trials
    [S, T] (rt, condition, responding accumulator, whether there is a trial):
    the LBA formula in FP64."""
    par = _params(m, theta)                                   # [S, n, C, J, 6]
    S, n = theta.shape[:2]
    T, J = rt.shape[1], par.shape[3]
    at = cond[:, None, :, None].expand(S, n, T, J)
    A, B, v, s, _, t0 = (par[..., k].gather(2, at) for k in range(6))
    t = rt[:, None, :, None] - t0
    on = t > 0
    t = torch.where(on, t, 1.0)
    zs, chi = t * s, A + B - t * v
    z1, z2 = chi / zs, (chi - A) / zs
    P1, P2 = torch.special.ndtr(z1), torch.special.ndtr(z2)
    dphi = (torch.exp(-0.5 * z2 * z2) - torch.exp(-0.5 * z1 * z1)) / math.sqrt(2 * math.pi)
    den = torch.special.ndtr(v / s).clamp(min=1e-10)
    pdf = torch.where(on, (v * (P1 - P2) + s * dphi) / (A * den), 0.0).clamp(min=1e-10)
    cdf = torch.where(on, (1 + (zs * dphi + (chi - A) * P2 - chi * P1) / A) / den, 0.0).clamp(min=1e-10)
    won = torch.arange(J, device=rt.device) == win[:, None, :, None]
    dens = torch.where(won, pdf, 1 - cdf).prod(-1)
    dens = torch.where(dens > 0, dens, 2.220446049250313e-16)
    return torch.where(have[:, None, :], torch.log(dens), 0.0).sum(-1)


def _tnorm(x, mu, sd):
    """Log density of the normal(mu, sd) truncated to [0, inf)."""
    z = (x - mu) / sd
    mass = torch.special.ndtr(mu / sd)
    return -0.5 * z * z - 0.5 * math.log(2 * math.pi) - torch.log(sd) - torch.log(mass)


# ---------------------------------------------------------------- inputs
def _simulate(m, truth, trials, gen):
    """Trials of S subjects with parameters truth [S, P], trials [S] each,
    spread over the conditions in turn: (rt, condition, response, have) [S, T]."""
    S, T = truth.shape[0], int(max(trials))
    par = _params(m, truth)                                   # [S, C, J, 6]
    C, J = par.shape[1], par.shape[2]
    cond = (torch.arange(T, device="cuda") % C)[None].expand(S, T)
    p = par.gather(1, cond[:, :, None, None].expand(S, T, J, 6))
    A, B, v, s, _, t0 = p.unbind(-1)
    shape = (S, T, J)
    d = v + s * torch.randn(shape, generator=gen, device="cuda", dtype=torch.float64)
    for _ in range(50):                                       # redrawn while none is positive
        bad = ~(d > 0).any(-1, keepdim=True)
        if not bool(bad.any()):
            break
        d = torch.where(bad, v + s * torch.randn(shape, generator=gen, device="cuda", dtype=torch.float64), d)
    u = torch.rand(shape, generator=gen, device="cuda", dtype=torch.float64)
    tt = torch.where(d > 0, t0 + (A + B - u * A) / d, math.inf)
    rt, resp = tt.min(-1)
    have = torch.arange(T, device="cuda")[None] < _dev(np.asarray(trials, np.int64))[:, None]
    return rt, cond, resp, have


def _subjects(m, rt, cond, resp, have):
    """SubjectData of every subject: trials sorted by cell."""
    cell_cond, _ = _conditions(m)
    cell_of = np.empty((cell_cond.max() + 1, m.n_acc), np.int64)
    cell_of[cell_cond, m.winner] = np.arange(m.n_cell)
    cell = _dev(cell_of)[cond, resp]
    cell = torch.where(have, cell, m.n_cell)
    cell, at = torch.sort(cell, dim=1, stable=True)
    rt = rt.gather(1, at).cpu().numpy()
    cell = cell.cpu().numpy()
    out = []
    for s in range(rt.shape[0]):
        off = np.searchsorted(cell[s], np.arange(m.n_cell + 1)).astype(np.int64)
        out.append(g.SubjectData(rt[s, :off[-1]].copy(), off))
    return out


def _near(x, n, gen, spread=0.05):
    """n vectors about every x: [S, P] -> [S, n, P]."""
    z = torch.randn((x.shape[0], n, x.shape[1]), generator=gen, device="cuda", dtype=torch.float64)
    return x[:, None, :] * torch.exp(spread * z)


def _truths(m, mean, scale, S, gen):
    """Subject parameters: truncated normals about the design's values."""
    mu, sd = _dev(mean), _dev(scale)
    x = mu + sd * torch.randn((S, len(mean)), generator=gen, device="cuda", dtype=torch.float64)
    for _ in range(200):
        if not bool((x <= 0).any()):
            break
        y = mu + sd * torch.randn(x.shape, generator=gen, device="cuda", dtype=torch.float64)
        x = torch.where(x > 0, x, y)
    return x


def _lls(m, theta, data):
    """_ll64 in pieces that keep each tensor near 100 MB."""
    S, n = theta.shape[:2]
    cost = n * data[0].shape[1] * m.n_acc
    if S == 1:
        k = max(1, 12_000_000 // (cost // n))
        return torch.cat([_ll64(m, theta[:, i:i + k], *data) for i in range(0, n, k)], 1)
    k = max(1, 12_000_000 // cost)
    return torch.cat([_ll64(m, theta[i:i + k], *(d[i:i + k] for d in data)) for i in range(0, S, k)])


def _state(th, lp, ll):
    return (th.T.cpu().numpy().copy(), lp.cpu().numpy(), ll.cpu().numpy())


def _loglike_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    m, mean, scale = _model(case["design"])
    truth = _truths(m, mean, 0.2 * scale, 1, gen)
    data = _simulate(m, truth, [case["trials"]], gen)
    n = case["thetas"]
    if case["draws"] == "prior":                              # U(0, 10), as the single-subject prior
        th = 10 * torch.rand((1, n, len(mean)), generator=gen, device="cuda", dtype=torch.float64)
    else:
        th = _near(truth, n, gen)
    return m, data, th


def _fit_job(m, data, subject, truth, chains, gen, seed):
    th = _near(truth[None], chains, gen)
    P = th.shape[2]
    lp = torch.full((chains,), -P * math.log(10.0), dtype=torch.float64)
    prior = g.PriorSpec.uniform(P, 0.0, 10.0, m.pnames)
    start = _state(th[0], lp, _lls(m, th, [d[None] for d in data])[0])
    return g.JobSpec(g.KIND_SUBJECT, seed, prior, start=start, subject=subject, nparameter_de=P)


def _population(m, mean, scale, chains, gen):
    x = torch.cat([_dev(mean), _dev(scale)])
    return _near(x[None], chains, gen)[0]                     # [chains, 2P]


def prepare(case, seed):
    """Data, priors and start states a program holds before the call."""
    seed = int(seed)
    if case["kind"] == "loglike":
        m, data, th = _loglike_inputs(case, seed)
        return {"kind": "loglike", "model": m, "data": _subjects(m, *data)[0], "thetas": th[0].cpu().numpy(),
                "precision": PRECISIONS[case["precision"]]}
    gen = torch.Generator(device="cuda").manual_seed(seed)
    m, mean, scale = _model(case["design"])
    P, n = len(mean), case["chains"]
    if case["kind"] == "fit":
        truth = _truths(m, mean, 0.2 * scale, 1, gen)
        data = _simulate(m, truth, [case["trials"]], gen)
        job = _fit_job(m, [d[0] for d in data], _subjects(m, *data)[0], truth[0], n, gen, 9032 + seed)
        cfg = g.make_config(case["nmc"], n, thin=case["thin"], sub_migration_prob=case["migration"],
                            precision=PRECISIONS[case["precision"]])
        return {"kind": "fit", "cfg": cfg, "model": m, "job": job}
    p_prior = g.PriorSpec.tnorm(np.zeros(P), 10.0, 0.0, np.inf, m.pnames)
    h_prior = g.PriorSpec.uniform(2 * P, 0.0, 10.0)
    phi = _population(m, mean, scale, n, gen)
    plp = torch.full((n,), -2 * P * math.log(10.0), dtype=torch.float64)
    truth = _truths(m, mean, scale, case["subjects"], gen)
    if case["kind"] == "hyper":
        pll = _tnorm(truth[:, None], phi[None, :, :P], phi[None, :, P:]).sum((0, 2))
        cfg = g.make_config(case["nmc"], n, thin=case["thin"])
        return {"kind": "hyper", "cfg": cfg, "p_prior": p_prior, "h_prior": h_prior,
                "data": truth.cpu().numpy(), "start": _state(phi, plp, pll), "seed": 9032 + seed}
    trials = torch.randint(case["trials_lo"], case["trials_hi"] + 1, (case["subjects"],), generator=gen,
                           device="cuda").cpu().numpy()
    data = _simulate(m, truth, trials, gen)
    subjects = _subjects(m, *data)
    th = _near(truth, n, gen)
    lp = _tnorm(th, phi[None, :, :P], phi[None, :, P:]).sum(-1)
    ll = _lls(m, th, data)
    pll = _tnorm(th, phi[None, :, :P], phi[None, :, P:]).sum((0, 2))
    th_h, lp_h, ll_h = th.transpose(1, 2).contiguous().cpu().numpy(), lp.cpu().numpy(), ll.cpu().numpy()
    starts = [(th_h[s], lp_h[s], ll_h[s]) for s in range(len(subjects))]
    jobs = [g.JobSpec(g.KIND_HIER, 9032 + seed, p_prior, h_prior=h_prior, phi_start=_state(phi, plp, pll),
                      subjects=subjects, subject_starts=starts, nparameter_de=2 * P)]
    if case["fits"]:
        ft = _truths(m, mean, 0.2 * scale, case["fits"], gen)
        fd = _simulate(m, ft, [768] * case["fits"], gen)
        fs = _subjects(m, *fd)
        jobs += [_fit_job(m, [d[k] for d in fd], fs[k], ft[k], n, gen, 1 + k + seed)
                 for k in range(case["fits"])]
    cfg = g.make_config(case["nmc"], n, thin=case["thin"], precision=PRECISIONS[case["precision"]])
    return {"kind": "hier", "cfg": cfg, "model": m, "jobs": jobs}


# ---------------------------------------------------------------- the calls
def run(state):
    """The call and its results. The posteriors of the subjects come as one
    array each of theta [subject, parameter, chain, column], log priors and
    log-likelihoods [subject, chain, column]."""
    if state["kind"] == "loglike":
        return g.loglike(state["model"], state["data"], state["thetas"], state["precision"])
    if state["kind"] == "fit":
        j = state["job"]
        p = g.run_subject(state["cfg"], state["model"], j.p_prior, j.subject, j.start, j.seed)
        return {"theta": p.theta, "lp": p.summed_log_prior, "ll": p.log_likelihoods}
    if state["kind"] == "hyper":
        p = g.run_hyper(state["cfg"], state["p_prior"], state["h_prior"], state["data"], state["start"],
                        state["seed"])
        return {"theta": p.theta, "lp": p.summed_log_prior, "ll": p.log_likelihoods}
    res = g.run_batch(state["cfg"], state["model"], state["jobs"])
    phi = res[0]["phi"]
    subs = [p for r in res for p in r["subjects"]]
    return {"phi": phi.theta, "phi_lp": phi.summed_log_prior, "phi_ll": phi.log_likelihoods,
            "theta": np.stack([p.theta for p in subs]), "lp": np.stack([p.summed_log_prior for p in subs]),
            "ll": np.stack([p.log_likelihoods for p in subs])}


def _iterations(case):
    return case["nmc"] * case["thin"] - 1


def work(case):
    """One evaluation of a trial under a vector is about 65 operations an
    accumulator (two normal tails, two densities, the products and a log); the
    bytes are trials and starts in, stored columns out, once each."""
    P = NPAR[case["design"]]
    per = 65.0 * NACC[case["design"]]
    if case["kind"] == "loglike":
        n, T = case["thetas"], case["trials"]
        return {"bytes": 8.0 * (T + n * P + n), "flops": per * n * T}
    n, it = case["chains"], _iterations(case)
    stored = 8.0 * n * case["nmc"]
    if case["kind"] == "fit":
        T = case["trials"]
        return {"bytes": 8.0 * T + stored * (P + 2), "flops": per * n * T * it}
    if case["kind"] == "hyper":
        # per chain and parameter: two draws, two prior terms, a likelihood term with its logarithms
        return {"bytes": 8.0 * case["subjects"] * P + stored * (2 * P + 2), "flops": 150.0 * n * P * it}
    S = case["subjects"]
    T = 0.5 * (case["trials_lo"] + case["trials_hi"]) * S + 768 * case["fits"]
    return {"bytes": 8.0 * T + stored * ((S + case["fits"]) * (P + 2) + 2 * P + 2), "flops": per * n * T * it}


def tolerance(case):
    """Likelihoods near the generating values: FP64 sums in another order, or
    the mixed path's terms (its logarithms carry about 1e-8 absolute each, its
    tails 3e-10 relative). At prior draws many survivors 1 - F sit within a few
    ulps of 0, where the last bit of a normal tail decides the term: two FP64
    implementations differ by 4e-4.
    Trajectories: all their numbers follow from accept decisions, which two
    correct evaluations take alike except where a draw falls between their
    acceptance ratios (about one in ten million), after which those chains
    differ by as much as the posterior is wide."""
    if case["kind"] != "loglike":
        return {"rel": 1e-2, "max": 0.99}
    if case["draws"] == "prior":
        return {"rel": 2e-3, "max": 0.1}
    return {"rel": 2e-12, "max": 1e-10} if case["precision"] == "plain" else {"rel": 2e-8, "max": 2e-7}


def exact(case, seed):
    """Likelihoods by the formula in FP64. Trajectories have no value of their
    own apart from the rounding that decides an acceptance; the likelihoods in
    them are the ones that `loglike` gives, bit for bit, and are held to 64
    bits there."""
    if case["kind"] != "loglike":
        return None
    m, data, th = _loglike_inputs(case, seed)
    return _lls(m, th, data)[0].cpu().numpy()
