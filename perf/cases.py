"""The work that programs built on this package have it do, as timed cases.

``listed()`` names twelve cases, ``draw(rng)`` gives further ones of the same ranges, ``prepare`` makes
what a program has in hand before the call, ``run`` makes one pass through the public entry points,
``work`` says what a pass cannot do without and ``exact`` computes a pass's numbers in 64 bits without
this package's kernels (where they are a function of the inputs alone: a nested-sampling run is a random
walk whose draws have no closed form).

Kinds of case:
  sample    the sampler plugin: UniDimSliceSampler.get_samples above a contour of a set of live points
  single    one run and its results: NestedSampler(model, ...)(key), then to_results
  ensemble  many seeds of one model: NestedSampler.run_batch(keys), then every run's log Z
  batch     runs kept on the device and stepped together: DeviceBatch.run, then log Z (as bench.py does)
  mstep     one objective and gradient of evidence maximisation: log_evidence, backward
  evidence  the tree count and evidence statistics of one large sample collection (C ABI)
  loglik    Model.forward and its gradient over a batch of points (C ABI)
"""
import ctypes as C
import math

import numpy as np
import torch

import jaxns_amd as J
from jaxns_amd import _lib
from jaxns_amd import distributions as tfpd
from jaxns_amd._lib import check, lib, ptr, stream_ptr
from jaxns_amd.engine import DeviceBatch, RunSpec
from jaxns_amd.evidence_maximisation import LinearRegressionEvidenceModel, LinRegAdjointStats, log_evidence
from jaxns_amd.samplers import EphemeralState, LivePointCollection

EVALS_PER_SLICE = 2.3  # likelihood evaluations of one slice (first proposal and shrinks) on these problems


def listed():
    return [
        # one new point from the sampler plugin: the smallest call there is, all launch and copy latency
        {"name": "sample-one-mvn-d5", "kind": "sample", "family": "mvn", "D": 5, "N": 200, "n": 1, "s": 5, "lpc": 2,
         "wpb": 2},
        # a single run with default settings, as a user first meets the package (MVN D=10, 300 live points, s=5)
        {"name": "single-mvn-d10", "kind": "single", "family": "mvn", "D": 10, "c": 300, "pe": 0},
        # parameter estimation: the same call with phantom samples and the posterior-peak stopping rule
        {"name": "single-gmm-d4-phantoms", "kind": "single", "family": "gmm", "D": 4, "c": 0, "pe": 1},
        # a likelihood given as a torch callable: the general form, one launch per step
        {"name": "single-callable-d3", "kind": "single", "family": "callable", "D": 3, "c": 100, "pe": 0},
        # an ensemble of seeds of a small model (bench.py's MVN D=10 workload through run_batch)
        {"name": "ensemble-mvn-d10-1024", "kind": "ensemble", "family": "mvn", "D": 10, "c": 300, "R": 1024, "lpc": 2,
         "wpb": 1},
        # bench.py's headline: 1024 runs of MVN D=32, 2048 live points, s=4
        {"name": "batch-mvn-d32-1024", "kind": "batch", "family": "mvn", "D": 32, "N": 2048, "s": 4, "R": 1024,
         "lpc": 4, "wpb": 2},
        # uneven runs: D in 4..64 and 128..1024 live points per run, 4-component mixtures (bench.py's mixture batch)
        {"name": "batch-gmm-uneven-64", "kind": "batch", "family": "gmm", "D": 64, "N": 1024, "s": 5, "R": 64,
         "lpc": 8, "wpb": 1},
        # Bayesian linear regression 4096 x 16, 1024 live points, s=5 (bench.py's regression workload)
        {"name": "batch-linreg-4096x16-16", "kind": "batch", "family": "linreg", "rows": 4096, "D": 16, "N": 1024,
         "s": 5, "R": 16, "lpc": 2, "wpb": 4},
        # one shell of a large regression (bench.py's 65536 x 128 workload, 4096 live points, s=3)
        {"name": "sample-linreg-65536x128", "kind": "sample", "family": "linreg", "rows": 65536, "D": 128, "N": 4096,
         "n": 2048, "s": 3, "lpc": 4, "wpb": 4},
        # the closure of evidence maximisation's M-step over the samples of a run (forward and backward)
        {"name": "mstep-linreg-4096x16", "kind": "mstep", "rows": 4096, "D": 16, "M": 30011, "lpc": 2},
        # results of a long run with phantom samples: tree count and evidence statistics of 2 million samples
        {"name": "evidence-2m", "kind": "evidence", "M": 2000003, "N": 4000, "k": 2},
        # the batched likelihood and its gradient (what a gradient-based program does with Model.forward)
        {"name": "loglik-grad-mvn-d32", "kind": "loglik", "family": "mvn", "D": 32, "B": 400003, "lpc": 4, "wpb": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sample", "sample", "single", "single", "ensemble", "batch", "batch", "mstep", "evidence",
                       "loglik"])
    if kind == "sample":
        if rng.random() < 0.3:
            D, N = rng.randint(20, 128), 2 * _log_int(rng, 64, 2048)
            return {"kind": kind, "family": "linreg", "rows": _log_int(rng, 500, 65536), "D": D, "N": N, "n": N // 2,
                    "s": 3, "lpc": 4 if D > 32 else 2, "wpb": 4}
        N = _log_int(rng, 50, 4000)
        return {"kind": kind, "family": rng.choice(["mvn", "gmm"]), "D": _log_int(rng, 1, 100), "N": N,
                "n": _log_int(rng, 1, max(2, N // 2)), "s": rng.randint(2, 6), "lpc": rng.choice([2, 4]),
                "wpb": rng.choice([1, 2, 4])}
    if kind == "single":
        family = rng.choice(["mvn", "gmm", "callable"])
        if family == "callable":
            return {"kind": kind, "family": family, "D": rng.randint(1, 5), "c": _log_int(rng, 40, 160), "pe": 0}
        if rng.random() < 0.4:  # parameter estimation with its default live points (30 per dimension)
            return {"kind": kind, "family": family, "D": rng.randint(2, 10), "c": 0, "pe": 1}
        D = _log_int(rng, 2, 24 if family == "mvn" else 10)
        return {"kind": kind, "family": family, "D": D, "c": _log_int(rng, 60, 1000), "pe": 0}
    if kind == "ensemble":
        return {"kind": kind, "family": rng.choice(["mvn", "gmm"]), "D": rng.randint(2, 14),
                "c": _log_int(rng, 60, 400), "R": _log_int(rng, 8, 1024), "lpc": rng.choice([2, 4]),
                "wpb": rng.choice([1, 2])}
    if kind == "batch":
        family = rng.choice(["mvn", "gmm", "linreg"])
        if family == "linreg":
            return {"kind": kind, "family": family, "rows": _log_int(rng, 300, 4096), "D": rng.randint(4, 16),
                    "N": _log_int(rng, 150, 1024), "s": 5, "R": rng.randint(2, 16), "lpc": 2, "wpb": 4}
        if family == "gmm":
            return {"kind": kind, "family": family, "D": rng.randint(16, 64), "N": rng.randint(300, 1024), "s": 5,
                    "R": rng.randint(4, 64), "lpc": 8, "wpb": 1}
        return {"kind": kind, "family": family, "D": rng.randint(4, 48), "N": _log_int(rng, 200, 2048), "s": 4,
                "R": _log_int(rng, 8, 300), "lpc": 4, "wpb": 2}
    if kind == "mstep":
        return {"kind": kind, "rows": _log_int(rng, 200, 8192), "D": rng.randint(2, 48), "M": _log_int(rng, 500, 60000),
                "lpc": rng.choice([2, 4])}
    if kind == "evidence":
        return {"kind": kind, "M": _log_int(rng, 3000, 2000000), "N": _log_int(rng, 50, 8000), "k": rng.randint(0, 4)}
    return {"kind": kind, "family": rng.choice(["mvn", "gmm"]), "D": rng.randint(2, 100), "B": _log_int(rng, 100, 400000),
            "lpc": rng.choice([2, 4]), "wpb": rng.choice([1, 2, 4])}


# ----------------------------------------------------------------------------- problems
def _mvn_arrays(D, rng):
    A = rng.normal(size=(D, D))
    return rng.normal(0.0, 0.5, D), A @ A.T / D + 0.05 * np.eye(D)


def _gmm_arrays(D, rng):
    return rng.uniform(-5, 5, size=(4, D)), rng.uniform(0.2, 1.0, size=4)


def _linreg_arrays(rows, D, rng, scaled):
    X = rng.normal(size=(rows, D))
    if scaled:  # 10 % of the columns x 100, as in the large regression workload
        X[:, rng.permutation(D)[:max(1, round(0.1 * D))]] *= 100.0
    sigma = 0.1 if scaled else 0.3
    w = rng.normal(size=D)
    return X, w, X @ w + sigma * rng.normal(size=rows), sigma


def _normal_prior(D):
    def prior_model():
        x = yield J.Prior(tfpd.Normal(loc=np.zeros(D), scale=np.ones(D)), name="x")
        return x
    return prior_model


def _box_prior(D, half):
    def prior_model():
        x = yield J.Prior(tfpd.Uniform(low=-half * np.ones(D), high=half * np.ones(D)), name="x")
        return x
    return prior_model


def _model(family, D, rng, rows=0):
    if family == "mvn":
        mu, cov = _mvn_arrays(D, rng)
        return J.Model(_normal_prior(D), J.MultivariateNormalLikelihood(mu, cov=cov))
    if family == "gmm":
        return J.Model(_box_prior(D, 10.0), J.GaussianMixtureLikelihood(*_gmm_arrays(D, rng)))
    if family == "linreg":
        X, _, y, sigma = _linreg_arrays(rows, D, rng, rows > 20000)
        return J.Model(_normal_prior(D), J.LinearRegressionLikelihood(X, y, sigma=sigma))
    centre = torch.as_tensor(rng.uniform(-1.0, 1.0, D), device="cuda")

    def log_likelihood(x):  # a curved ridge about a centre, batched over the leading axis
        d = x - centre
        return -0.5 * (d * d).sum(-1) / 0.09 - 2.0 * torch.cos(3.0 * d).sum(-1) ** 2

    return J.Model(_box_prior(D, 3.0), log_likelihood)


def _posterior_like_u(rows, D, gen, spread):
    """Points of the unit cube as a run meets them: normal scores, `spread` of the prior's width about a centre."""
    centre = 0.5 * torch.randn(D, generator=gen, device="cuda", dtype=torch.float64)
    z = centre + spread * torch.randn(rows, D, generator=gen, device="cuda", dtype=torch.float64)
    return torch.special.ndtr(z).float().clamp(1e-6, 1.0 - 1e-6)


# ----------------------------------------------------------------------------- prepare
def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed, np.random.default_rng(seed))


def _prepare_sample(case, seed, rng):
    D, N = case["D"], case["N"]
    model = _model(case["family"], D, rng, case.get("rows", 0))
    lik = model.log_likelihood
    # live points as a shell meets them: prior draws and their log-likelihoods, the contour at their median
    U = rng.uniform(1e-4, 1.0 - 1e-4, size=(N, D)).astype(np.float32)
    Ud = torch.from_numpy(U).cuda()
    if case["family"] == "linreg":
        W = torch.special.ndtri(Ud.double())
        R = torch.from_numpy(lik.y).cuda()[None, :]
        X = torch.from_numpy(lik.X).cuda()
        L = torch.cat([lik.log_const - 0.5 * ((R - w @ X.T) ** 2).sum(1) / lik.sigma ** 2 for w in W.split(512)])
    else:
        L = lik.torch_log_prob(model.likelihood_inputs_torch(Ud)[0])
    L = L.cpu().numpy()
    live = LivePointCollection(sender_node_idx=np.zeros(N, np.int32), U_sample=U, log_L_constraint=np.full(N, -np.inf),
                               log_L=L, num_likelihood_evaluations=np.ones(N, np.int32))
    sampler = J.UniDimSliceSampler(model, num_slices=case["s"] * D, num_phantom_save=0, midpoint_shrink=True,
                                   lanes_per_chain=case["lpc"], waves_per_block=case["wpb"])
    state = sampler.pre_process(EphemeralState(key=seed, live_points_collection=live))
    return {"kind": "sample", "sampler": sampler, "state": state, "contour": float(np.median(L)), "key": (seed, 3),
            "n": case["n"]}


def _prepare_single(case, seed, rng):
    model = _model(case["family"], case["D"], rng)
    ns = J.NestedSampler(model, num_live_points=case["c"] or None, s=5, parameter_estimation=bool(case["pe"]),
                         max_samples=None if not case["c"] else 50 * case["c"])
    # the program's own arrays, which each run's results go into (a run's length varies from seed to seed)
    most, D = ns._spec(0).max_samples, case["D"]
    arrays = {k: np.full((most, D), np.nan) for k in ("samples", "U")}
    arrays.update({k: np.full(most, np.nan) for k in ("log_L", "log_dp", "log_X", "log_post")})
    arrays.update({k: np.zeros(most, np.int64) for k in ("num_live", "evals")})
    return {"kind": "single", "ns": ns, "key": seed, "arrays": arrays}


def _prepare_ensemble(case, seed, rng):
    model = _model(case["family"], case["D"], rng)
    ns = J.NestedSampler(model, num_live_points=case["c"], s=5, lanes_per_chain=case["lpc"],
                         waves_per_block=case["wpb"])
    return {"kind": "ensemble", "ns": ns, "keys": [1000 * seed + i for i in range(case["R"])]}


def _prepare_batch(case, seed, rng):
    specs = []
    model = None
    sizes = np.random.default_rng(case["R"])  # the runs' sizes belong to the case, their problems to the seed
    for r in range(case["R"]):
        D, N = case["D"], case["N"]
        if case["family"] == "gmm":  # every run a mixture and size of its own
            D = int(sizes.integers(4, D + 1)) if r else D
            N = int(sizes.integers(128, N + 1)) if r else N
            model = _model("gmm", D, rng)
        elif model is None:
            model = _model(case["family"], D, rng, case.get("rows", 0))
        length = {"mvn": 45, "gmm": 300, "linreg": 200}[case["family"]]
        specs.append(RunSpec(model=model, num_live_points=N, num_slices=case["s"] * D, k_phantom=0,
                             max_samples=N * length, seed=1000 * seed + r))
    batch = DeviceBatch(specs, lanes_per_chain=case["lpc"], waves_per_block=case["wpb"])
    term = dict(dlogZ=math.log(1.0 + 1e-3), max_samples=float(max(s.max_samples for s in specs)))
    return {"kind": "batch", "batch": batch, "term": term}


def _mstep_arrays(case, rng):
    X, w, y, sigma = _linreg_arrays(case["rows"], case["D"], rng, False)
    # samples along a run's way to the posterior: spreads from the prior's width down to the posterior's
    M, D = case["M"], case["D"]
    width = sigma / math.sqrt(case["rows"])
    scale = np.exp(np.linspace(0.0, math.log(width), M))
    from scipy.special import ndtr
    U = np.clip(ndtr(w[None, :] + scale[:, None] * rng.normal(size=(M, D))), 1e-6, 1 - 1e-6).astype(np.float32)
    log_w = D * np.log(scale) - 0.5 * D * math.log(2.0 * math.pi) - math.log(M)
    return X, y, U, log_w, np.array([math.log(sigma) + 0.1, 0.2])


def _prepare_mstep(case, seed, rng):
    X, y, U, log_w, theta = _mstep_arrays(case, rng)
    family = LinearRegressionEvidenceModel(J.RegressionData(X, y))
    return {"kind": "mstep", "stats": LinRegAdjointStats(family, U, lanes_per_chain=case["lpc"]),
            "log_w": torch.from_numpy(log_w).cuda(),
            "theta": torch.tensor(theta, dtype=torch.float64, device="cuda", requires_grad=True)}


def _collection(case, seed):
    """A run's sample collection: shells of N // 2 points in ascending log L, each sent by the node below
    its contour, followed by its phantoms (k per chain, anywhere above the contour); the live points last."""
    M, N, k = case["M"], case["N"], case["k"]
    S = max(1, N // 2)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    block = S * (1 + k)
    i = torch.arange(M, device="cuda")
    shell, pos = i // block, i % block
    # log X falls by about S / N a shell; log L = -X^(2/8) of an 8-dimensional Gaussian peak, widths apart
    within = torch.rand(M, generator=gen, device="cuda", dtype=torch.float64)
    fall = S / N * torch.where(pos < S, (pos + within) / S, 1.0 + 2.0 * within)
    log_X = -(shell * (S / N) + fall)
    log_L = -50.0 * torch.exp(log_X / 4.0)
    sender = torch.clamp((shell - 1) * block + S - 1, min=0).to(torch.int32)
    return log_L, sender


def _prepare_evidence(case, seed, rng):
    M = case["M"]
    log_L, sender = _collection(case, seed)
    dev = dict(device="cuda")
    return {"kind": "evidence", "M": M, "log_L": log_L, "sender": sender,
            "idx": torch.empty(M, dtype=torch.int64, **dev), "nl": torch.empty(M, dtype=torch.int64, **dev),
            "per8": torch.empty((8, M), dtype=torch.float64, **dev), "fin": torch.empty(8, dtype=torch.float64, **dev),
            "ws1": torch.empty(int(lib().hipns_count_crossed_edges_workspace_size(M)), dtype=torch.uint8, **dev),
            "ws2": torch.empty(int(lib().hipns_evidence_scan_workspace_size(M)), dtype=torch.uint8, **dev)}


def _loglik_points(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return _posterior_like_u(case["B"], case["D"], gen, 0.7)


def _prepare_loglik(case, seed, rng):
    D, B = case["D"], case["B"]
    model = _model(case["family"], D, rng)
    batch = DeviceBatch([RunSpec(model=model, num_live_points=64, num_slices=5 * D, max_samples=6400)],
                        lanes_per_chain=case["lpc"], waves_per_block=case["wpb"])
    U = torch.full((B, batch.dps), 0.5, dtype=torch.float32, device="cuda")
    U[:, :D] = _loglik_points(case, seed)
    return {"kind": "loglik", "batch": batch, "U": U, "D": D, "B": B,
            "log_L": torch.empty(B, dtype=torch.float64, device="cuda"),
            "log_L_grad": torch.empty(B, dtype=torch.float64, device="cuda"),
            "grad": torch.zeros((B, batch.dps), dtype=torch.float32, device="cuda")}


_PREPARE = {"sample": _prepare_sample, "single": _prepare_single, "ensemble": _prepare_ensemble,
            "batch": _prepare_batch, "mstep": _prepare_mstep, "evidence": _prepare_evidence,
            "loglik": _prepare_loglik}


# ----------------------------------------------------------------------------- run
def run(state):
    return _RUN[state["kind"]](state)


def _run_sample(st):
    s, ph = st["sampler"].get_samples(st["key"], st["contour"], st["state"], st["n"])
    return {"U": s.U_sample, "log_L": s.log_L, "evals": s.num_likelihood_evaluations}


def _run_single(st):
    reason, state = st["ns"](st["key"])
    r = st["ns"].to_results(reason, state)
    found = {"samples": r.samples["x"], "U": r.U_samples, "log_L": r.log_L_samples, "log_dp": r.log_dp_mean,
             "log_X": r.log_X_mean, "log_post": r.log_posterior_density, "num_live": r.num_live_points_per_sample,
             "evals": r.num_likelihood_evaluations_per_sample}
    for k, v in found.items():
        st["arrays"][k][:len(v)] = v
    return {**st["arrays"], "log_Z": r.log_Z_mean, "log_Z_uncert": r.log_Z_uncert, "ESS": r.ESS, "H": r.H_mean,
            "num_samples": int(r.total_num_samples), "phantoms": int(r.total_phantom_samples),
            "reason": int(r.termination_reason)}


def _batch_outputs(batch):
    """log Z of every run and the sample collections (entries past a run's last sample hold the defaults),
    with the final live points."""
    log_Z = batch.log_Z()
    return {"log_Z": log_Z, "log_L": batch.samp_logL, "sender": batch.samp_sender, "evals": batch.samp_evals,
            "live_U": list(batch.live_U), "live_log_L": list(batch.live_logL)}


def _run_ensemble(st):
    reasons, states = st["ns"].run_batch(st["keys"])
    return {"reasons": np.array(reasons), **_batch_outputs(states[0].batch)}


def _run_batch(st):
    st["batch"].run(st["term"], init_efficiency_threshold=0.1, graph_iters=8)
    return _batch_outputs(st["batch"])


def _run_mstep(st):
    theta = st["theta"]
    theta.grad = None
    log_Z = log_evidence(theta, st["stats"], st["log_w"])
    log_Z.backward()
    return {"log_Z": log_Z.detach(), "grad": theta.grad}


def _run_evidence(st):
    M, s = st["M"], stream_ptr()
    check(lib().hipns_count_crossed_edges(ptr(st["sender"]), ptr(st["log_L"]), M, -1, ptr(st["idx"]), ptr(st["nl"]),
                                          ptr(st["ws1"]), st["ws1"].numel(), s), "hipns_count_crossed_edges")
    log_L = st["log_L"].index_select(0, st["idx"])
    n = st["nl"].to(torch.float64)
    check(lib().hipns_evidence_scan(ptr(log_L), ptr(n), M, -1, ptr(st["per8"]), ptr(st["fin"]), ptr(st["ws2"]),
                                    st["ws2"].numel(), s), "hipns_evidence_scan")
    return {"idx": st["idx"], "num_live": st["nl"], "per_sample": st["per8"], "final": st["fin"]}


def _run_loglik(st):
    b = st["batch"]
    args = (ptr(b.runs_dev), b.runs_host, C.byref(b.bufs), C.byref(b.launch), stream_ptr())
    check(lib().hipns_log_likelihood(ptr(st["U"]), st["B"], ptr(st["log_L"]), *args), "hipns_log_likelihood")
    check(lib().hipns_log_likelihood_grad(ptr(st["U"]), st["B"], ptr(st["log_L_grad"]), ptr(st["grad"]), *args),
          "hipns_log_likelihood_grad")
    return {"log_L": st["log_L"], "log_L_grad": st["log_L_grad"], "grad": st["grad"]}


_RUN = {"sample": _run_sample, "single": _run_single, "ensemble": _run_ensemble, "batch": _run_batch,
        "mstep": _run_mstep, "evidence": _run_evidence, "loglik": _run_loglik}


# ----------------------------------------------------------------------------- work
def _flops_per_eval(case):
    D = case["D"]
    if case.get("family") == "linreg":
        return 2.0 * case["rows"] * (D + 1)
    if case.get("family") == "mvn":
        return 2.0 * D * D + 40.0 * D
    return 3.0 * 4 * D + 10.0 * D


def _shells(case):
    """Shells of half the live points until the remaining evidence is small: two per nat of compression."""
    D = case["D"]
    if case.get("family") == "linreg":
        return D * math.log(case["rows"] / 0.09) + 16.0
    return 24.0 + 0.6 * D if case.get("family") == "mvn" else 10.0 + 4.5 * D


def work(case):
    kind, D = case["kind"], case.get("D", 1)
    if kind == "sample":
        evals = case["n"] * case["s"] * D * EVALS_PER_SLICE
        data = 6.0 * case["rows"] * D if case["family"] == "linreg" else 4.0 * D * D
        return {"bytes": data + case["n"] * (8.0 * D + 24.0), "flops": evals * _flops_per_eval(case)}
    if kind in ("single", "ensemble", "batch"):
        N, R = case.get("N") or case["c"] or 30 * D, case.get("R", 1)
        s = case.get("s", 5)
        samples = R * N * (_shells(case) / 2.0 + 1.0)
        if kind == "batch" and case["family"] == "gmm":
            samples *= 0.35  # D and N uniform below their largest values
        return {"bytes": samples * (8.0 * D + 48.0), "flops": samples * s * D * EVALS_PER_SLICE * _flops_per_eval(case)}
    if kind == "mstep":
        return {"bytes": 4.0 * case["M"] * D + 12.0 * case["M"] + 6.0 * case["rows"] * D,
                "flops": 2.0 * case["M"] * case["rows"] * (D + 2)}
    if kind == "evidence":
        # log L and sender in; sample indices, live-point counts and eight statistics out
        return {"bytes": case["M"] * (12.0 + 16.0 + 64.0), "flops": case["M"] * 100.0}
    return {"bytes": case["B"] * (8.0 * D + 16.0 + 4.0 * D), "flops": case["B"] * 3.0 * _flops_per_eval(case)}


# ----------------------------------------------------------------------------- exact
def exact(case, seed):
    if case["kind"] in ("mstep", "evidence", "loglik"):
        return {"mstep": _exact_mstep, "evidence": _exact_evidence, "loglik": _exact_loglik}[case["kind"]](
            case, seed, np.random.default_rng(seed))
    return None  # a random walk: no value of its own


def _exact_mstep(case, seed, rng):
    X, y, U, log_w, theta = _mstep_arrays(case, rng)
    X, y = torch.from_numpy(X).cuda(), torch.from_numpy(y).cuda()
    s2, tau = math.exp(2.0 * theta[0]), math.exp(theta[1])
    w = tau * torch.special.ndtri(torch.from_numpy(U).cuda().double())
    rss, wxr = [], []
    for part in w.split(2048):
        r = y[None, :] - part @ X.T
        rss.append((r * r).sum(1))
        wxr.append((part * (r @ X)).sum(1))
    rss, wxr = torch.cat(rss), torch.cat(wxr)
    N = case["rows"]
    terms = -0.5 * N * math.log(2.0 * math.pi * s2) - 0.5 * rss / s2 + torch.from_numpy(log_w).cuda()
    p = torch.softmax(terms, 0)
    return {"log_Z": torch.logsumexp(terms, 0), "grad": torch.stack([(p * (rss / s2 - N)).sum(), (p * wxr).sum() / s2])}


def _exact_evidence(case, seed, rng):
    log_L, sender = _collection(case, seed)
    M = case["M"]
    order = torch.argsort(log_L, stable=True)
    # nodes: the root, then the samples; each adds one edge to its sender's and is crossed by one
    degree = torch.zeros(M + 1, dtype=torch.int64, device="cuda")
    degree.index_add_(0, sender.long().clamp(min=0), torch.ones(M, dtype=torch.int64, device="cuda"))
    in_order = torch.cat([degree[:1], degree[1:][order]])
    nl = 1 + torch.cumsum(in_order - 1, 0)[:-1]
    L, n = log_L[order], nl.double()
    prev = torch.cat([torch.full((1,), -math.inf, dtype=torch.float64, device="cuda"), L[:-1]])
    mid = torch.logaddexp(L, prev) - math.log(2.0)
    X = torch.cumsum(torch.log(n) - torch.log1p(n), 0)
    X2 = torch.cumsum(torch.log(n) - torch.log(n + 2.0), 0)
    first = torch.zeros(1, dtype=torch.float64, device="cuda")
    Xp, X2p = torch.cat([first, X[:-1]]), torch.cat([first, X2[:-1]])
    dZ = mid - torch.log1p(n) + Xp
    Z = torch.logcumsumexp(dZ, 0)
    both = torch.log1p(n) + torch.log(n + 2.0)
    ZX = X + torch.logcumsumexp(mid + torch.log(n) - both + X2p - X, 0)
    ZXp = torch.cat([torch.full((1,), -math.inf, dtype=torch.float64, device="cuda"), ZX[:-1]])
    sq = math.log(2.0) - both + 2.0 * mid + X2p
    Z2 = torch.logcumsumexp(torch.logaddexp(math.log(2.0) - torch.log1p(n) + mid + ZXp, sq), 0)
    dZ2 = torch.logcumsumexp(sq, 0)
    per = torch.stack([L, X, X2, Z, ZX, Z2, dZ, dZ2])
    return {"idx": order, "num_live": nl, "per_sample": per, "final": per[:, -1].clone()}


def _exact_loglik(case, seed, rng):
    D = case["D"]
    u = _loglik_points(case, seed).double()
    if case["family"] == "mvn":
        mu, cov = (torch.from_numpy(a).cuda() for a in _mvn_arrays(D, rng))
        q = torch.special.ndtri(u)
        dq = math.sqrt(2.0 * math.pi) * torch.exp(0.5 * q * q)
        chol = torch.linalg.cholesky(cov)
        z = torch.linalg.solve_triangular(chol, (q - mu).T, upper=False)
        L = -0.5 * (z * z).sum(0) - 0.5 * D * math.log(2.0 * math.pi) - torch.log(torch.diagonal(chol)).sum()
        g = -torch.linalg.solve_triangular(chol.T, z, upper=True).T * dq
    else:
        means, sig = (torch.from_numpy(a).cuda() for a in _gmm_arrays(D, rng))
        x = -10.0 + 20.0 * u
        c = torch.stack([-0.5 * ((x - m) ** 2).sum(1) / s ** 2 - 0.5 * D * torch.log(2.0 * math.pi * s ** 2)
                         for m, s in zip(means, sig)], 1) - math.log(4.0)
        L, p = torch.logsumexp(c, 1), torch.softmax(c, 1)
        g = sum(p[:, k:k + 1] * (means[k] - x) / sig[k] ** 2 for k in range(4)) * 20.0
    grad = torch.zeros((case["B"], -(-D // 32) * 32), dtype=torch.float64, device="cuda")
    grad[:, :D] = g
    return {"log_L": L, "log_L_grad": L.clone(), "grad": grad}
