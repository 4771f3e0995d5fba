"""The work this framework does for its users, as cases to time.

Most cases evaluate a model's potential energy and its gradient for a batch of
chains (``potential_energy`` and autograd), which is what every leapfrog step
of HMC and NUTS costs; two run a whole ``MCMC``, one the diagnostics of draws
that are on the GPU.  Designs and positions follow the benchmark workloads
(``numpyro_amd/workloads.py``), made on the GPU from the seed: covtype-like
designs (ten normal columns, binary columns, an intercept), designs with a
fifth of the columns scaled by ten, returns of the stochastic-volatility model,
ragged batches of hierarchical regressions; positions lie where a sampler's
chains do, a few posterior standard deviations around the generating values.
"""
import math

import numpy as np
import torch

from numpyro_amd import random as nrandom
from numpyro_amd.diagnostics import device_diagnostics
from numpyro_amd.infer import MCMC, NUTS
from numpyro_amd.models import (HierarchicalLogistic, LogisticRegression, StochasticVolatility,
                                SubsampledLogisticRegression, potential_energy)


def listed():
    return [
        # the smallest call: a study-sized regression on four chains, latency
        {"name": "logit-small", "kind": "logit", "N": 1000, "D": 26, "C": 4, "dtype": "fp32",
         "design": "covtype"},
        # one chain on the covtype design: what the reference quotes its leapfrog on
        {"name": "logit-covtype-1", "kind": "logit", "N": 581012, "D": 55, "C": 1,
         "dtype": "fp32", "design": "covtype"},
        # the same design with the many chains that a GPU holds, plain fp32
        {"name": "logit-covtype-256", "kind": "logit", "N": 581012, "D": 55, "C": 256,
         "dtype": "fp32", "design": "covtype"},
        # the tall and wide design in plain fp32, 1024 chains
        {"name": "logit-wide-fp32", "kind": "logit", "N": 2000000, "D": 256, "C": 1024,
         "dtype": "fp32", "design": "scaled"},
        # the default of the benchmark: the same with X stored in bf16
        {"name": "logit-wide-bf16", "kind": "logit", "N": 2000000, "D": 256, "C": 1024,
         "dtype": "bf16", "design": "scaled"},
        # X stored in fp8: a quarter of the memory, for designs that are kept in numbers
        {"name": "logit-fp8", "kind": "logit", "N": 500000, "D": 250, "C": 250, "dtype": "fp8",
         "design": "scaled"},
        # stochastic volatility, non-centred: the prefix-sum adjoint
        {"name": "sv-nc", "kind": "sv", "T": 3000, "C": 128, "noncentred": True,
         "transform": "exp"},
        # many ragged hierarchical regressions at once, four chains each
        {"name": "hier-1024", "kind": "hier", "G": 1024, "K": 4, "nmin": 50, "nmax": 5000,
         "dmin": 4, "dmax": 64},
        # HMCECS: every chain's own subsample of the tall design, Taylor proxy
        {"name": "ecs-wide", "kind": "ecs", "N": 2000000, "D": 256, "C": 1024, "m": 1000,
         "proxy": 2},
        # ESS and split R-hat of the draws of a stochastic-volatility run
        {"name": "diag-sv", "kind": "diag", "C": 128, "S": 600, "P": 3002},
        # a whole NUTS run of the small regression: warmup, adaptation, draws
        {"name": "nuts-small", "kind": "nuts-logit", "N": 1000, "D": 26, "C": 4, "warmup": 50,
         "samples": 50},
        # NUTS draws of the stochastic-volatility model continued at a given step size
        {"name": "nuts-sv", "kind": "nuts-sv", "T": 3000, "C": 128, "samples": 10,
         "step": 0.01},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["small", "few", "many", "many", "bf16", "fp8", "sv", "sv", "hier", "ecs",
                       "diag", "diag", "nuts-logit", "nuts-sv"])
    if kind == "small":
        return {"kind": "logit", "N": _log(rng, 200, 8000), "D": rng.randint(2, 64),
                "C": rng.randint(1, 16), "dtype": "fp32", "design": "covtype"}
    if kind == "few":
        return {"kind": "logit", "N": _log(rng, 40000, 1000000), "D": rng.randint(30, 256),
                "C": rng.randint(1, 16), "dtype": "fp32",
                "design": rng.choice(["covtype", "scaled"])}
    if kind in ("many", "bf16"):
        return {"kind": "logit", "N": _log(rng, 200000, 2000000), "D": rng.randint(20, 256),
                "C": _log(rng, 130, 1024), "dtype": "fp32" if kind == "many" else "bf16",
                "design": rng.choice(["covtype", "scaled"])}
    if kind == "fp8":
        return {"kind": "logit", "N": _log(rng, 200000, 500000), "D": rng.randint(20, 250),
                "C": _log(rng, 2, 250), "dtype": "fp8", "design": rng.choice(["covtype", "scaled"])}
    if kind == "sv":
        return {"kind": "sv", "T": _log(rng, 300, 5000), "C": _log(rng, 4, 512),
                "noncentred": rng.choice([True, False]),
                "transform": rng.choice(["exp", "exp", "softplus"])}
    if kind == "hier":
        return {"kind": "hier", "G": _log(rng, 16, 1024), "K": rng.choice([1, 2, 4, 8]),
                "nmin": rng.randint(20, 200), "nmax": rng.randint(1000, 5000),
                "dmin": rng.randint(2, 16), "dmax": rng.randint(32, 64)}
    if kind == "ecs":
        return {"kind": "ecs", "N": _log(rng, 50000, 2000000), "D": rng.randint(20, 256),
                "C": _log(rng, 16, 1024), "m": _log(rng, 100, 1000),
                "proxy": rng.choice([1, 2, 2])}
    if kind == "diag":
        return {"kind": "diag", "C": _log(rng, 2, 256), "S": _log(rng, 100, 1000),
                "P": _log(rng, 3, 1500)}
    if kind == "nuts-logit":
        return {"kind": "nuts-logit", "N": _log(rng, 300, 2000), "D": rng.randint(4, 40),
                "C": rng.randint(1, 8), "warmup": rng.randint(30, 50),
                "samples": rng.randint(20, 50)}
    return {"kind": "nuts-sv", "T": _log(rng, 500, 3000), "C": _log(rng, 8, 128),
            "samples": rng.randint(5, 10), "step": 0.01}


# ---- inputs ---------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) + 1)
    return g


def _design(N, D, design, g):
    """X [N, D], generating coefficients [D] and labels [N], float32."""
    if design == "covtype":
        nb = max(0, D - 11)  # ten normal columns, then binary ones, then the intercept
        X = torch.randn((N, D), generator=g, device="cuda")
        if nb:
            X[:, D - 1 - nb:D - 1] = (torch.rand((N, nb), generator=g, device="cuda") < 0.1).float()
        if D > 1:
            X[:, D - 1] = 1.0
        beta = 0.5 * torch.randn(D, generator=g, device="cuda")
    else:
        X = torch.randn((N, D), generator=g, device="cuda")
        cols = torch.randperm(D, generator=g, device="cuda")[:max(1, D // 5)]
        X[:, cols] *= 10.0
        beta = 0.1 * torch.randn(D, generator=g, device="cuda")
    y = (torch.rand(N, generator=g, device="cuda") < torch.sigmoid(X @ beta)).float()
    return X, y, beta


def _positions(X, beta, C, g):
    """Chains around beta, about a posterior standard deviation per coordinate."""
    sd = 2.5 / X.square().sum(0).sqrt().clamp_min(1.0)
    return (beta + sd * torch.randn((C, X.shape[1]), generator=g, device="cuda")).contiguous()


def _returns(T, g):
    """Returns of the stochastic-volatility model (sigma 0.03, nu 10) and their path."""
    zeta = torch.randn(T, generator=g, device="cuda")
    s = 0.03 * torch.cumsum(zeta, 0)
    chi2 = torch.randn((10, T), generator=g, device="cuda").square().sum(0)
    t = torch.randn(T, generator=g, device="cuda") * torch.sqrt(10.0 / chi2)
    return (torch.exp(s) * t).contiguous(), zeta, s


def _sv_positions(T, C, noncentred, transform, zeta, s, g):
    def un(v):
        return math.log(math.expm1(v)) if transform == "softplus" else math.log(v)
    z = torch.empty((C, T + 2), device="cuda")
    z[:, 0] = un(10.0)
    if noncentred:
        z[:, 1] = un(0.03)
        z[:, 2:] = zeta
        z += 0.1 * torch.randn((C, T + 2), generator=g, device="cuda")
    else:
        z[:, 1:T + 1] = s
        z[:, T + 1] = un(0.03)
        z += 0.01 * torch.randn((C, T + 2), generator=g, device="cuda")
    return z


def _hier_data(case, g):
    r = np.random.default_rng(int(torch.randint(0, 1 << 30, (1,), generator=g, device="cuda")))
    ns = r.integers(case["nmin"], case["nmax"] + 1, case["G"]).tolist()
    ds = r.integers(case["dmin"], case["dmax"] + 1, case["G"]).tolist()
    flat = torch.randn(sum(n * d for n, d in zip(ns, ds)), generator=g, device="cuda")
    eta = torch.randn((case["G"], case["dmax"]), generator=g, device="cuda")
    mu = torch.randn(case["G"], generator=g, device="cuda")
    u = torch.rand(sum(ns), generator=g, device="cuda")
    z = torch.zeros((case["G"] * case["K"], max(ds) + 2), device="cuda")
    noise = 0.3 * torch.randn(z.shape, generator=g, device="cuda")
    Xs, ys, o, p = [], [], 0, 0
    for i, (n, d) in enumerate(zip(ns, ds)):
        X = flat[o:o + n * d].view(n, d)
        ys.append((u[p:p + n] < torch.sigmoid(X @ (mu[i] + 0.7 * eta[i, :d]))).float())
        Xs.append(X)
        rows = slice(i * case["K"], (i + 1) * case["K"])
        z[rows, :d] = eta[i, :d]
        z[rows, d] = mu[i]
        z[rows, d + 1] = math.log(0.7)
        z[rows, :d + 2] += noise[rows, :d + 2]
        o, p = o + n * d, p + n
    return Xs, ys, z


def _draws(case, g):
    """Draws [C, S, P] of chains with autocorrelations from -0.3 to 0.95."""
    C, S, P = case["C"], case["S"], case["P"]
    rho = torch.linspace(-0.3, 0.95, P, device="cuda")
    x = torch.randn((C, S, P), generator=g, device="cuda")
    amp = torch.sqrt(1.0 - rho * rho)
    for t in range(1, S):
        x[:, t] = rho * x[:, t - 1] + amp * x[:, t]
    return x + torch.randn(P, generator=g, device="cuda")


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "logit":
        X, y, beta = _design(case["N"], case["D"], case["design"], g)
        z = _positions(X, beta, case["C"], g).requires_grad_(True)
        return {"kind": kind, "model": LogisticRegression(X, y, x_dtype=case["dtype"]), "z": z}
    if kind == "sv":
        r, zeta, s = _returns(case["T"], g)
        z = _sv_positions(case["T"], case["C"], case["noncentred"], case["transform"], zeta, s, g)
        model = StochasticVolatility(r, noncentred=case["noncentred"],
                                     positive_transform=case["transform"])
        return {"kind": kind, "model": model, "z": z.requires_grad_(True)}
    if kind == "hier":
        Xs, ys, z = _hier_data(case, g)
        return {"kind": kind, "model": HierarchicalLogistic(Xs, ys, chains_per_group=case["K"]),
                "z": z.requires_grad_(True)}
    if kind == "ecs":
        X, y, beta, z, idx = _ecs_data(case, g)
        model = SubsampledLogisticRegression(X, y, case["m"], num_blocks=10,
                                             proxy_degree=case["proxy"], reference=beta)
        model.idx = idx
        model.keys = torch.zeros((case["C"], 2), dtype=torch.int32, device="cuda")
        return {"kind": kind, "model": model, "z": z.requires_grad_(True)}
    if kind == "diag":
        return {"kind": kind, "x": _draws(case, g)}
    if kind == "nuts-logit":
        X, y, beta = _design(case["N"], case["D"], "covtype", g)
        mcmc = MCMC(NUTS(LogisticRegression(X, y)), num_warmup=case["warmup"],
                    num_samples=case["samples"], num_chains=case["C"])
        return {"kind": kind, "mcmc": mcmc, "key": nrandom.PRNGKey(seed), "init": None}
    r, zeta, s = _returns(case["T"], g)
    z = _sv_positions(case["T"], case["C"], True, "exp", zeta, s, g)
    mcmc = MCMC(NUTS(StochasticVolatility(r, noncentred=True), step_size=case["step"]),
                num_warmup=0, num_samples=case["samples"], num_chains=case["C"])
    return {"kind": kind, "mcmc": mcmc, "key": nrandom.PRNGKey(seed), "init": z}


def _ecs_data(case, g):
    X, y, beta = _design(case["N"], case["D"], "scaled", g)
    z = _positions(X, beta, case["C"], g)
    idx = torch.randint(0, case["N"], (case["C"], case["m"]), generator=g, device="cuda",
                        dtype=torch.int32)
    return X, y, beta, z, idx


def run(state):
    if state["kind"] == "diag":
        ess, rhat = device_diagnostics(state["x"])
        return {"ess": ess, "rhat": rhat}
    if state["kind"].startswith("nuts"):
        mcmc = state["mcmc"]
        mcmc.run(state["key"], init_params=state["init"])
        return {"samples": mcmc.get_samples(group_by_chain=True),
                "extra": mcmc.get_extra_fields(group_by_chain=True)}
    u = potential_energy(state["model"], state["z"])
    (grad,) = torch.autograd.grad(u.sum(), state["z"])
    return {"u": u.detach(), "grad": grad}


def work(case):
    kind = case["kind"]
    if kind == "logit":
        N, D, C = case["N"], case["D"], case["C"]
        elt = {"fp32": 4, "bf16": 2, "fp8": 1}[case["dtype"]]
        return {"bytes": elt * N * D + 4 * N + 8 * C * D + 8 * C, "flops": 4.0 * N * D * C}
    if kind == "sv":
        return {"bytes": 4 * case["T"] + 8 * case["C"] * (case["T"] + 2),
                "flops": 20.0 * case["C"] * case["T"]}
    if kind == "hier":
        n, d = 0.5 * (case["nmin"] + case["nmax"]), 0.5 * (case["dmin"] + case["dmax"])
        return {"bytes": 4 * case["G"] * n * (d + 1) + 8 * case["G"] * case["K"] * (d + 2),
                "flops": 4.0 * case["G"] * case["K"] * n * d}
    if kind == "ecs":
        C, m, D = case["C"], case["m"], case["D"]
        # rows are read once each however many chains hold them
        rows = min(case["N"], C * m)
        return {"bytes": rows * (4 * D + 32) + 4 * C * m + 8 * C * D + 8 * D * D,
                "flops": 4.0 * C * m * D + 2.0 * C * D * D}
    if kind == "diag":
        return {"bytes": 4 * case["C"] * case["S"] * case["P"] + 16 * case["P"],
                "flops": 10.0 * case["C"] * case["S"] * case["P"]}
    if kind == "nuts-logit":
        it = case["warmup"] + case["samples"]  # at least one gradient each
        return {"bytes": 4 * case["N"] * (case["D"] + 1) + 4 * case["C"] * case["samples"] * case["D"],
                "flops": 4.0 * it * case["N"] * case["D"] * case["C"]}
    return {"bytes": 4 * case["T"] + 4 * case["C"] * (case["T"] + 2) * (1 + case["samples"]),
            "flops": 20.0 * case["samples"] * case["C"] * case["T"]}


# ---- the same in 64 bits -----------------------------------------------------------

def _stored(X, dtype):
    """The design that a storage form stands for, in float64."""
    if dtype == "bf16":
        return X.to(torch.bfloat16).double()
    if dtype == "fp8":
        m = X.abs().amax(0).double() / 448.0
        f, e = torch.frexp(m)
        e = torch.where(f == 0.5, e - 1, e)  # the least power of two that is >= m
        s = torch.where(m > 0, torch.ldexp(torch.ones_like(m), e), torch.ones_like(m))
        return (X / s.float()).to(torch.float8_e4m3fn).double() * s
    return X.double()


def _normal_prior(z):
    return 0.5 * (z * z).sum(1) + z.shape[1] * 0.5 * math.log(2 * math.pi)


def _bern(l, y):
    return torch.nn.functional.softplus(l) - y * l


def _exact_logit(case, g):
    X, y, beta = _design(case["N"], case["D"], case["design"], g)
    z = _positions(X, beta, case["C"], g).double()
    u, grad = _normal_prior(z), z.clone()
    scale = _stored(X, case["dtype"]) if X.numel() <= 1 << 27 else None
    rows = max(1, (1 << 27) // max(case["C"], case["D"]))
    for r0 in range(0, case["N"], rows):
        # bf16 rounds element by element; fp8's scales need all rows of a column
        xc = scale[r0:r0 + rows] if scale is not None else _stored(X[r0:r0 + rows], case["dtype"])
        yc = y[r0:r0 + rows].double()[:, None]
        l = xc @ z.T
        u = u + _bern(l, yc).sum(0)
        grad = grad + (torch.sigmoid(l) - yc).T.contiguous() @ xc
    return {"u": u, "grad": grad}


def _positive(v, transform):
    """The positive value and log|J| of an unconstrained site."""
    if transform == "softplus":
        return torch.nn.functional.softplus(v), torch.nn.functional.logsigmoid(v)
    return torch.exp(v), v


def _exact_sv(case, g):
    r, zeta, s0 = _returns(case["T"], g)
    z = _sv_positions(case["T"], case["C"], case["noncentred"], case["transform"], zeta, s0, g)
    z = z.double().requires_grad_(True)
    r, T = r.double(), case["T"]
    nu, lj_nu = _positive(z[:, 0:1], case["transform"])
    if case["noncentred"]:
        sig, lj_sig = _positive(z[:, 1:2], case["transform"])
        s = sig * torch.cumsum(z[:, 2:], 1)
        path = 0.5 * z[:, 2:].square().sum(1) + T * 0.5 * math.log(2 * math.pi)
    else:
        sig, lj_sig = _positive(z[:, T + 1:], case["transform"])
        s = z[:, 1:T + 1]
        step = torch.diff(s, dim=1, prepend=torch.zeros_like(s[:, :1]))
        path = (0.5 * (step / sig).square()).sum(1) + T * (torch.log(sig)[:, 0]
                                                           + 0.5 * math.log(2 * math.pi))
    obs = (0.5 * (nu + 1) * torch.log1p((r * torch.exp(-s)).square() / nu) + s).sum(1) \
        + T * (0.5 * torch.log(nu * math.pi) + torch.lgamma(0.5 * nu)
               - torch.lgamma(0.5 * (nu + 1)))[:, 0]
    u = path + obs + (50.0 * sig - math.log(50.0) - lj_sig + 0.1 * nu - math.log(0.1)
                      - lj_nu)[:, 0]
    (grad,) = torch.autograd.grad(u.sum(), z)
    return {"u": u.detach(), "grad": grad}


def _exact_hier(case, g):
    Xs, ys, z32 = _hier_data(case, g)
    K = case["K"]
    u, grad = [], torch.zeros_like(z32, dtype=torch.float64)
    half = 0.5 * math.log(2 * math.pi)
    for i, (X, y) in enumerate(zip(Xs, ys)):
        d = X.shape[1]
        z = z32[i * K:(i + 1) * K, :d + 2].double()
        eta, mu, lt = z[:, :d], z[:, d], z[:, d + 1]
        tau = torch.exp(lt)
        x = X.double()
        yc = y.double()[:, None]
        l = x @ (mu[:, None] + tau[:, None] * eta).T
        gb = (torch.sigmoid(l) - yc).T.contiguous() @ x
        u.append(_bern(l, yc).sum(0) + 0.5 * eta.square().sum(1) + d * half + 0.5 * mu * mu + half
                 - (math.log(2.0 / math.pi) - torch.log1p(tau * tau)) - lt)
        rows = grad[i * K:(i + 1) * K]
        rows[:, :d] = eta + tau[:, None] * gb
        rows[:, d] = mu + gb.sum(1)
        rows[:, d + 1] = tau * (eta * gb).sum(1) + 2 * tau * tau / (1 + tau * tau) - 1.0
    return {"u": torch.cat(u), "grad": grad}


def _exact_ecs(case, g):
    X, y, beta, z32, idx = _ecs_data(case, g)
    N, D, C, m = case["N"], case["D"], case["C"], case["m"]
    b, z = beta.double(), z32.double()
    delta = z - b
    LL = torch.zeros((), dtype=torch.float64, device="cuda")
    G = torch.zeros(D, dtype=torch.float64, device="cuda")
    H = torch.zeros((D, D), dtype=torch.float64, device="cuda")
    for r0 in range(0, N, 1 << 18):
        xc, yc = X[r0:r0 + (1 << 18)].double(), y[r0:r0 + (1 << 18)].double()
        l = xc @ b
        p = torch.sigmoid(l)
        LL -= _bern(l, yc).sum()
        G += xc.T @ (yc - p)
        if case["proxy"] == 2:
            H -= xc.T @ (xc * (p * (1 - p))[:, None])
    Hd = delta @ H
    full = LL + delta @ G + 0.5 * (delta * Hd).sum(1)
    gfull = G + Hd
    u, grad = [], []
    for c in range(C):
        x, yc = X[idx[c].long()].double(), y[idx[c].long()].double()
        l, lr = x @ z[c], x @ b
        p, pr = torch.sigmoid(l), torch.sigmoid(lr)
        w = pr * (1 - pr) if case["proxy"] == 2 else torch.zeros_like(pr)
        dl = l - lr
        diff = -_bern(l, yc) - (-_bern(lr, yc) + (yc - pr) * dl - 0.5 * w * dl * dl)
        cc = (yc - p) - (yc - pr) + w * dl
        mean = diff.mean()
        nm = N / m
        est = full[c] + N * mean - 0.5 * N * nm * ((diff * diff).mean() - mean * mean)
        ge = gfull[c] + (nm * (1 - nm * (diff - mean)) * cc) @ x
        u.append(0.5 * (z[c] * z[c]).sum() + 0.5 * D * math.log(2 * math.pi) - est)
        grad.append(z[c] - ge)
    return {"u": torch.stack(u), "grad": torch.stack(grad)}


def _variances(x):
    """_compute_chain_variance_stats over x [C, S, P]."""
    S = x.shape[1]
    within = x.var(1).mean(0)
    est = within * (S - 1) / S
    if x.shape[0] > 1:
        return within, est + x.mean(1).var(0)
    return est, est


def _exact_diag(case, g):
    x = _draws(case, g).double()
    C, S = case["C"], case["S"]
    c = x - x.mean(1, keepdim=True)
    gamma = torch.zeros((S, case["P"]), dtype=torch.float64, device="cuda")
    for i in range(C):
        f = torch.fft.rfft(c[i], n=2 * S, dim=0)
        gamma += torch.fft.irfft(f * f.conj(), n=2 * S, dim=0)[:S] / (S * C)
    within, est = _variances(x)
    rho = 1.0 - (within - gamma) / est
    rho[0] = 1.0
    n = S // 2
    R = rho[0:2 * n:2] + rho[1:2 * n:2]
    R = torch.cat([R[:1], torch.cummin(R[1:].clamp_min(0.0), 0).values])
    ess = C * S / (-1.0 + 2.0 * R.sum(0))
    h = S // 2
    w, e = _variances(torch.cat([x[:, :h], x[:, S - h:]], 0))
    return {"ess": ess, "rhat": torch.sqrt(e / w)}


def exact(case, seed):
    g = _gen(seed)
    f = {"logit": _exact_logit, "sv": _exact_sv, "hier": _exact_hier, "ecs": _exact_ecs,
         "diag": _exact_diag}.get(case["kind"])
    return f(case, g) if f else None  # a chain's draws have no value in 64 bits
