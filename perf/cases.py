"""Performance cases: the calls a user of the framework makes in earnest.

A fit evaluates the log-likelihood (or the log-likelihood and its gradient)
hundreds of times on one data set, so that call at every size carries the
use: n = 400 to 40,000 in FP64 over the univariate, nugget, bivariate and
space-time kernels, tile sizes 64 to 960, and the mixed-precision
evaluation up to n = 90,000.  Kriging of held-out locations follows a fit.

Locations are the generator's Morton-sorted jittered grid (or its space-time
slots).  Observations are drawn from the seed as a sum of random plane waves
whose spectral distribution is the Matern kernel's, which has its covariance;
fields at the sizes of the mixed path cannot be drawn by a factorisation here
without running the framework's own.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import exageostat_amd

UNI = "univariate_matern_stationary"
NUG = "univariate_matern_nuggets_stationary"
BIV = "bivariate_matern_parsimonious"
ST = "univariate_spacetime_matern_stationary"

# The options of the benchmark's mixed evaluation.
MIXED = dict(fp32_corr=1e-2, bf16=True, fp64_corr=0.0, diag_thick=1, ir_steps=2, ir_tol=0.0)

TIME_SLOTS = 4
WAVES = 1024
EXACT_ROWS = 6000  # rows up to which exact() forms the dense matrices


def _case(name, what, kernel, n, ts, beta, nu, **more):
    c = {"what": what, "kernel": kernel, "n": n, "ts": ts, "beta": beta, "nu": nu, "sigma2": 1.0, "precision": 0}
    if name:
        c["name"] = name
    c.update(more)
    return c


def listed():
    return [
        # The smallest fits: a few hundred stations, one evaluation of many.
        _case("loglik_n400", "loglik", UNI, 400, 64, 0.1, 0.5),
        _case("grad_n900_nugget", "gradient", NUG, 900, 64, 0.1, 0.8, nugget=0.05),
        # The reference's small synthetic data set (1,600 points in tiles of
        # 320), at a smoothness that has no closed form, as inside a fit.
        _case("loglik_n1600", "loglik", UNI, 1600, 320, 0.07, 0.8, sigma2=1.3),
        # Space-time data: 800 stations at four times.
        _case("loglik_spacetime_n3200", "loglik", ST, 3200, 320, 0.1, 0.6),
        # A data set of an odd size with measurement error, ragged last tile.
        _case("loglik_n5003_nugget", "loglik", NUG, 5003, 320, 0.1, 0.6, nugget=0.05),
        # Kriging of held-out stations after a fit.
        _case("predict_n6000", "predict", UNI, 6000, 320, 0.1, 0.5, n_miss=600),
        # Two variables at 4,500 locations.
        _case("loglik_bivariate_n9000", "loglik", BIV, 9000, 192, 0.1, 0.5, sigma2b=1.3, nu2=1.0, rho=0.5),
        # A gradient-based fit of a medium data set.
        _case("grad_n12000", "gradient", UNI, 12000, 960, 0.1, 0.5),
        _case("loglik_n20000", "loglik", UNI, 20000, 960, 0.1, 0.5),
        # The mixed-precision evaluation at a medium size.
        _case("mixed_n30720", "loglik", UNI, 30720, 960, 0.1, 0.5, precision=2),
        # The size of the gradient-fit benchmark (200 x 200 grid, nugget).
        _case("loglik_n40000_nugget", "loglik", NUG, 40000, 960, 0.1, 0.55, nugget=0.01),
        # The benchmark's headline: 300 x 300 grid, mixed precision.
        _case("mixed_n90000", "loglik", UNI, 90000, 960, 0.1, 0.5, precision=2),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _tile_size(rng, n):
    """The tile sizes in use, the larger ones for the larger matrices."""
    if n < 1000:
        return rng.choice([64, 128])
    if n < 4000:
        return rng.choice([128, 192, 320])
    if n < 10000:
        return rng.choice([192, 256, 320, 640, 960])
    return rng.choice([640, 960, 1024])


def draw(rng):
    kind = rng.choice(["loglik", "loglik", "gradient", "predict", "bivariate", "spacetime", "mixed"])
    beta = round(rng.uniform(0.04, 0.12), 4)
    # A smoothness with a closed form, or one that an optimiser passes
    # through; rougher fields keep large matrices well conditioned.
    nu = rng.choice([0.5, round(rng.uniform(0.45, 0.9), 3)])
    if kind == "bivariate":
        n = 2 * _log_uniform(rng, 300, 8000)
        return _case("", "loglik", BIV, n, _tile_size(rng, n), beta, 0.5, sigma2b=1.3, nu2=0.9, rho=0.4)
    if kind == "spacetime":
        n = TIME_SLOTS * _log_uniform(rng, 100, 4000)
        return _case("", "loglik", ST, n, _tile_size(rng, n), beta, nu)
    if kind == "mixed":
        n = _log_uniform(rng, 8000, 80000)
        return _case("", "loglik", UNI, n, 960, 0.1, 0.5, precision=2)
    if kind == "predict":
        n = _log_uniform(rng, 500, 20000)
        return _case("", "predict", UNI, n, _tile_size(rng, n), beta, nu, n_miss=max(10, n // rng.choice([10, 23])))
    kernel = rng.choice([UNI, NUG])
    nugget = {"nugget": 0.05} if kernel == NUG else {}
    n = _log_uniform(rng, 300, 40000 if kind == "loglik" else 20000)
    return _case("", kind, kernel, n, _tile_size(rng, n), beta, nu, **nugget)


def _theta(case):
    k = case["kernel"]
    if k == UNI:
        return [case["sigma2"], case["beta"], case["nu"]]
    if k == NUG:
        return [case["sigma2"], case["beta"], case["nu"], case["nugget"]]
    if k == BIV:
        return [case["sigma2"], case["sigma2b"], case["beta"], case["nu"], case["nu2"], case["rho"]]
    # a, alpha, beta (interaction), delta of the space-time kernel
    return [case["sigma2"], case["beta"], case["nu"], 0.6, 0.9, 0.5, 0.2]


def _locations(case, seed):
    """x, y, t (t None but for space-time)."""
    if case["kernel"] == ST:
        return exageostat_amd.mle.generate_xy_loc_st(case["n"] // TIME_SLOTS, TIME_SLOTS, seed)
    nloc = case["n"] // 2 if case["kernel"] == BIV else case["n"]
    x, y = exageostat_amd.generate_xy_loc(nloc, seed)
    return x, y, None


def _field(rng, x, y, t, nu, beta):
    """Sum of plane waves of a Matern(nu, beta) spectrum at the locations."""
    u = 2.0 * rng.gamma(nu, 1.0, WAVES)  # chi^2 with 2 nu degrees of freedom
    w = rng.standard_normal((3, WAVES)) / (beta * np.sqrt(u))
    phase = rng.uniform(0.0, 2.0 * math.pi, WAVES)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    w, phase = torch.from_numpy(w).to(dev), torch.from_numpy(phase).to(dev)
    X, Y = torch.from_numpy(x).to(dev), torch.from_numpy(y).to(dev)
    out = torch.empty(len(x), dtype=torch.float64, device=dev)
    for lo in range(0, len(x), 8192):
        hi = min(len(x), lo + 8192)
        a = X[lo:hi, None] * w[0] + Y[lo:hi, None] * w[1] + phase
        if t is not None:  # the waves drift slowly from one time to the next
            a += torch.from_numpy(t[lo:hi]).to(dev)[:, None] * (beta * w[2])
        out[lo:hi] = torch.cos(a).sum(1)
    return (out * math.sqrt(2.0 / WAVES)).cpu().numpy()


def _observations(case, seed, x, y, t):
    rng = np.random.default_rng(seed)
    z = math.sqrt(case["sigma2"]) * _field(rng, x, y, t, case["nu"], case["beta"])
    if case["kernel"] == NUG:
        z += math.sqrt(case["nugget"]) * rng.standard_normal(len(z))
    if case["kernel"] == BIV:
        own = _field(rng, x, y, t, case["nu2"], case["beta"])
        r = case["rho"]
        second = math.sqrt(case["sigma2b"]) * (r * z / math.sqrt(case["sigma2"]) + math.sqrt(1.0 - r * r) * own)
        z = np.stack([z, second], 1).ravel()
    return z


def _data(case, seed):
    x, y, t = _locations(case, seed)
    z = _observations(case, seed, x, y, t)
    d = {"theta": np.array(_theta(case)), "x": x, "y": y, "t": t, "z": z}
    if case["what"] == "predict":
        # held-out locations at random; both sets keep the sorted order
        perm = np.random.default_rng(seed + 11).permutation(case["n"])
        miss, obs = np.sort(perm[:case["n_miss"]]), np.sort(perm[case["n_miss"]:])
        d.update(x=x[obs], y=y[obs], z=z[obs], xm=x[miss], ym=y[miss], zm=z[miss])
    return d


def prepare(case, seed):
    d = _data(case, seed)
    m = exageostat_amd.ExactMLE(d["x"], d["y"], case["ts"], kernel=case["kernel"], t=d["t"],
                                precision=case["precision"])
    if case["precision"] == 2:
        m.set_mixed(**MIXED)
    if case["what"] != "predict":
        m.set_z(d["z"])
    return {"what": case["what"], "model": m, "data": d}


def run(state):
    m, d = state["model"], state["data"]
    if state["what"] == "predict":
        z, mse = m.predict(d["theta"], d["x"], d["y"], d["z"], d["xm"], d["ym"], d["zm"])
        return {"z": z, "mse": mse}
    if state["what"] == "gradient":
        ll, grad = m.loglik(d["theta"], grad=True)
        return {"loglik": ll, "logdet": m.logdet, "dotp": m.dotp, "grad": grad}
    ll = m.loglik(d["theta"])
    return {"loglik": ll, "logdet": m.logdet, "dotp": m.dotp}


def work(case):
    n = float(case["n"])
    params = len(_theta(case))
    if case["what"] == "predict":
        miss = float(case["n_miss"])
        obs = n - miss
        # factorisation, two solves, and the product with the cross-covariance
        return {"bytes": 8.0 * (3 * obs + 4 * miss + 1), "flops": obs ** 3 / 3 + 2 * obs ** 2 + 2 * obs * miss}
    flops = n ** 3 / 3 + n ** 2
    if case["what"] == "gradient":
        flops += 2 * n ** 3 / 3 + n ** 2 + 2 * params * n ** 2
    coords = {BIV: 1.0, ST: 3.0}.get(case["kernel"], 2.0)
    return {"bytes": 8.0 * ((coords + 1) * n + 2 * params + 3), "flops": flops}


# ------------------------------------------------------------- in 64 bits --
_STEP = 0.2


def _bessel_k(nu, x, derivative=False):
    """K_nu(x), or d K_nu / d nu, from its integral over cosh by the
    trapezoidal rule, whose error falls as exp(-pi^2 / step)."""
    lo = float(x.min())
    steps = int(math.ceil(math.acosh(max(2.0, 750.0 / lo)) / _STEP)) + 1
    out = torch.zeros_like(x)
    for i in range(steps + 1):
        t = i * _STEP
        weight = t * math.sinh(nu * t) if derivative else math.cosh(nu * t)
        out += (0.5 if i == 0 else 1.0) * _STEP * weight * torch.exp(-math.cosh(t) * x)
    return out


def _correlation(nu, d, beta):
    """Matern correlation at distances d (1 where d = 0) and x = d / beta
    with 1 in the place of each zero."""
    x = torch.where(d == 0, torch.ones_like(d), d / beta)
    con = 1.0 / (2.0 ** (nu - 1.0) * math.gamma(nu))
    m = con * x ** nu * _bessel_k(nu, x)
    return torch.where(d == 0, torch.ones_like(d), m), x, con


def _distance(xa, ya, xb, yb):
    dx = torch.from_numpy(xa)[:, None] - torch.from_numpy(xb)
    dy = torch.from_numpy(ya)[:, None] - torch.from_numpy(yb)
    return torch.sqrt(dx * dx + dy * dy)


def _covariance(case, a, b):
    th = _theta(case)
    d = _distance(a[0], a[1], b[0], b[1])
    if case["kernel"] == BIV:
        s1, s2, beta, nu1, nu2, rho = th
        nu12 = 0.5 * (nu1 + nu2)
        s12 = rho * math.sqrt(nu1 * nu2) / nu12 * math.sqrt(s1 * s2)
        C = torch.empty(2 * d.shape[0], 2 * d.shape[1], dtype=torch.float64)
        C[0::2, 0::2] = s1 * _correlation(nu1, d, beta)[0]
        C[1::2, 1::2] = s2 * _correlation(nu2, d, beta)[0]
        C[0::2, 1::2] = C[1::2, 0::2] = s12 * _correlation(nu12, d, beta)[0]
        return C
    if case["kernel"] == ST:
        s, beta_s, nu, av, alpha, beta, delta = th
        u = (torch.from_numpy(a[2])[:, None] - torch.from_numpy(b[2])).abs()
        psi = u ** (2.0 * alpha) / av + 1.0
        return s * _correlation(nu, d / psi ** (0.5 * beta), beta_s)[0] / psi ** (beta + delta)
    C = th[0] * _correlation(th[2], d, th[1])[0]
    if case["kernel"] == NUG:
        C[d == 0] += th[3]
    return C


def exact(case, seed):
    if case["n"] > EXACT_ROWS:
        return None
    d = _data(case, seed)
    loc = (d["x"], d["y"], d["t"])
    z = torch.from_numpy(d["z"])
    C = _covariance(case, loc, loc)
    L = torch.linalg.cholesky(C)
    alpha = torch.cholesky_solve(z[:, None], L)[:, 0]
    if case["what"] == "predict":
        zm = (_covariance(case, (d["xm"], d["ym"], None), loc) @ alpha).numpy()
        return {"z": zm, "mse": float(np.mean((d["zm"] - zm) ** 2))}
    logdet = 2.0 * float(torch.log(torch.diagonal(L)).sum())
    dotp = float(z @ alpha)
    out = {"loglik": -0.5 * dotp - 0.5 * logdet - 0.5 * case["n"] * math.log(2.0 * math.pi),
           "logdet": logdet, "dotp": dotp}
    if case["what"] == "gradient":
        # d l / d theta_p = -1/2 <C^-1 - alpha alpha^T, dC / d theta_p>
        W = torch.cholesky_inverse(L) - torch.outer(alpha, alpha)
        s, beta, nu = d["theta"][:3]
        dist = _distance(d["x"], d["y"], d["x"], d["y"])
        M, x, con = _correlation(nu, dist, beta)
        psi = float(torch.digamma(torch.tensor(nu, dtype=torch.float64)))
        d_beta = s * con * x ** (nu + 1.0) * _bessel_k(nu - 1.0, x) / beta
        d_nu = s * (M * (torch.log(x) - math.log(2.0) - psi) + con * x ** nu * _bessel_k(nu, x, derivative=True))
        zero = dist == 0
        d_beta[zero] = d_nu[zero] = 0.0
        g = [(W * M).sum(), (W * d_beta).sum(), (W * d_nu).sum()]
        if case["kernel"] == NUG:
            g.append(W[zero].sum())
        out["grad"] = -0.5 * np.array([float(v) for v in g])
    return out
