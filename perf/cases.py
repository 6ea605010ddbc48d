"""Performance cases of the kernel-density engine: what a sampler or a served
session asks of it, through the public entry points.

A case is a dict of plain values.  ``op`` says which call it times:

* ``eval``   m2lnp of m points under a prepared KDE / VKDE of n kernels, from
             host arrays (``entry: host``) or from tensors resident in HBM
             (``entry: device``), in FP64, FP32 or the mixed precision;
* ``fit``    a refit on a new sample: reset, add the n observations,
             ``prepare_interp`` and the fitted weights;
* ``half``   one half-step of the APES ensemble sampler: the refit, n
             proposals drawn from it, and the transition densities of the
             proposals' batch and of the current walkers (2 n points);
* ``multi``  the waiting evals of several served sessions in one call.

Samples come from the targets the engine is used on: correlated Gaussians, a
banana, a Gaussian mixture, and Gaussians of condition number 1e4.
"""
import ctypes as C
import math

import numpy as np
import torch

import numcosmo_amd as na
from numcosmo_amd._lib import check, lib

PREC = {"fp64": 0, "mixed": 1, "fp32": 2}


def listed():
    return [
        # one walker's density, as an unbatched sampler or a plot asks for it: latency
        {"name": "point_d4", "op": "eval", "kind": "vkde", "kernel": "st", "nu": 3.0, "d": 4, "n": 1000, "m": 1,
         "precision": "fp64", "entry": "host", "target": "banana", "fit": True},
        # a small KDE with a common covariance, host arrays, the default precision
        {"name": "kde_gauss_d4_fp64", "op": "eval", "kind": "kde", "kernel": "gauss", "nu": 0.0, "d": 4, "n": 1000,
         "m": 10000, "precision": "fp64", "entry": "host", "target": "gaussian", "fit": True},
        # an ordinary batch on a fitted VKDE, in both precisions, points resident
        {"name": "vkde_d8_fp64", "op": "eval", "kind": "vkde", "kernel": "st", "nu": 3.0, "d": 8, "n": 4000,
         "m": 100000, "precision": "fp64", "entry": "device", "target": "banana", "fit": True},
        {"name": "vkde_d8_mixed", "op": "eval", "kind": "vkde", "kernel": "st", "nu": 3.0, "d": 8, "n": 4000,
         "m": 100000, "precision": "mixed", "entry": "device", "target": "banana", "fit": True},
        # the headline evaluation (mixed), and half its points in FP64; equal
        # weights, so that the densities have a 64-bit check at this size
        {"name": "vkde_d16_mixed", "op": "eval", "kind": "vkde", "kernel": "st", "nu": 3.0, "d": 16, "n": 20000,
         "m": 200000, "precision": "mixed", "entry": "device", "target": "gaussian", "fit": False},
        {"name": "vkde_d16_fp64", "op": "eval", "kind": "vkde", "kernel": "st", "nu": 3.0, "d": 16, "n": 20000,
         "m": 100000, "precision": "fp64", "entry": "device", "target": "gaussian", "fit": False},
        # many parameters, an ill-conditioned target
        {"name": "vkde_d64_mixed", "op": "eval", "kind": "vkde", "kernel": "st", "nu": 5.0, "d": 64, "n": 20000,
         "m": 100000, "precision": "mixed", "entry": "device", "target": "cond", "fit": False},
        # the FP32 rung with sizes that fill no tile
        {"name": "vkde_gauss_d27_fp32", "op": "eval", "kind": "vkde", "kernel": "gauss", "nu": 0.0, "d": 27, "n": 3001,
         "m": 20011, "precision": "fp32", "entry": "host", "target": "gaussian", "fit": False},
        # evals of six served sessions (n log-uniform on [500, 20000], m = 10 n)
        {"name": "served_multi", "op": "multi", "kind": "vkde", "kernel": "st", "nu": 3.0, "d": 8, "n": 500,
         "d2": 16, "n2": 3163, "sessions": 6, "precision": "mixed", "target": "gaussian", "fit": False},
        # one half-step of the ensemble sampler at its benchmark size
        {"name": "apes_half_d16", "op": "half", "kind": "vkde", "kernel": "st", "nu": 1.0, "d": 16, "n": 3200,
         "precision": "mixed", "target": "mixture"},
        # refits: few parameters (many active-set solves), and a large one
        {"name": "fit_d4", "op": "fit", "kind": "vkde", "kernel": "st", "nu": 3.0, "d": 4, "n": 2503,
         "target": "gaussian"},
        {"name": "fit_d32", "op": "fit", "kind": "vkde", "kernel": "st", "nu": 3.0, "d": 32, "n": 10000,
         "target": "gaussian"},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges: dimensions 2 to 64, 500 to
    20000 kernels, 1 to 200000 points, every kernel, precision and entry."""
    what = rng.random()
    kernel, nu = ("gauss", 0.0) if rng.random() < 0.25 else ("st", float(rng.choice([1, 3, 3, 5])))
    target = rng.choice(["gaussian", "banana", "mixture", "cond"])
    d = _logint(rng, 2, 64)
    lo = max(500, 40 * d + 160)     # every local covariance has 2 d + 8 neighbours or more

    if what < 0.58:
        precision = rng.choice(["fp64", "fp64", "mixed", "mixed", "mixed", "fp32"])
        n = _logint(rng, lo, 20000)
        # the largest listed evals in that precision bound the work
        most = (8.0e11 if precision == "mixed" else 3.0e11) / (n * float(d * d + 8 * d))
        m = _logint(rng, 1, max(2, min(200000, most)))
        return {"op": "eval", "kind": "kde" if rng.random() < 0.2 else "vkde", "kernel": kernel, "nu": nu, "d": d,
                "n": n, "m": m, "precision": precision, "entry": rng.choice(["host", "device"]), "target": target,
                "fit": n <= 4000 and 4 <= d <= 16}

    if what < 0.68:
        n = _logint(rng, 500, 1500)
        return {"op": "multi", "kind": "vkde", "kernel": "st", "nu": 3.0, "d": int(rng.choice([4, 8])), "n": n,
                "d2": int(rng.choice([4, 8, 16])), "n2": _logint(rng, 500, 4000), "sessions": rng.randint(2, 6),
                "precision": "mixed", "target": "gaussian", "fit": False}

    if what < 0.8:
        d = min(max(d, 4), 20)
        n = _logint(rng, max(500, 40 * d + 160), 4000)
        return {"op": "half", "kind": "vkde", "kernel": "st", "nu": 1.0, "d": d, "n": n, "precision": "mixed",
                "target": target}

    d = max(d, 4)
    n = _logint(rng, lo, 2503 if d < 8 else 6000)
    return {"op": "fit", "kind": "vkde" if rng.random() < 0.85 else "kde", "kernel": kernel, "nu": nu, "d": d, "n": n,
            "target": target}


# ---- inputs ---------------------------------------------------------------

def _gen(seed, tag):
    return np.random.Generator(np.random.Philox(key=(int(seed) * 1009 + tag) % (1 << 64)))


def _spd(g, d, lam):
    Q, R = np.linalg.qr(g.standard_normal((d, d)))
    Q = Q * np.sign(np.diag(R))[None, :]
    return (Q * lam[None, :]) @ Q.T


class _Target:
    """A seeded target: draws and their exact m2lnp."""

    def __init__(self, name, d, g):
        self.name, self.d = name, d
        ncomp = 4 if name == "mixture" else 1
        self.means = g.uniform(-5.0, 5.0, size=(ncomp, d)) if ncomp > 1 else np.zeros((1, d))
        self.L = []
        for _ in range(ncomp):
            if name == "banana":
                self.L.append(np.eye(d))
            elif name == "cond":
                self.L.append(np.linalg.cholesky(_spd(g, d, np.logspace(0.0, 4.0, d))))
            else:
                self.L.append(np.linalg.cholesky(_spd(g, d, 10.0 ** g.uniform(-1.0, 1.0, size=d))))

    def draw(self, g, n):
        Z = g.standard_normal((n, self.d))
        comp = g.integers(0, len(self.L), size=n)
        X = np.empty_like(Z)
        for c, L in enumerate(self.L):
            sel = comp == c
            X[sel] = self.means[c] + Z[sel] @ L.T
        if self.name == "banana":
            X[:, 1] += 0.5 * (X[:, 0] ** 2 - 1.0)
        return X

    def m2lnp(self, X):
        if self.name == "banana":
            X = X.copy()
            X[:, 1] -= 0.5 * (X[:, 0] ** 2 - 1.0)
        t = []
        for mean, L in zip(self.means, self.L):
            Z = np.linalg.solve(L, (X - mean).T)
            t.append(-0.5 * np.sum(Z * Z, axis=0) - np.sum(np.log(np.diag(L))))
        t = np.stack(t)
        mx = t.max(axis=0)
        return (-2.0 * (mx + np.log(np.sum(np.exp(t - mx), axis=0) / len(self.L)))
                + self.d * math.log(2.0 * math.pi))


def _sessions(case):
    """(d, n) of the served sessions: two dimensions in turn, n geometric between n and n2."""
    s = case["sessions"]
    return [(case["d"] if i % 2 == 0 else case["d2"],
             max(int(round(case["n"] * (case["n2"] / case["n"]) ** (i / max(1, s - 1)))), 840 if i % 2 else 500))
            for i in range(s)]


def _inputs(case, seed, part=0):
    """Sample, its m2lnp, evaluation points and sampling variates, from the seed alone."""
    d, n = case["d"], case["n"]
    g = _gen(seed, 16 * part + 1)
    tgt = _Target(case["target"], d, g)
    X = tgt.draw(g, n)
    inp = {"X": X, "m2lnp": tgt.m2lnp(X)}
    if case["op"] in ("eval", "multi"):
        inp["Xe"] = tgt.draw(g, case["m"] if case["op"] == "eval" else 10 * n)
    elif case["op"] == "half":
        inp["Xe"] = tgt.draw(g, 2 * n)
        inp["u"] = g.random(n)
        inp["z"] = g.standard_normal((n, d))
        inp["chi2"] = g.chisquare(case["nu"], size=n)
    return inp


def _handle(case):
    k = (na.StatsDistKernelGauss.new(case["d"]) if case["kernel"] == "gauss"
         else na.StatsDistKernelST.new(case["d"], case["nu"]))
    return (na.StatsDistVKDE if case["kind"] == "vkde" else na.StatsDistKDE).new(k, na.StatsDistCV.NONE)


def _part(case, i):
    d, n = _sessions(case)[i]
    return dict(case, d=d, n=n)


# ---- what is timed ----------------------------------------------------------

def prepare(case, seed):
    if case["op"] == "multi":
        sds, Xs = [], []
        for i in range(case["sessions"]):
            c = _part(case, i)
            inp = _inputs(c, seed, i)
            sd = _handle(c)
            sd.add_obs_array(inp["X"])
            sd.prepare()
            sds.append(sd)
            Xs.append(inp["Xe"])
        return {"case": case, "sds": sds, "Xs": Xs}

    inp = _inputs(case, seed)
    sd = _handle(case)
    st = {"case": case, "sd": sd, "inp": inp}
    if case["op"] == "half":
        sd.set_mixed_tolerance(1.5e-6)      # what the ensemble sampler sets on its own handles
    if case["op"] == "eval":
        sd.add_obs_array(inp["X"])
        if case["fit"]:
            sd.prepare_interp(inp["m2lnp"])
        else:
            sd.prepare()
        if case["entry"] == "device":
            st["dX"] = torch.tensor(inp["Xe"], dtype=torch.float64, device="cuda")
            st["dout"] = torch.empty(case["m"], dtype=torch.float64, device="cuda")
    return st


def run(st):
    case = st["case"]
    prec = PREC[case.get("precision", "fp64")]

    if case["op"] == "multi":
        return na.ncm_stats_dist.eval_m2lnp_multi(st["sds"], st["Xs"], precision=prec)

    sd, inp = st["sd"], st["inp"]

    if case["op"] == "eval":
        if case["entry"] == "device":
            check(lib().nckde_eval_m2lnp_device(sd._h, C.c_void_p(st["dX"].data_ptr()), case["m"],
                                                C.c_void_p(st["dout"].data_ptr()), prec,
                                                C.c_void_p(torch.cuda.current_stream().cuda_stream)))
            return st["dout"]
        return sd.eval_m2lnp_batch(inp["Xe"], prec)

    sd.reset()
    sd.add_obs_array(inp["X"])
    sd.prepare_interp(inp["m2lnp"])
    w = sd.peek_weights()

    if case["op"] == "fit":
        return w

    prop, idx = sd.sample_batch(inp["u"], inp["z"], inp["chi2"])
    return {"weights": w, "idx": idx, "proposals": prop, "m2lnp": sd.eval_m2lnp_batch(inp["Xe"], prec)}


# ---- the work a pass cannot do without ---------------------------------------

def _eval_work(case, m):
    d, n = case["d"], case["n"]
    if case["kind"] == "kde":
        return {"bytes": 8.0 * (n * (d + 1) + m * (d + 1)), "flops": 3.0 * d * n * m + 1.0 * d * d * m}
    # the triangular product, the differences and the squared norm of every pair
    return {"bytes": 8.0 * (n * (d * (d + 1) // 2 + d + 1) + m * (d + 1)), "flops": (d * (d + 1.0) + 3.0 * d) * n * m}


def _fit_work(case):
    d, n = case["d"], case["n"]
    fl = n * (n + 1.0) * n + n ** 3 / 3.0 + 6.0 * n * n          # normal equations, one factor, its products
    fl += (3.0 * d if case["kind"] == "kde" else d * (d + 1.0) + 3.0 * d) * n * n    # interpolation matrix
    if case["kind"] == "vkde":
        k = max(2, int(0.05 * n))
        fl += 3.0 * d * n * n + 1.0 * k * d * (d + 1) * n + n * d ** 3 / 3.0         # neighbours, covariances
    return {"bytes": 8.0 * (n * d + 2 * n), "flops": fl}


def work(case):
    if case["op"] == "eval":
        return _eval_work(case, case["m"])
    if case["op"] == "multi":
        parts = [_eval_work(_part(case, i), 10 * _sessions(case)[i][1]) for i in range(case["sessions"])]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    w = _fit_work(case)
    if case["op"] == "half":
        e = _eval_work(case, 2 * case["n"])
        return {"bytes": w["bytes"] + e["bytes"] + 24.0 * case["n"] * case["d"], "flops": w["flops"] + e["flops"]}
    return w


def tolerance(case):
    # about four times the largest error against `exact` seen over 50 cases:
    # FP64 2e-14 (a KDE with a fitted weight vector; left at 1e-12, since
    # another order in the fit moves the weights), mixed 6e-8, FP32 3.8e-8
    if case["op"] in ("eval", "multi"):
        return {"fp64": {"rel": 1e-12}, "mixed": {"rel": 2.5e-7}, "fp32": {"rel": 2e-7}}[case["precision"]]
    # fitted weights: 4e-13 from 8 dimensions on; with fewer the normal
    # equations are worse conditioned (1.7e-11 between two orders of the sums
    # at 600 points, and the active set may end one step apart)
    if case["op"] == "fit":
        return {"rel": 1e-9 if case["d"] < 8 else 1e-11}
    return {"rel": 2.5e-7, "differ": 0.001}


# ---- the same in plain 64-bit torch ------------------------------------------

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _lnnorm_const(case):
    d, nu = case["d"], case["nu"]
    if case["kernel"] == "gauss":
        return 0.5 * d * math.log(2.0 * math.pi)
    return math.lgamma(nu / 2) - math.lgamma((nu + d) / 2) + 0.5 * d * (math.log(math.pi) + math.log(nu))


def _lnK(case, chi2):
    if case["kernel"] == "gauss":
        return -0.5 * chi2
    return -0.5 * (case["nu"] + case["d"]) * torch.log1p(chi2 / case["nu"])


def _cov(X):
    c = X - X.mean(dim=-2, keepdim=True)
    return c.transpose(-1, -2).contiguous() @ c / (X.shape[-2] - 1)


def _model(case, X):
    """Centres, inverse factors W (z = W (x - theta)), log-norms and bandwidth."""
    d, n = case["d"], case["n"]
    X = torch.as_tensor(X, dtype=torch.float64)
    eye = torch.eye(d, dtype=torch.float64)
    Lg = torch.linalg.cholesky(_cov(X))
    lnc = _lnnorm_const(case)
    if case["kind"] == "kde":
        if case["kernel"] == "gauss":
            h = (4.0 / (n * (d + 2.0))) ** (1.0 / (d + 4.0))
        else:
            nu = max(case["nu"], 3.0)
            h = (16.0 * (nu - 2) ** 2 * (1 + d + nu) * (3 + d + nu)
                 / ((2.0 + d) * (d + nu) * (2 + d + nu) * (d + 2 * nu) * (2 + d + 2 * nu) * n)) ** (1.0 / (d + 4.0))
        W = torch.linalg.solve_triangular(Lg, eye, upper=False)[None]
        ln = torch.full((n,), lnc + float(torch.log(torch.diagonal(Lg)).sum()), dtype=torch.float64)
        return X, W, Lg[None], ln, h
    dev = _dev()
    k = max(2, int(0.05 * n))
    Y = torch.linalg.solve_triangular(Lg, X.T.contiguous(), upper=False).T.contiguous().to(dev)
    Xd = X.to(dev)
    covs = []
    step = max(1, int(4e7 / (n * 2 + k * d * 2)))
    for a in range(0, n, step):
        q = Y[a:a + step]
        d2 = torch.zeros((q.shape[0], n), dtype=torch.float64, device=dev)
        for l in range(d):
            d2 += (q[:, l, None] - Y[None, :, l]) ** 2
        idx = torch.topk(d2, k, dim=1, largest=False, sorted=False).indices
        covs.append(_cov(Xd[idx]).cpu())
    L = torch.linalg.cholesky(torch.cat(covs))
    W = torch.linalg.solve_triangular(L, eye.expand(n, d, d).contiguous(), upper=False)
    return X, W, L, lnc + torch.log(torch.diagonal(L, dim1=1, dim2=2)).sum(dim=1), 1.0


def _chi2(X, W, h, P, a, b):
    """chi2 of kernels a..b at the points P: (b - a) x m."""
    D = P[None, :, :] - X[a:b, None, :]
    Wt = (W[a:b] if W.shape[0] > 1 else W.expand(b - a, -1, -1)).transpose(-1, -2).contiguous()
    return (D @ Wt).square_().sum(dim=-1) / (h * h)


def _eval_exact(case, model, w, P):
    X, W, _, ln, h = model
    dev = _dev()
    X, W, P = X.to(dev), W.to(dev), torch.as_tensor(P, dtype=torch.float64, device=dev)
    n, d, m = X.shape[0], X.shape[1], P.shape[0]
    b = (torch.log(torch.as_tensor(w, dtype=torch.float64)) - ln - d * math.log(h)).to(dev)
    out = torch.empty(m, dtype=torch.float64, device=dev)
    ms = min(m, 65536)
    ks = max(1, min(n, int(1.5e8 / (ms * d))))
    for p in range(0, m, ms):
        Pp = P[p:p + ms]
        M = torch.full((Pp.shape[0],), -math.inf, dtype=torch.float64, device=dev)
        S = torch.zeros_like(M)
        for a in range(0, n, ks):
            t = _lnK(case, _chi2(X, W, h, Pp, a, min(n, a + ks))) + b[a:a + ks, None]
            Mn = torch.maximum(M, t.max(dim=0).values)
            S = S * torch.exp(M - Mn) + torch.exp(t - Mn).sum(dim=0)
            M = Mn
        out[p:p + ms] = -2.0 * (M + torch.log(S))
    return out.cpu().numpy()


def _weights_exact(case, model, m2lnp):
    """The non-negative least-squares weights: the active-set steps of the
    fit on refined normal equations, then the shrink of 0.01."""
    X, W, _, ln, h = model
    dev = _dev()
    n, d = X.shape
    Xd, Wd = X.to(dev), W.to(dev)
    f = np.exp(-0.5 * (m2lnp - m2lnp.min()))
    A = np.empty((n, n))
    ks = max(1, int(1.0e8 / (n * d)))
    for a in range(0, n, ks):
        e = min(n, a + ks)
        t = _lnK(case, _chi2(Xd, Wd, h, Xd, a, e)) - (ln[a:e, None].to(dev) + d * math.log(h))
        A[:, a:e] = torch.exp(t).cpu().numpy().T
    A /= f[:, None]
    M = A.T @ A
    At = torch.from_numpy(A)

    def feasible(P, most):
        idx = np.flatnonzero(P)
        while True:
            L = torch.linalg.cholesky(torch.from_numpy(M[np.ix_(idx, idx)]))
            Ai = At[:, torch.from_numpy(idx)]
            x = torch.zeros(len(idx), 1, dtype=torch.float64)
            for _ in range(4):
                x = x + torch.cholesky_solve(Ai.T @ (1.0 - Ai @ x), L)
            x = x[:, 0].numpy()
            bad = np.flatnonzero(x < 1e-300)
            if not len(bad):
                full = np.zeros(n)
                full[idx] = x
                return full
            if len(bad) > most:
                bad = bad[np.argsort(x[bad], kind="stable")[:most]]
            idx = np.delete(idx, bad)

    eps = 2.220446049250313e-16
    x = feasible(np.ones(n, bool), n)
    r = 1.0 - A @ x
    rn = float(np.linalg.norm(r))
    for _ in range(40):
        g = A.T @ r
        P = x > 0
        cand = np.flatnonzero(~P & (g > rn * eps))
        cand = cand[np.argsort(-g[cand], kind="stable")]
        frac, better = 1.0, False
        while len(cand):
            add = int(max(1, len(cand) * frac))
            frac *= 0.5
            T = P.copy()
            T[cand[:add]] = True
            xt = feasible(T, add)
            rt = 1.0 - A @ xt
            if rn - float(np.linalg.norm(rt)) > rn * eps:
                x, r, rn, better = xt, rt, float(np.linalg.norm(rt)), True
                break
            if add == 1:
                break
        if not better:
            break
    else:
        return None
    return x * (0.99 / x.sum()) + 0.01 / n


def _one_exact(case, seed, part=0):
    inp = _inputs(case, seed, part)
    model = _model(case, inp["X"])
    w = np.full(case["n"], 1.0 / case["n"])
    if case.get("fit", True):
        try:
            w = _weights_exact(case, model, inp["m2lnp"])
        except torch.linalg.LinAlgError:    # normal equations too ill-conditioned for this check
            w = None
    return inp, model, w


def exact(case, seed):
    if case["op"] == "multi":
        out = []
        for i in range(case["sessions"]):
            c = _part(case, i)
            inp, model, w = _one_exact(c, seed, i)
            out.append(_eval_exact(c, model, w, inp["Xe"]))
        return out
    # the active set of a fit with few parameters or many kernels takes too long here
    if case.get("fit", True) and (case["n"] > 4000 or (case["op"] != "eval" and case["d"] < 8)):
        return None
    if not torch.cuda.is_available() and case["op"] == "eval" and _eval_work(case, case["m"])["flops"] > 2e11:
        return None
    inp, model, w = _one_exact(case, seed)
    if w is None:
        return None
    if case["op"] == "eval":
        return _eval_exact(case, model, w, inp["Xe"])
    if case["op"] == "fit":
        return w
    cum = np.concatenate([[0.0], np.cumsum(w)])
    cum /= cum[-1]
    idx = np.maximum(np.searchsorted(cum[:case["n"]], inp["u"], side="right") - 1, 0)
    t = (model[2][torch.from_numpy(idx)] @ torch.from_numpy(inp["z"])[:, :, None])[:, :, 0].numpy()
    t = t * (model[4] * np.sqrt(case["nu"] / inp["chi2"]))[:, None]
    return {"weights": w, "idx": idx.astype(np.uint32), "proposals": inp["X"][idx] + t,
            "m2lnp": _eval_exact(case, model, w, inp["Xe"])}
