"""The calls that a program makes of this package, as measurable cases.

Each case is one call (or one short chain of calls) through the public entry
points with its inputs already on the GPU.  ``FAMILIES`` names the kinds of
call; ``listed()`` has one case of each, ``draw`` another one of any.

* ``knopp_small``   ``sinkhorn`` with its default method on a small float64
                    problem: the call of a notebook or of a loop over pairs
                    of histograms, where latency counts.
* ``log_f64``       ``sinkhorn(method="sinkhorn_log")`` in float64 at a small
                    reg, to the default stopThr: a few thousand points.
* ``knopp_f32``     ``sinkhorn`` on a float32 cost of thousands of points
                    with odd sizes (rows that are not 16-byte aligned).
* ``log_large``     ``sinkhorn_log`` on the largest dense float32 costs
                    (1 GiB), a fixed number of iterations.
* ``batch``         ``solve_batch``: many equal, small problems in one call.
* ``batch_grad``    ``solve_sample_batch`` and the gradient of its values with
                    respect to both point sets: a loss inside a training step.
* ``points_warm``   many point-cloud problems of one size solved from the
                    learned warm start (network, then solver).
* ``points_graph``  a batch of uneven point-cloud problems replayed through a
                    captured graph, as a server with fixed sizes does.
* ``online``        ``sinkhorn_online``: the squared Euclidean cost of two
                    large clouds, never stored, in the precisions it offers.
* ``lazy``          ``empirical_sinkhorn2(isLazy=True)`` on 2-D and 3-D
                    samples: loss and potentials.
* ``stabilized``    ``sinkhorn(method="sinkhorn_stabilized")`` at a reg where
                    the scalings have to be absorbed.
* ``gromov``        ``solve_gromov_batch`` (fused): small graph pairs.

Outputs of the solvers that take float32 points are returned as float32, the
type in which such a program keeps them.
"""

import math

import numpy as np
import torch

import pot_amd
from pot_amd import batch, online, ragged
from pot_amd import warmstart

FAMILIES = ("knopp_small", "log_f64", "knopp_f32", "log_large", "batch", "batch_grad",
            "points_warm", "points_graph", "online", "lazy", "stabilized", "gromov")


def listed():
    return [
        {"name": "knopp_small", "kind": "knopp_small", "n": 100, "m": 120, "reg": 0.05},
        {"name": "log_f64", "kind": "log_f64", "n": 2048, "m": 2048, "reg": 0.01},
        {"name": "knopp_f32", "kind": "knopp_f32", "n": 5000, "m": 4999, "reg": 0.05},
        {"name": "log_large", "kind": "log_large", "n": 16384, "m": 16384, "reg": 0.01,
         "iters": 100},
        {"name": "batch", "kind": "batch", "B": 512, "n": 64, "m": 64, "reg": 0.05,
         "dtype": "float32", "solver": "log_sinkhorn"},
        {"name": "batch_grad", "kind": "batch_grad", "B": 64, "n": 200, "m": 180, "d": 8,
         "reg": 1.0, "dtype": "float32"},
        {"name": "points_warm", "kind": "points_warm", "B": 4096, "n": 1024, "m": 1024},
        {"name": "points_graph", "kind": "points_graph", "B": 512, "lo": 64, "hi": 1024,
         "sizes": 2},
        {"name": "online", "kind": "online", "n": 16384, "m": 16384, "d": 64, "reg": 0.01,
         "iters": 40, "precision": "f32"},
        {"name": "lazy", "kind": "lazy", "n": 5000, "m": 4000, "d": 3, "reg": 0.5},
        {"name": "stabilized", "kind": "stabilized", "n": 1000, "m": 900, "reg": 0.002,
         "iters": 300},
        {"name": "gromov", "kind": "gromov", "B": 16, "n": 48, "m": 40, "reg": 0.05},
    ]


def _size(rng, lo, hi):
    """A whole number, spread over the logarithm of the range."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _reg(rng, lo, hi):
    return float("%.3g" % math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(FAMILIES)
    c = {"kind": kind}
    if kind == "knopp_small":
        c |= {"n": _size(rng, 20, 512), "m": _size(rng, 20, 512), "reg": _reg(rng, 0.03, 0.5)}
    elif kind == "log_f64":
        c |= {"n": _size(rng, 256, 4096), "m": _size(rng, 256, 4096), "reg": _reg(rng, 0.01, 0.1)}
    elif kind == "knopp_f32":
        c |= {"n": _size(rng, 700, 8192), "m": _size(rng, 700, 8192), "reg": _reg(rng, 0.03, 0.5)}
    elif kind == "log_large":
        c |= {"n": _size(rng, 6000, 16384), "m": _size(rng, 6000, 16384),
              "reg": _reg(rng, 0.01, 0.1), "iters": rng.randrange(40, 100)}
    elif kind == "batch":
        n, m = _size(rng, 12, 256), _size(rng, 12, 256)
        c |= {"B": _size(rng, 8, max(16, min(2048, (1 << 23) // (n * m)))), "n": n, "m": m,
              "reg": _reg(rng, 0.03, 0.3), "dtype": rng.choice(["float32", "float64"]),
              "solver": rng.choice(["log_sinkhorn", "log_sinkhorn", "sinkhorn"])}
    elif kind == "batch_grad":
        n, m = _size(rng, 30, 500), _size(rng, 30, 500)
        c |= {"B": _size(rng, 4, max(8, min(256, (1 << 22) // (n * m)))), "n": n, "m": m,
              "d": rng.randrange(2, 17), "reg": _reg(rng, 0.8, 4.0),
              "dtype": rng.choice(["float32", "float64"])}
    elif kind == "points_warm":
        n = rng.choice([256, 512, 768, 1024, rng.randrange(200, 1024)])
        c |= {"B": _size(rng, 256, 4000), "n": n, "m": n}
    elif kind == "points_graph":
        lo = rng.randrange(32, 257)
        c |= {"B": _size(rng, 32, 512), "lo": lo, "hi": rng.randrange(lo + 64, 1025),
              "sizes": rng.randrange(1000)}
    elif kind == "online":
        n, m = _size(rng, 2000, 24000), _size(rng, 2000, 24000)
        c |= {"n": min(n, (1 << 28) // m), "m": m, "d": rng.choice([16, 32, 50, 64, 100, 128]),
              "reg": _reg(rng, 0.01, 0.1), "iters": 30,
              "precision": rng.choice(["f32", "f32", "bf16x3", "bf16"])}
        if c["d"] > 64:
            c["iters"] = 15
    elif kind == "lazy":
        c |= {"n": _size(rng, 800, 10000), "m": _size(rng, 800, 10000), "d": rng.randrange(2, 4),
              "reg": _reg(rng, 0.3, 2.0)}
    elif kind == "stabilized":
        c |= {"n": _size(rng, 200, 2500), "m": _size(rng, 200, 2500), "reg": _reg(rng, 0.001, 0.02),
              "iters": 20 * rng.randrange(5, 15)}
    else:
        c |= {"B": _size(rng, 4, 64), "n": _size(rng, 8, 64), "m": _size(rng, 8, 64),
              "reg": _reg(rng, 0.03, 0.2)}
    return c


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, dtype=torch.float64):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _weights(g, *shape, dtype=torch.float64):
    """Positive weights that sum to one along the last axis."""
    w = 0.2 + torch.rand(shape, generator=g, device="cuda", dtype=dtype)
    return w / w.sum(-1, keepdim=True)


def _sq(x, y):
    """Squared Euclidean costs of (..., n, d) and (..., m, d)."""
    M = x.square().sum(-1)[..., :, None] + y.square().sum(-1)[..., None, :]
    return M.sub_(2.0 * x @ y.transpose(-1, -2).contiguous()).clamp_(min=0.0)


def _plane_cost(g, n, m, dtype):
    """x ~ N(0, I), y ~ N((2, 2), [[1, .5], [.5, 1]]), M / max M."""
    x = _randn(g, n, 2)
    z = _randn(g, m, 2)
    y = torch.stack([2.0 + z[:, 0], 2.0 + 0.5 * z[:, 0] + math.sqrt(0.75) * z[:, 1]], 1)
    M = _sq(x, y)
    return (M / M.max()).to(dtype)


def _mixtures(g, rows, of, B, kmax):
    """One Gaussian mixture of 1 to kmax components in 16 dimensions for each
    of B problems (means ~ U[-3, 3]^16, deviations ~ U[0.3, 1.5]), and `rows`
    points, row r of problem of[r]."""
    means = 6.0 * torch.rand((B, kmax, 16), generator=g, device="cuda") - 3.0
    dev = 0.3 + 1.2 * torch.rand((B, kmax), generator=g, device="cuda")
    k = torch.randint(1, kmax + 1, (B,), generator=g, device="cuda")
    pick = (torch.rand(rows, generator=g, device="cuda") * k[of]).long().clamp_(max=kmax - 1)
    return means[of, pick] + dev[of, pick][:, None] * _randn(g, rows, 16, dtype=torch.float32)


def _regs(g, B):
    """reg ~ logU[5e-3, 5e-2], on the host as the solvers take it."""
    t = torch.rand(B, generator=g, device="cuda", dtype=torch.float64)
    return torch.exp(math.log(5e-3) + t * math.log(10.0)).cpu().numpy()


def _uneven(case):
    """The sizes are part of the case: the graph is captured for them."""
    r = np.random.default_rng(case["sizes"])
    return (r.integers(case["lo"], case["hi"] + 1, case["B"]),
            r.integers(case["lo"], case["hi"] + 1, case["B"]))


def _inputs(case, seed):
    """The tensors of a case, by name."""
    g, kind = _gen(seed), case["kind"]
    if kind in ("knopp_small", "log_f64", "stabilized", "knopp_f32"):
        dt = torch.float32 if kind == "knopp_f32" else torch.float64
        n, m = case["n"], case["m"]
        return {"M": _plane_cost(g, n, m, dt), "a": _weights(g, n, dtype=dt),
                "b": _weights(g, m, dtype=dt)}
    if kind == "log_large":
        n, m = case["n"], case["m"]
        x = _randn(g, n, 64, dtype=torch.float32)
        y = 0.5 + math.sqrt(2.0) * _randn(g, m, 64, dtype=torch.float32)
        M = _sq(x, y)
        return {"M": M.div_(M.max()), "a": _weights(g, n, dtype=torch.float32),
                "b": _weights(g, m, dtype=torch.float32)}
    if kind == "batch":
        dt = getattr(torch, case["dtype"])
        M = _sq(_randn(g, case["B"], case["n"], 2), 1.0 + _randn(g, case["B"], case["m"], 2))
        M = M / M.amax((1, 2), keepdim=True)
        return {"M": M.to(dt), "a": _weights(g, case["B"], case["n"], dtype=dt),
                "b": _weights(g, case["B"], case["m"], dtype=dt)}
    if kind == "batch_grad":
        dt = getattr(torch, case["dtype"])
        x = _randn(g, case["B"], case["n"], case["d"], dtype=dt)
        y = 0.5 + _randn(g, case["B"], case["m"], case["d"], dtype=dt)
        return {"X": x, "Y": y}
    if kind == "points_warm":
        B, n, m = case["B"], case["n"], case["m"]
        of = torch.arange(B, device="cuda")
        x = _mixtures(g, B * n, of.repeat_interleave(n), B, 8).view(B, n, 16)
        y = _mixtures(g, B * m, of.repeat_interleave(m), B, 8).view(B, m, 16)
        return {"X": x, "Y": y, "regs": _regs(g, B)}
    if kind == "points_graph":
        B = case["B"]
        ns, ms = _uneven(case)
        of = torch.arange(B, device="cuda")
        x = _mixtures(g, int(ns.sum()), of.repeat_interleave(torch.tensor(ns, device="cuda")), B, 4)
        y = _mixtures(g, int(ms.sum()), of.repeat_interleave(torch.tensor(ms, device="cuda")), B, 4)
        return {"X": x, "Y": y, "regs": _regs(g, B), "ns": ns, "ms": ms}
    if kind == "online":
        n, m, d = case["n"], case["m"], case["d"]
        return {"X": _randn(g, n, d, dtype=torch.float32),
                "Y": 0.5 + math.sqrt(2.0) * _randn(g, m, d, dtype=torch.float32),
                "a": _weights(g, n), "b": _weights(g, m)}
    if kind == "lazy":
        return {"X": _randn(g, case["n"], case["d"], dtype=torch.float32),
                "Y": 0.5 + _randn(g, case["m"], case["d"], dtype=torch.float32)}
    B, n, m = case["B"], case["n"], case["m"]
    x, y = _randn(g, B, n, 2), _randn(g, B, m, 2)
    C1, C2 = _sq(x, x).sqrt(), _sq(y, y).sqrt()
    eye1, eye2 = (torch.eye(k, device="cuda", dtype=torch.bool) for k in (n, m))
    C1 = (0.5 * (C1 + C1.transpose(1, 2))).masked_fill_(eye1, 0.0)
    C2 = (0.5 * (C2 + C2.transpose(1, 2))).masked_fill_(eye2, 0.0)
    M = _sq(_randn(g, B, n, 3), _randn(g, B, m, 3))
    return {"C1": C1 / C1.max(), "C2": C2 / C2.max(), "M": M / M.max(),
            "a": _weights(g, B, n), "b": _weights(g, B, m)}


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["kind"] == "batch_grad":
        s["X"].requires_grad_(True)
        s["Y"].requires_grad_(True)
    elif case["kind"] == "points_warm":
        s["net"] = warmstart.load_default(torch.device("cuda", 0))
    elif case["kind"] == "points_graph":
        s["graph"] = ragged.RaggedGraph(s["ns"], s["ms"], 16, numItermax=2000, stopThr=1e-6,
                                        cost="points")
    return s


# ----------------------------------------------------------------- calls

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "knopp_small":
        return pot_amd.sinkhorn(s["a"], s["b"], s["M"], case["reg"])
    if kind == "log_f64":
        P, log = pot_amd.sinkhorn(s["a"], s["b"], s["M"], case["reg"], method="sinkhorn_log",
                                  log=True)
        return {"plan": P, "log_u": log["log_u"], "log_v": log["log_v"], "niter": log["niter"]}
    if kind == "knopp_f32":
        return pot_amd.sinkhorn(s["a"], s["b"], s["M"], case["reg"], stopThr=1e-6)
    if kind == "log_large":
        return pot_amd.sinkhorn(s["a"], s["b"], s["M"], case["reg"], method="sinkhorn_log",
                                numItermax=case["iters"], stopThr=0.0, warn=False)
    if kind == "batch":
        r = pot_amd.solve_batch(s["M"], case["reg"], s["a"], s["b"], solver=case["solver"])
        return {"plan": r.plan, "value": r.value, "value_linear": r.value_linear,
                "potentials": r.potentials}
    if kind == "batch_grad":
        r = pot_amd.solve_sample_batch(s["X"], s["Y"], case["reg"])
        dX, dY = torch.autograd.grad(r.value.sum(), (s["X"], s["Y"]))
        return {"value": r.value.detach(), "plan": r.plan, "dX": dX, "dY": dY}
    if kind == "points_warm":
        R = ragged.points_from_clouds(s["X"], s["Y"], s["regs"])
        cmax = ragged.points_cmax(R)
        u0 = warmstart.predict_u0(s["net"], R, s["X"], s["Y"], s["regs"])
        r = ragged.sinkhorn_log_ragged_points(R, u0=u0, numItermax=2000, stopThr=1e-6,
                                              check_every=1, cmax=cmax, unsolved="nan",
                                              fallback_thr=warmstart.FALLBACK_THR)
        return {"u": r.u.float(), "v": r.v.float()}
    if kind == "points_graph":
        r = s["graph"].solve(s["X"], s["Y"], s["regs"])
        return {"u": r.u.float(), "v": r.v.float()}
    if kind == "online":
        u, v, _ = online.sinkhorn_online(s["X"], s["Y"], case["reg"], s["a"], s["b"],
                                         numItermax=case["iters"], stopThr=0.0, warn=False,
                                         precision=case["precision"])
        return {"u": u.float(), "v": v.float()}
    if kind == "lazy":
        loss, log = pot_amd.empirical_sinkhorn2(s["X"], s["Y"], case["reg"], stopThr=1e-5,
                                                numIterMax=1000, isLazy=True, log=True,
                                                warn=False)
        return {"loss": loss, "f": log["u"], "g": log["v"]}
    if kind == "stabilized":
        return pot_amd.sinkhorn(s["a"], s["b"], s["M"], case["reg"], method="sinkhorn_stabilized",
                                numItermax=case["iters"], warn=False)
    r = batch.solve_gromov_batch(s["C1"], s["C2"], reg=case["reg"], a=s["a"], b=s["b"],
                                 M=s["M"], alpha=0.5, symmetric=True, max_iter=20)
    return {"plan": r.plan, "value": r.value, "value_quad": r.value_quad}


def work(case):
    """Inputs read once and outputs written once; 4 n m flops an iteration
    (one multiply-add per element in each half-step), plus the squared
    distances where the cost is computed on the fly.  Where a case stops on
    its own error, the iterations are those of its usual stop."""
    kind = case["kind"]
    if kind in ("points_warm", "points_graph"):
        if kind == "points_warm":
            el, pts = float(case["n"]) * case["m"] * case["B"], (case["n"] + case["m"]) * case["B"]
            its = 40
        else:
            mean = 0.5 * (case["lo"] + case["hi"])
            el, pts, its = mean * mean * case["B"], 2 * mean * case["B"], 60
        return {"bytes": pts * (16 * 4 + 4.0), "flops": its * el * (4 + 4 * 16)}
    n, m = case["n"], case["m"]
    el = float(n) * m
    if kind in ("online", "lazy"):
        its = case.get("iters", 60)
        return {"bytes": (n + m) * (4.0 * case["d"] + 12), "flops": its * el * (4 + 4 * case["d"])}
    if kind == "gromov":
        B = case["B"]
        one = 8.0 * (n * n + m * m + 2 * el)
        return {"bytes": B * one, "flops": B * 10.0 * (2 * el * (n + m) + 20 * 4 * el)}
    if kind in ("batch", "batch_grad"):
        B, size = case["B"], 8 if case["dtype"] == "float64" else 4
        its = 30 if kind == "batch" else 50
        read = el if kind == "batch" else 2 * (n + m) * case["d"]
        return {"bytes": B * size * (read + el + 2.0 * (n + m)), "flops": B * its * 4 * el}
    size = 4 if kind in ("knopp_f32", "log_large") else 8
    its = case.get("iters", 50)
    return {"bytes": size * (2 * el + n + m), "flops": its * 4 * el}


# ---------------------------------------------- the same in plain float64

def _sinkhorn64(M, a, b, reg, u, iters, stop, rows_first=False, first=0, every=10, error=None):
    """Alternating log-domain updates of (B, n, m) costs; the error of the
    marginal that is not exact is looked at in the iterations first, first +
    every, ...; `error(sums, weights)` gives one number per problem, and all
    stop together.  Returns (u, v)."""
    K = -M / reg
    la, lb = a.log(), b.log()
    v = torch.zeros_like(b) if u is None else None
    if error is None:
        def error(s, w):
            return (s - w).square().sum(-1).sqrt().max()
    for i in range(iters):
        if rows_first:
            u = la - torch.logsumexp(K + v[:, None, :], 2)
            v = lb - torch.logsumexp(K + u[:, :, None], 1)
        else:
            v = lb - torch.logsumexp(K + u[:, :, None], 1)
            u = la - torch.logsumexp(K + v[:, None, :], 2)
        if stop > 0 and i >= first and (i - first) % every == 0:
            P = torch.exp(K + u[:, :, None] + v[:, None, :])
            e = error(P.sum(2), a) if rows_first else error(P.sum(1), b)
            if e < stop:
                break
    return u, v


def _plan64(M, u, v, reg):
    return torch.exp(u[:, :, None] + v[:, None, :] - M / reg)


def _sq64(x, y):
    """As differences: no cancellation for near points."""
    out = torch.zeros((*x.shape[:-1], y.shape[-2]), dtype=torch.float64, device=x.device)
    for k in range(x.shape[-1]):
        out += (x[..., :, None, k] - y[..., None, :, k]).square()
    return out


def _stabilized64(M, a, b, reg, iters, stop=1e-9, tau=1e3):
    n, m = M.shape
    al, be = torch.zeros_like(a), torch.zeros_like(b)
    u, v = torch.full_like(a, 1.0 / n), torch.full_like(b, 1.0 / m)

    def kernel():
        return torch.exp((al[:, None] + be[None, :] - M) / reg)

    def plan():
        return torch.exp((al[:, None] + be[None, :] - M) / reg + u.log()[:, None] + v.log()[None])

    K = kernel()
    for i in range(iters):
        v = b / (K.t() @ u)
        u = a / (K @ v)
        if max(u.abs().max(), v.abs().max()) > tau:
            al, be = al + reg * u.log(), be + reg * v.log()
            u, v = torch.full_like(a, 1.0 / n), torch.full_like(b, 1.0 / m)
            K = kernel()
        if i % 20 == 0 and (plan().sum(0) - b).norm() <= stop:
            break
    return plan()


def _gromov64(s, reg, alpha=0.5, outer=20):
    C1, C2, M, a, b = (s[k] for k in ("C1", "C2", "M", "a", "b"))

    def product(T, p, q):
        const = (C1.square() @ p[..., None]) + (C2.square() @ q[..., None]).transpose(1, 2)
        return const - 2.0 * (C1 @ T) @ C2.transpose(1, 2).contiguous()

    T = a[:, :, None] * b[:, None, :] / (a.sum(1) * b.sum(1)).sqrt()[:, None, None]
    log_T = (T + 1e-15).log()
    for _ in range(outer):
        K = log_T - ((1 - alpha) * M + 2 * alpha * product(T, a, b)) / reg
        u, v = _sinkhorn64(-K, a, b, 1.0, None, 50, 1e-5, rows_first=True)
        last, log_T = T, K + u[:, :, None] + v[:, None, :]
        T = log_T.exp()
        if (T - last).abs().mean((1, 2)).max() < 1e-5:
            break
    quad = (product(T, T.sum(2), T.sum(1)) * T).sum((1, 2))
    return {"plan": T, "value": (1 - alpha) * (M * T).sum((1, 2)) + alpha * quad,
            "value_quad": alpha * quad}


def _graph64(case, s):
    """Each problem to its own stop, in groups of like size (padded with
    weights of zero)."""
    ns, ms = s["ns"], s["ms"]
    xs, ys = s["X"].double().split(ns.tolist()), s["Y"].double().split(ms.tolist())
    us, vs = [None] * len(ns), [None] * len(ns)
    order = np.argsort(ns * ms)
    for k in range(0, len(order), 32):
        ids = order[k:k + 32]
        n, m = int(ns[ids].max()), int(ms[ids].max())
        K = torch.full((len(ids), n, m), -math.inf, dtype=torch.float64, device="cuda")
        la = torch.full((len(ids), n), -math.inf, dtype=torch.float64, device="cuda")
        lb = torch.full((len(ids), m), -math.inf, dtype=torch.float64, device="cuda")
        for j, p in enumerate(ids):
            C = _sq64(xs[p], ys[p])
            K[j, :ns[p], :ms[p]] = -C / (C.max() * s["regs"][p])
            la[j, :ns[p]], lb[j, :ms[p]] = -math.log(ns[p]), -math.log(ms[p])
        left = torch.arange(len(ids), device="cuda")
        u = torch.zeros_like(la)
        for i in range(2000):
            v = (lb - torch.logsumexp(K + u[:, :, None], 1)).nan_to_num_(neginf=-math.inf)
            v[lb == -math.inf] = -math.inf
            u = la - torch.logsumexp(K + v[:, None, :], 2)
            u[la == -math.inf] = -math.inf
            if i % 10 == 0 or i == 1999:
                P = torch.exp(K + u[:, :, None] + v[:, None, :])
                ok = (P.sum(1) - lb.exp()).norm(dim=1) < 1e-6
                if i == 1999:
                    ok[:] = True
                for j in torch.nonzero(ok).flatten().tolist():
                    p = ids[int(left[j])]
                    us[p], vs[p] = u[j, :ns[p]].clone(), v[j, :ms[p]].clone()
                go = ~ok
                if not bool(go.any()):
                    break
                if bool(ok.any()):
                    K, la, lb, u, left = K[go], la[go], lb[go], u[go], left[go]
    return {"u": torch.cat(us), "v": torch.cat(vs)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "points_warm":
        return None  # the start that the network predicts is part of the result
    if kind == "points_graph" and case["B"] * (0.5 * (case["lo"] + case["hi"])) ** 2 > 2e8:
        return None  # too long in 64 bits
    s = _inputs(case, seed)
    if kind == "gromov":
        return _gromov64(s, case["reg"])
    if kind == "points_graph":
        return _graph64(case, s)
    if kind == "stabilized":
        return _stabilized64(s["M"], s["a"], s["b"], case["reg"], case["iters"])
    if kind in ("knopp_small", "knopp_f32", "log_f64", "log_large"):
        M, a, b = (s[k].double()[None] for k in ("M", "a", "b"))
        knopp = kind.startswith("knopp")
        u0 = torch.full_like(a, -math.log(a.shape[1]) if knopp else 0.0)
        if kind == "log_large":
            iters, stop = case["iters"], 0.0
        else:
            iters, stop = 1000, 1e-6 if kind == "knopp_f32" else 1e-9
        s.clear()
        u, v = _sinkhorn64(M, a, b, case["reg"], u0, iters, stop)
        P = _plan64(M, u, v, case["reg"])[0]
        if kind != "log_f64":
            return P
        return {"plan": P, "log_u": u[0], "log_v": v[0], "niter": None}
    if kind == "batch":
        M, a, b, reg = s["M"].double(), s["a"].double(), s["b"].double(), case["reg"]
        u, v = _sinkhorn64(M, a, b, reg, None, 1000, 1e-5, rows_first=True)
        P = _plan64(M, u, v, reg)
        lin = (M * P).sum((1, 2))
        pots = (u, v)
        if case["solver"] == "sinkhorn":
            pots = (u.exp(), v.exp())
        return {"plan": P, "value": lin + reg * (P * (P + 1e-16).log()).sum((1, 2)),
                "value_linear": lin, "potentials": pots}
    if kind == "batch_grad":
        X, Y, reg = s["X"].double(), s["Y"].double(), case["reg"]
        a = torch.full(X.shape[:2], 1.0 / X.shape[1], dtype=torch.float64, device="cuda")
        b = torch.full(Y.shape[:2], 1.0 / Y.shape[1], dtype=torch.float64, device="cuda")
        M = _sq64(X, Y)
        u, v = _sinkhorn64(M, a, b, reg, None, 1000, 1e-5, rows_first=True)
        P = _plan64(M, u, v, reg)
        return {"value": (M * P).sum((1, 2)) + reg * (P * (P + 1e-16).log()).sum((1, 2)),
                "plan": P, "dX": 2.0 * (P.sum(2)[..., None] * X - P @ Y),
                "dY": 2.0 * (P.sum(1)[..., None] * Y - P.transpose(1, 2).contiguous() @ X)}
    X, Y = s["X"].double(), s["Y"].double()
    if kind == "online":
        M = _sq64(X, Y)
        M /= M.max()
        a, b = s["a"][None], s["b"][None]
        u, v = _sinkhorn64(M[None], a, b, case["reg"], torch.zeros_like(a), case["iters"], 0.0)
        return {"u": u[0], "v": v[0]}
    n, m = case["n"], case["m"]
    a = torch.full((1, n), 1.0 / n, dtype=torch.float64, device="cuda")
    b = torch.full((1, m), 1.0 / m, dtype=torch.float64, device="cuda")
    M = _sq64(X, Y)[None]
    # rows first, and the source marginal is looked at after the target update
    u, v = _sinkhorn64(M, a, b, case["reg"], None, 1000, 1e-5, rows_first=True, first=9,
                       error=lambda p, w: (p - w).abs().sum())
    return {"loss": (M * _plan64(M, u, v, case["reg"])).sum(), "f": u[0], "g": v[0]}
