"""Performance cases: ensemble solves and gradients as a program runs them.

Each case is one call of ``tsit5.solve`` or ``rodas5P.solve`` (the gradient
cases with their backward pass) on inputs that are already on the GPU, the way
a parameter scan, a likelihood or a training loop calls them. Families:

  lorenz     Tsit5, 3 variables, rho ~ U[0, 28], 20 saves over [0, 1]: the
             smallest calls, a few thousand trajectories at most
  scatter    Tsit5, Lorenz from scattered initial states over [0, 5], two
             saves: a large non-stiff scan that returns endpoints
  bbn        Rodas5P FP32, the four-species nucleosynthesis network over its
             prior box (exp, sqrt, a 1.5 power): a likelihood evaluation
  robertson  Rodas5P, dense 3x3, lognormal rates, 50 log-spaced saves: the
             stiff scan this package is quoted on; FP32 or FP64 LU
  divergent  Rodas5P, dense 3x3, rates and initial states spread over a decade,
             five saves: lanes whose step counts differ
  ring       Rodas5P, stiff Van der Pol ring, sparse or dense LU: mid-sized
             coupled systems, a thousand trajectories
  nonstiff   Tsit5, the same ring with mu = 1
  ring_grad  Rodas5P, value and gradient in the rate by forward sensitivities
  arrow      Rodas5P FP32, block-arrow systems whose step counts spread over
             two decades: the large uneven ensemble
  fit        Rodas5P FP64, squared-error loss of a Van der Pol chain against
             data, gradient in the initial state and the rate by the discrete
             adjoint: 2 variables (dense) up to 20 (sparse)
"""

import functools
import math

import numpy as np
import torch

from menodax_amd import rodas5P, tsit5

DEV = "cuda"
F64 = torch.float64


# --- the systems: the callback solve() takes, and the same right-hand side over
# --- (N, n) tensors for exact() ------------------------------------------------
def lorenz(y, t, p):
    sigma = 10.0
    beta = 8.0 / 3.0
    return (
        sigma * (y[1] - y[0]),
        y[0] * (p[0] - y[2]) - y[1],
        y[0] * y[1] - beta * y[2],
    )


def robertson(y, t, p):
    return (
        -p[0] * y[0] + p[1] * y[1] * y[2],
        p[0] * y[0] - p[1] * y[1] * y[2] - p[2] * y[1] ** 2,
        p[2] * y[1] ** 2,
    )


BBN_Q = 1.293


def _bbn(exp, sqrt):
    tau_n = 879.4 / 6.582119e-22
    pi = math.pi

    def bbn(y, x, p):
        eta = 10.0 ** (p[0] - 10.0)
        temp = BBN_Q / x
        g_star = 3.91 + (10.75 - 3.91) * (temp > 0.511) + (7.0 / 4.0) * (p[1] - 3.044)
        hubble = sqrt(4.0 * pi ** 3 * g_star / 45.0) * temp ** 2 / 1.2209e22
        n_b = eta * (2.0 * 1.2020569 / pi ** 2 * temp ** 3)
        gamma_np = (255.0 / tau_n) * (12.0 + 6.0 * x + x ** 2) / x ** 5 + 1.0 / tau_n
        gamma_pn = gamma_np * exp(-x)
        k_d = n_b * (3.0 / 4.0) * (4.0 * pi / (938.272 * temp)) ** 1.5 * exp(2.225 / temp)
        r_np = n_b * 4.0e-11 * (y[0] * y[1] - y[2] / k_d)
        r_dd = n_b * 3.4e-5 * y[2] ** 2
        den = hubble * x
        return (
            (gamma_pn * y[1] - gamma_np * y[0] - r_np) / den,
            (gamma_np * y[0] - gamma_pn * y[1] - r_np) / den,
            (r_np - 2.0 * r_dd) / den,
            r_dd / den,
        )

    return bbn


bbn = _bbn(math.exp, math.sqrt)


@functools.lru_cache(maxsize=None)
def vdp(n_osc, mu, d, wrap):
    """A lattice of Van der Pol oscillators: the callback (p[0] scales ``mu``)
    and the Jacobian's sparsity mask; a ring, or with ``wrap`` false a chain."""
    mask = np.zeros((2 * n_osc, 2 * n_osc), dtype=bool)
    parts = []
    for o in range(n_osc):
        i, j = 2 * o, 2 * o + 1
        x, v = f"y[{i}]", f"y[{j}]"
        near = [(o + s) % n_osc if wrap else o + s for s in (-1, 1)]
        near = [m for m in near if 0 <= m < n_osc and m != o]
        mask[i, j] = mask[j, i] = mask[j, j] = True
        for m in near:
            mask[j, 2 * m] = True
        lap = " + ".join([f"y[{2 * m}]" for m in near] + [f"-{float(len(near))!r} * {x}"])
        parts += [f"({v}) + 0.0",
                  f"(p[0] * {mu!r} * (1.0 - {x} * {x}) * {v} + -1.0 * {x} + {d!r} * ({lap})) + 0.0"]
    return _callback("vdp", parts), mask


@functools.lru_cache(maxsize=None)
def arrow(n):
    """dy/dt = A y + 0.01 y*y, A block arrow: 2x2 rotation blocks, a lone
    variable and a hub that every other variable feeds."""
    rng = np.random.default_rng(7)
    terms = [[f"p[{j}] * y[{j}]"] for j in range(n)]
    mask = np.eye(n, dtype=bool)
    for k in range((n - 2) // 2):
        b = 2 * k
        terms[b].append(f"p[{n + k}] * y[{b + 1}]")
        terms[b + 1].append(f"-p[{n + k}] * y[{b}]")
        mask[b, b + 1] = mask[b + 1, b] = True
    for j in range(n - 1):
        terms[n - 1].append(f"{float(rng.uniform(-0.2, 0.2))!r} * y[{j}]")
    mask[n - 1, :] = mask[:, n - 1] = True
    parts = ["(" + " + ".join(t) + f" + 0.01 * (y[{j}] * y[{j}])) + 0.0" for j, t in enumerate(terms)]
    return _callback("arrow", parts), mask


def _callback(name, parts):
    space = {}
    exec("def %s(y, t, p):\n    return (\n        %s,\n    )\n" % (name, ",\n        ".join(parts)), space)
    return space[name]


def _columns(f):
    """A callback over (N, n) tensors."""
    def over(t, y, p):
        return torch.stack([c + 0.0 * y[:, 0] for c in f(y.unbind(1), t, p.unbind(1))], 1)
    return over


def _lattice(mu, d, wrap):
    def over(t, y, p):
        x, v = y[:, 0::2], y[:, 1::2]
        if wrap:
            lap = x.roll(1, 1) + x.roll(-1, 1) - 2.0 * x
        elif x.shape[1] == 1:
            lap = 0.0 * x
        else:
            step = x[:, 1:] - x[:, :-1]
            lap = torch.cat([step, 0.0 * x[:, :1]], 1) - torch.cat([0.0 * x[:, :1], step], 1)
        dv = p[:, :1] * mu * (1.0 - x * x) * v - x + d * lap
        return torch.stack([v, dv], 2).flatten(1)
    return over


# --- the cases -------------------------------------------------------------------
def listed():
    return [
        {"name": "lorenz_1024", "family": "lorenz", "n": 1024},
        {"name": "scatter_100000", "family": "scatter", "n": 100000},
        {"name": "bbn_1024", "family": "bbn", "n": 1024},
        {"name": "robertson_65536", "family": "robertson", "n": 65536, "lu": "fp32"},
        {"name": "divergent_30011_fp64", "family": "divergent", "n": 30011, "lu": "fp64"},
        {"name": "ring64_sparse_1000", "family": "ring", "n": 1000, "osc": 32, "sparse": True, "lu": "fp32"},
        {"name": "ring32_dense_1000_fp64", "family": "ring", "n": 1000, "osc": 16, "sparse": False, "lu": "fp64"},
        {"name": "nonstiff64_1000", "family": "nonstiff", "n": 1000, "osc": 32},
        {"name": "ring64_grad_1000", "family": "ring_grad", "n": 1000, "osc": 32},
        {"name": "arrow50_100000", "family": "arrow", "n": 100000, "vars": 50},
        {"name": "fit2_8192", "family": "fit", "n": 8192, "osc": 1},
        {"name": "fit20_8192", "family": "fit", "n": 8192, "osc": 10},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["lorenz", "scatter", "bbn", "robertson", "divergent", "ring", "nonstiff", "ring_grad",
                         "arrow", "fit"])
    c = {"family": family}
    if family in ("lorenz", "bbn"):
        c["n"] = _log_int(rng, 64, 8192)
    elif family in ("scatter", "robertson", "divergent"):
        c["n"] = _log_int(rng, 1000, 200000)
    elif family in ("ring", "nonstiff", "ring_grad"):
        c["n"] = _log_int(rng, 100, 2000)
        c["osc"] = rng.randint(6, 32)
    elif family == "arrow":
        c["n"] = _log_int(rng, 1000, 60000)
        c["vars"] = rng.randint(20, 50)
    else:
        c["n"] = _log_int(rng, 500, 8192)
        c["osc"] = rng.randint(1, 10)
    if family in ("robertson", "divergent"):
        c["lu"] = rng.choice(["fp32", "fp64"])
    if family == "ring":
        c["sparse"] = rng.random() < 0.7
        c["lu"] = rng.choice(["fp32", "fp64"])
    return c


TIMES = {
    "lorenz": np.linspace(0.0, 1.0, 20),
    "scatter": np.array([0.0, 5.0]),
    "bbn": np.array([BBN_Q / 10.0, BBN_Q / 0.01]),
    "robertson": np.concatenate([[0.0], np.logspace(-5.0, 5.0, 49)]),
    "divergent": np.array([0.0, 1e-6, 1e-2, 1e2, 1e5]),
    "ring": np.linspace(0.0, 1.0, 5),
    "nonstiff": np.linspace(0.0, 1.0, 5),
    "ring_grad": np.linspace(0.0, 1.0, 5),
    "arrow": np.linspace(0.0, 10.0, 20),
    "fit": np.linspace(0.0, 3.0, 20),
}


def _inputs(case, seed):
    """(y0, params, data) on the GPU; ``data`` is what a fit compares with."""
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    n, family = case["n"], case["family"]

    def uniform(lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(*shape, generator=g, device=DEV, dtype=F64)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=DEV, dtype=F64)

    if family == "lorenz":
        y0 = torch.tensor([1.0, 0.0, 0.0], device=DEV, dtype=F64).repeat(n, 1)
        return y0, uniform(0.0, 28.0, n, 1), None
    if family == "scatter":
        y0 = torch.tensor([1000.0, -500.0, 500.0], device=DEV, dtype=F64) * (1.0 - uniform(0.0, 1.0, n, 1))
        return y0, 0.5 * uniform(0.95, 1.05, n, 1), None
    if family == "bbn":
        x0 = BBN_Q / 10.0
        y0 = torch.tensor([math.exp(-x0) / (1.0 + math.exp(-x0)), 1.0 / (1.0 + math.exp(-x0)), 1e-20, 0.0],
                          device=DEV, dtype=F64)
        return y0, torch.cat([uniform(0.5, 1.0, n, 1), uniform(2.0, 4.0, n, 1)], 1), None
    rates = torch.tensor([0.04, 1e4, 3e7], device=DEV, dtype=F64)
    if family == "robertson":
        y0 = torch.tensor([1.0, 0.0, 0.0], device=DEV, dtype=F64).repeat(n, 1)
        return y0, rates * torch.exp(0.3 * normal(n, 3)), None
    if family == "divergent":
        alpha = 0.99 * uniform(0.0, 1.0, n)
        eps = 10.0 ** (-1.0 - 7.0 * uniform(0.0, 0.25, n))
        y0 = torch.stack([(1 - eps) * alpha, eps, (1 - eps) * (1 - alpha)], 1)
        return y0, rates * 10.0 ** uniform(-1.0, 1.0, n, 3), None
    if family in ("ring", "nonstiff", "ring_grad"):
        osc = case["osc"]
        target = uniform(0.25, 3.0, n, osc) * torch.sign(uniform(-1.0, 1.0, n, osc))
        x = 2.0 + 0.1 * (target - 2.0)
        return torch.stack([x, 0.2 * normal(n, osc)], 2).flatten(1), uniform(0.95, 1.05, n, 1), None
    if family == "arrow":
        v = case["vars"]
        ceiling = uniform(1.0, 5.0, n, 1)
        lam = -(10.0 ** (-1.0 + uniform(0.0, 1.0, n, v) * (ceiling + 1.0)))
        scale = torch.exp(uniform(math.log(0.05), math.log(200.0), n, 1))
        return uniform(-1.0, 1.0, n, v), torch.cat([lam, scale * uniform(0.5, 1.5, n, (v - 2) // 2)], 1), None
    nv = 2 * case["osc"]
    data = uniform(-2.0, 2.0, n, 1, nv) * torch.cos(torch.linspace(0.0, 3.0, 20, device=DEV, dtype=F64))[:, None]
    return uniform(-2.0, 2.0, n, nv), 10.0 ** uniform(1.0, 2.0, n, 1), data


def _system(case):
    """(callback, the same over tensors or None, stiff, solve, its options)"""
    family = case["family"]
    quoted = dict(rtol=1e-6, atol=1e-8)
    if family in ("lorenz", "scatter"):
        first = {"first_step": 1e-4} if family == "scatter" else {}
        return lorenz, _columns(lorenz), False, tsit5.solve, dict(quoted, **first)
    if family == "bbn":
        return bbn, _columns(_bbn(torch.exp, torch.sqrt)), True, rodas5P.solve, dict(
            lu_precision="fp32", rtol=1e-4, atol=1e-9, first_step=0.1, max_steps=256)
    if family in ("robertson", "divergent"):
        return robertson, _columns(robertson), True, rodas5P.solve, dict(quoted, lu_precision=case["lu"])
    if family == "nonstiff":
        fn, _ = vdp(case["osc"], 1.0, 10.0, True)
        return fn, _lattice(1.0, 10.0, True), False, tsit5.solve, dict(quoted, first_step=1e-4)
    if family in ("ring", "ring_grad"):
        fn, mask = vdp(case["osc"], 100.0, 10.0, True)
        return fn, _lattice(100.0, 10.0, True), True, rodas5P.solve, dict(
            quoted, first_step=1e-4, lu_precision=case.get("lu", "fp32"),
            sparsity=mask if case.get("sparse", True) else None)
    if family == "arrow":
        fn, mask = arrow(case["vars"])
        return fn, None, True, rodas5P.solve, dict(quoted, lu_precision="fp32", sparsity=mask)
    fn, mask = vdp(case["osc"], 1.0, 0.1, False)
    return fn, _lattice(1.0, 0.1, False), True, rodas5P.solve, dict(
        rtol=1e-8, atol=1e-10, lu_precision="fp64", sparsity=mask if case["osc"] > 1 else None)


def prepare(case, seed):
    y0, p, data = _inputs(case, seed)
    fn, _, _, solve, kw = _system(case)
    # a scan's time grid lives on the GPU with its inputs; the likelihood's is
    # the pair of constants its author wrote
    t = torch.tensor(TIMES[case["family"]], device=DEV)
    if case["family"] == "bbn":
        t = TIMES["bbn"]
    return {"family": case["family"], "fn": fn, "solve": solve, "kw": kw, "y0": y0, "p": p, "t": t, "data": data}


def run(s):
    solve, kw = s["solve"], s["kw"]
    if s["family"] == "ring_grad":
        p = s["p"].detach().requires_grad_(True)
        hist = solve(s["fn"], s["y0"], s["t"], p, **kw)
        (grad,) = torch.autograd.grad(hist[:, -1].sum(), (p,))
        return {"hist": hist.detach(), "grad_p": grad}
    if s["family"] == "fit":
        y0 = s["y0"].detach().requires_grad_(True)
        p = s["p"].detach().requires_grad_(True)
        hist = solve(s["fn"], y0, s["t"], p, adjoint=True, **kw)
        grads = torch.autograd.grad(((hist - s["data"]) ** 2).sum(), (y0, p))
        return {"hist": hist.detach(), "grad_y0": grads[0], "grad_p": grads[1]}
    hist, stats = solve(s["fn"], s["y0"], s["t"], s["p"], return_stats=True, **kw)
    return {"hist": hist, "stats": stats}


# --- the least work ----------------------------------------------------------------
#: accepted plus rejected steps of a trajectory, on average
STEPS = {"lorenz": 45, "scatter": 415, "bbn": 124, "robertson": 95, "divergent": 110, "ring": 36, "nonstiff": 24,
         "ring_grad": 36, "arrow": 719, "fit": 195}


def work(case):
    """Bytes: inputs, history and counters (and gradients) once each. Flops: the
    method's stage sums and right-hand sides (about eight operations a component)
    over the average steps, and the dense elimination where the LU is dense; a
    gradient's backward pass as twice its forward pass."""
    family, n = case["family"], case["n"]
    nv = {"lorenz": 3, "scatter": 3, "bbn": 4, "robertson": 3, "divergent": 3}.get(family) or case.get("vars") or 2 * case["osc"]
    n_p = {"bbn": 2, "robertson": 3, "divergent": 3}.get(family, 1)
    if family == "arrow":
        n_p = nv + (nv - 2) // 2
    saves = len(TIMES[family])
    explicit = family in ("lorenz", "scatter", "nonstiff")
    step = nv * ((6 * 8 + 44) if explicit else (8 * 8 + 105))
    if not explicit:
        dense = nv <= 4 or not case.get("sparse", True)
        step += 2 * nv ** 3 // 3 + 16 * nv * nv if dense else 8 * 12 * nv + 20 * nv
    flops = n * STEPS[family] * step * (3 if family == "fit" and nv > 2 else 1)
    size = 8 * n * (nv + n_p + saves * nv) + 12 * n
    if family == "ring_grad":
        flops, size = 2 * flops, size + 8 * n * n_p
    if family == "fit":
        flops, size = 3 * flops, size + 8 * n * (nv + n_p + saves * nv)
    return {"bytes": size, "flops": flops}


# --- 64-bit values -------------------------------------------------------------------
def _jacobian(f, y):
    """df/dy of f(y) (N, ...), the derivative's axis last."""
    cols = []
    for j in range(y.shape[1]):
        e = torch.zeros_like(y)
        e[:, j] = 1.0
        cols.append(torch.func.jvp(f, (y,), (e,))[1])
    return torch.stack(cols, -1)


def _tangent(f, t, y, s, p, pd):
    """J(y) s + f_p pd for s of (N, n, m) and pd of (n_p, m)."""
    m = s.shape[2]
    wide = lambda x: x.repeat_interleave(m, 0)  # noqa: E731
    flat = s.transpose(1, 2).flatten(0, 1)
    dp = pd.t().repeat(y.shape[0], 1)
    out = torch.func.jvp(lambda z, q: f(wide(t), z, q), (wide(y), wide(p)), (flat, dp))[1]
    return out.unflatten(0, (-1, m)).transpose(1, 2)


def _integrate(f, stiff, y, times, p, s=None, pd=None, columns=8, rtol=1e-9, atol=1e-13):
    """y (and the sensitivities s) at ``times`` by extrapolation of the linearly
    implicit Euler rule (of Euler's rule where the system is not stiff), every
    trajectory with steps of its own."""
    n, nv = y.shape
    t = torch.full((n,), float(times[0]), device=DEV, dtype=F64)
    h = torch.full((n,), float(times[-1] - times[0]) * 1e-6, device=DEV, dtype=F64)
    grid = torch.tensor(times, device=DEV, dtype=F64)
    at = torch.ones(n, dtype=torch.long, device=DEV)
    eye = torch.eye(nv, device=DEV, dtype=F64)
    hist = y[:, None].repeat(1, len(times), 1)
    sens = None if s is None else s[:, None].repeat(1, len(times), 1, 1)
    rows = torch.arange(n, device=DEV)
    for _ in range(4000):
        live = at < len(times)
        if not bool(live.any()):
            return hist, sens
        goal = grid[at.clamp(max=len(times) - 1)]
        dt = torch.where(live, torch.minimum(h, goal - t), torch.zeros_like(h))
        J = _jacobian(lambda z: f(t, z, p), y) if stiff else None
        C = None if s is None else _jacobian(lambda z: _tangent(f, t, z, s, p, pd), y)
        table = []
        for k in range(1, columns + 1):
            hk = dt / k
            lu = torch.linalg.lu_factor(eye - hk[:, None, None] * J) if stiff else None
            yk, sk = y, s
            for i in range(k):
                ti = t + hk * (i + 1) if stiff else t + hk * i
                dy = hk[:, None] * f(ti, yk, p)
                if stiff:
                    dy = torch.linalg.lu_solve(*lu, dy[:, :, None])[:, :, 0]
                if s is not None:
                    couple = torch.einsum("nimj,nj->nim", C, dy)
                    g = hk[:, None, None] * (_tangent(f, ti, yk, sk, p, pd) + couple)
                    sk = sk + torch.linalg.lu_solve(*lu, g)
                yk = yk + dy
            row = [yk if s is None else torch.cat([yk, sk.flatten(1)], 1)]
            for m in range(1, k):
                row.append(row[-1] + (row[-1] - table[-1][m - 1]) / (k / (k - m) - 1.0))
            table.append(row)
        new, low = table[-1][-1], table[-1][-2]
        old = y if s is None else torch.cat([y, s.flatten(1)], 1)
        scale = atol + rtol * torch.maximum(old.abs(), new.abs()).clamp(min=1e-3 if s is not None else 0.0)
        err = ((new - low) / scale).abs().amax(1).nan_to_num(nan=1e10, posinf=1e10).clamp(1e-10, 1e10)
        ok = live & (err <= 1.0)
        there = ok & (dt >= goal - t)
        factor = (0.8 * err ** (-1.0 / columns)).clamp(0.1, 5.0)
        h = torch.where(live, torch.where(ok, torch.maximum(h * factor.clamp(max=1.0), dt * factor), dt * factor), h)
        t = torch.where(there, goal, torch.where(ok, t + dt, t))
        y = torch.where(ok[:, None], new[:, :nv], y)
        if s is not None:
            s = torch.where(ok[:, None, None], new[:, nv:].reshape(s.shape), s)
            sens[rows[there], at[there]] = s[there]
        hist[rows[there], at[there]] = y[there]
        at = at + there
    return None, None


def exact(case, seed):
    """The solution of the differential equations themselves; None for the
    counters, and for what takes too long: the uneven ensemble, and gradients
    of coupled systems."""
    y0, p, data = _inputs(case, seed)
    fn, f, stiff, _, _ = _system(case)
    family, times = case["family"], TIMES[case["family"]]
    if f is None or (family == "fit" and case["osc"] > 1):
        return None
    n, nv = case["n"], y0.shape[-1]
    y0 = y0.expand(n, nv).contiguous()
    if family == "fit":
        s = torch.eye(nv, nv + 1, device=DEV, dtype=F64).repeat(n, 1, 1)
        pd = torch.zeros(1, nv + 1, device=DEV, dtype=F64)
        pd[0, nv] = 1.0
        hist, sens = _integrate(f, stiff, y0, times, p, s, pd)
        if hist is None:
            return None
        grad = torch.einsum("nsi,nsik->nk", 2.0 * (hist - data), sens)
        return {"hist": hist, "grad_y0": grad[:, :nv], "grad_p": grad[:, nv:]}
    hist, _ = _integrate(f, stiff, y0, times, p)
    if hist is not None and family == "ring_grad":
        return {"hist": hist, "grad_p": None}
    return None if hist is None else {
        "hist": hist, "stats": {k: None for k in ("accepted_steps", "rejected_steps", "loop_steps")}}
