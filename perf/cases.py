"""Workloads of ripley_hip as its users run them, for timing one revision of
the library against another.

A case is a dict of plain values.  ``prepare`` makes what a program holds
before the call (coefficient fields on the GPU, the PDE object with its
operator, a network), ``run`` is one pass through the public entry points
and returns what the program gets, ``work`` the bytes and operations the
pass cannot do without, ``exact`` the same outputs in 64-bit torch.

Kinds of work:

* ``poisson``     LinearPDE.getSolution of a scalar PDE from new coefficients:
                  assemble, constrain, solve.  Every Krylov method and
                  preconditioner is an option.
* ``advection``   the same for a non-symmetric PDE (convection, reaction,
                  coefficients on quadrature points): BiCGStab.
* ``elasticity``  the same for linear elasticity (block size = dimension).
* ``system``      getSystem of a general coupled PDE and the product with its
                  operator: one explicit time step.
* ``many_rhs``    one operator, many right-hand sides (solve_many).
* ``batch``       many uneven independent systems solved together.
* ``train``       loss and gradients of the learned preconditioner's network.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "esys-escript.github.io_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import ripley_hip as R  # noqa: E402
from ripley_hip import batch as RB  # noqa: E402
from ripley_hip import learned as RL  # noqa: E402

_WEIGHTS = os.path.join(_PKG, "ripley_hip", "weights", "lpc_coarse_log10grf_s1_l8.npy")


def listed():
    return [
        # the smallest call: one step of a coarse 2-D model, where latency,
        # launches and host work are all there is
        {"name": "poisson_rect_smallest", "kind": "poisson", "n0": 20, "n1": 13, "n2": 0, "method": "PCG",
         "prec": "JACOBI", "sym": True, "field": "ln", "sigma": 1.0, "corr": 4.0, "tol": 1e-8},
        # the reference's CPU-sized Poisson problem: Rectangle 256 x 256,
        # unit coefficient, PASO's default solver on full storage
        {"name": "poisson_rect_256", "kind": "poisson", "n0": 256, "n1": 256, "n2": 0, "method": "PCG",
         "prec": "JACOBI", "sym": False, "field": "one", "sigma": 0.0, "corr": 8.0, "tol": 1e-8},
        # an ordinary 3-D model with odd sides, default solver
        {"name": "poisson_brick_odd", "kind": "poisson", "n0": 61, "n1": 47, "n2": 53, "method": "PCG",
         "prec": "JACOBI", "sym": True, "field": "ln", "sigma": 1.0, "corr": 8.0, "tol": 1e-8},
        # the headline: heterogeneous Poisson on Brick 128^3, textbook PCG
        {"name": "poisson_brick_128_plain", "kind": "poisson", "n0": 128, "n1": 128, "n2": 128,
         "method": "PCG_PLAIN", "prec": "JACOBI", "sym": True, "field": "log10", "sigma": 1.0, "corr": 8.0,
         "tol": 1e-8},
        # the same problem with the multigrid flexible CG and its trained
        # network, the fastest way to that solution
        {"name": "poisson_brick_128_learned", "kind": "poisson", "n0": 128, "n1": 128, "n2": 128,
         "method": "FCG_LEARNED", "prec": "NETWORK", "sym": True, "field": "log10", "sigma": 1.0, "corr": 8.0,
         "tol": 1e-8},
        # PASO's stronger preconditioner on a mid-size model
        {"name": "poisson_brick_96_gauss_seidel", "kind": "poisson", "n0": 96, "n1": 95, "n2": 97, "method": "PCG",
         "prec": "GAUSS_SEIDEL", "sym": False, "field": "log10", "sigma": 1.0, "corr": 8.0, "tol": 1e-8},
        # convection and reaction: the non-symmetric default, full storage
        {"name": "advection_brick", "kind": "advection", "n0": 63, "n1": 64, "n2": 40, "speed": 20.0, "react": 1.0,
         "tol": 1e-10},
        # layered elasticity under gravity, Brick 96^3, 3 x 3 blocks
        {"name": "elasticity_brick_96", "kind": "elasticity", "n0": 96, "n1": 96, "n2": 96, "layers": 8,
         "method": "PCG", "tol": 1e-8},
        # explicit step of a coupled PDE with every coefficient, on
        # quadrature points
        {"name": "system_brick_48", "kind": "system", "n0": 48, "n1": 47, "n2": 49, "eq": 3, "expanded": True},
        # 64 point loads on one operator (the largest case)
        {"name": "many_rhs_brick_96", "kind": "many_rhs", "n0": 96, "n1": 96, "n2": 96, "rhs": 64,
         "method": "PCG_MIXED", "sigma": 1.5, "corr": 8.0, "tol": 1e-8},
        # an ensemble of uneven 2-D models
        {"name": "batch_rectangles", "kind": "batch", "count": 24, "lo": 64, "hi": 400, "method": "PCG_MIXED",
         "sigma": 1.0, "corr": 8.0, "tol": 1e-8, "sizes": 7},
        # one gradient of the network's training, on the level it corrects
        {"name": "train_17", "kind": "train", "n0": 17, "n1": 17, "n2": 17, "corr": 3.0, "sigma": 1.0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["poisson"] * 8 + ["advection"] * 2 + ["elasticity"] * 2 + ["system", "many_rhs", "batch", "train"])
    if kind == "poisson":
        flat = rng.random() < 0.4
        base = _log_int(rng, 8, 512) if flat else _log_int(rng, 6, 112)
        side = [max(4, int(base * rng.uniform(0.7, 1.3))) for _ in range(2 if flat else 3)]
        method, prec = rng.choice([("PCG", "JACOBI")] * 3 + [("PCG_PLAIN", "JACOBI")] * 3 +
                                  [("MINRES", "JACOBI"), ("PCG_MIXED", "JACOBI"), ("PCG", "GAUSS_SEIDEL"),
                                   ("PCG", "ILU0")] + ([] if flat else [("FCG_LEARNED", "NONE")] * 2))
        if method == "FCG_LEARNED":
            side = [8 * max(2, round(s / 8)) for s in side]
        if prec in ("GAUSS_SEIDEL", "ILU0"):
            side = [min(s, 300 if flat else 90) for s in side]
        return {"kind": kind, "n0": side[0], "n1": side[1], "n2": 0 if flat else side[2], "method": method,
                "prec": prec, "sym": rng.random() < 0.7, "field": rng.choice(["ln", "log10"]),
                "sigma": round(rng.uniform(0.3, 1.0), 2), "corr": round(rng.uniform(3.0, 10.0), 1), "tol": 1e-8}
    if kind == "advection":
        base = _log_int(rng, 8, 72)
        flat = rng.random() < 0.4
        side = [max(4, int(base * rng.uniform(0.7, 1.3) * (3 if flat else 1))) for _ in range(2 if flat else 3)]
        return {"kind": kind, "n0": side[0], "n1": side[1], "n2": 0 if flat else side[2],
                "speed": round(rng.uniform(1.0, 30.0), 1), "react": round(rng.uniform(0.1, 10.0), 2), "tol": 1e-10}
    if kind == "elasticity":
        flat = rng.random() < 0.3
        base = _log_int(rng, 16, 160) if flat else _log_int(rng, 6, 72)
        side = [max(4, int(base * rng.uniform(0.7, 1.3))) for _ in range(2 if flat else 3)]
        return {"kind": kind, "n0": side[0], "n1": side[1], "n2": 0 if flat else side[2],
                "layers": rng.randrange(2, 9), "method": rng.choice(["PCG", "PCG_PLAIN", "PCG_MIXED"]), "tol": 1e-8}
    if kind == "system":
        base = _log_int(rng, 8, 48)
        return {"kind": kind, "n0": base, "n1": max(4, base + rng.randrange(-3, 4)), "n2": max(4, base + rng.randrange(-3, 4)),
                "eq": rng.randrange(1, 4), "expanded": rng.random() < 0.5}
    if kind == "many_rhs":
        base = _log_int(rng, 16, 80)
        return {"kind": kind, "n0": base, "n1": max(4, base + rng.randrange(-5, 6)), "n2": max(4, base + rng.randrange(-5, 6)),
                "rhs": rng.choice([64, 64, 64, 32, 16, 7]), "method": rng.choice(["PCG_MIXED", "PCG_MIXED", "PCG_PLAIN"]),
                "sigma": round(rng.uniform(0.5, 1.5), 2), "corr": 8.0, "tol": 1e-8}
    if kind == "batch":
        return {"kind": kind, "count": rng.randrange(4, 25), "lo": 32, "hi": _log_int(rng, 96, 384),
                "method": rng.choice(["PCG_MIXED", "PCG_PLAIN"]), "sigma": round(rng.uniform(0.5, 1.0), 2), "corr": 8.0,
                "tol": 1e-8, "sizes": rng.randrange(1 << 20)}
    side = [rng.randrange(9, 34) for _ in range(3)]
    return {"kind": kind, "n0": side[0], "n1": side[1], "n2": side[2], "corr": round(rng.uniform(2.0, 5.0), 1),
            "sigma": round(rng.uniform(0.5, 1.0), 2)}


# ------------------------------------------------------------------- inputs


def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(int(seed) * 2654435761 % (1 << 62) + 12345)
    return g


def _sides(case):
    return tuple(int(case[k]) for k in ("n0", "n1", "n2") if case[k])


def _random_field(shape, corr, gen):
    """Gaussian field of unit variance and covariance exp(-r^2 / (2 corr^2))
    (in cells) on the grid `shape` (x first), flattened x fastest."""
    pad = [int(2 * math.ceil((s + 4.0 * corr) / 2.0)) for s in shape][::-1]
    r2 = torch.zeros(pad, dtype=torch.float64, device=_dev())
    for ax, m in enumerate(pad):
        k = torch.arange(m, device=_dev())
        d = torch.minimum(k, m - k).to(torch.float64)
        r2 += (d * d).reshape([-1 if a == ax else 1 for a in range(len(pad))])
    lam = torch.fft.fftn(torch.exp(-r2 / (2.0 * corr * corr))).real.clamp_min(0.0)
    white = torch.randn(pad, dtype=torch.float64, device=_dev(), generator=gen)
    f = torch.fft.ifftn(torch.sqrt(lam) * torch.fft.fftn(white)).real
    return f[tuple(slice(0, s) for s in shape[::-1])].reshape(-1).contiguous()


def _kappa(case, sides, gen):
    E = int(np.prod(sides))
    if case.get("field") == "one":
        return torch.ones(E, dtype=torch.float64, device=_dev())
    g = case["sigma"] * _random_field(sides, case["corr"], gen)
    return torch.pow(10.0, g) if case.get("field") == "log10" else torch.exp(g)


def _source(sides, gen):
    """A source per element: uniform in [0.5, 1.5]."""
    return 0.5 + torch.rand(int(np.prod(sides)), dtype=torch.float64, device=_dev(), generator=gen)


def _centres(sides):
    """Element centres on the unit square / cube, (E, dim), x fastest."""
    ax = [(torch.arange(n, dtype=torch.float64, device=_dev()) + 0.5) / n for n in sides]
    g = torch.meshgrid(*ax[::-1], indexing="ij")
    return torch.stack([t.reshape(-1) for t in g[::-1]], dim=1)


def _quadrature(sides):
    """Coordinates (E, Q, dim) of the 2-point Gauss points, x fastest."""
    d = len(sides)
    h = torch.tensor([1.0 / n for n in sides], dtype=torch.float64, device=_dev())
    off = torch.tensor([[0.5 / math.sqrt(3.0) * (1 if (q >> a) & 1 else -1) for a in range(d)] for q in range(1 << d)],
                       dtype=torch.float64, device=_dev())
    return _centres(sides)[:, None, :] + off * h


def _advection_inputs(case, seed):
    """Diffusion per element, a recirculating velocity and a reaction on the
    quadrature points, a source per element."""
    sides = _sides(case)
    gen = _generator(seed)
    kap = torch.exp(0.5 * _random_field(sides, 6.0, gen))
    x = _quadrature(sides)
    ph = 2.0 * math.pi * torch.rand(2, dtype=torch.float64, device=_dev(), generator=gen)
    vel = torch.zeros(x.shape, dtype=torch.float64, device=_dev())
    vel[..., 0] = case["speed"] * torch.sin(math.pi * x[..., 0] + ph[0]) * torch.cos(math.pi * x[..., 1])
    vel[..., 1] = -case["speed"] * torch.cos(math.pi * x[..., 0] + ph[0]) * torch.sin(math.pi * x[..., 1])
    if len(sides) == 3:
        vel[..., 2] = 0.5 * case["speed"] * torch.sin(math.pi * x[..., 2] + ph[1])
    react = case["react"] * (1.0 + 0.5 * torch.sin(2.0 * math.pi * x[..., 0]))
    return sides, kap, vel, react, _source(sides, gen)


def _lame_inputs(case, seed):
    """Lame parameters of horizontal layers, uniform in [1e9, 5e10] Pa."""
    sides = _sides(case)
    gen = _generator(seed)
    v = 1e9 + (5e10 - 1e9) * torch.rand((2, case["layers"]), dtype=torch.float64, device=_dev(), generator=gen)
    k = torch.arange(sides[-1], device=_dev()) * case["layers"] // sides[-1]
    rep = int(np.prod(sides[:-1]))
    return sides, v[0][k].repeat_interleave(rep), v[1][k].repeat_interleave(rep)


def _lame_tensor(lam, mu, d):
    eye = torch.eye(d, dtype=torch.float64, device=lam.device)
    bl = torch.einsum("ij,kl->ijkl", eye, eye)
    bm = torch.einsum("ik,jl->ijkl", eye, eye) + torch.einsum("il,jk->ijkl", eye, eye)
    return lam[:, None, None, None, None] * bl + mu[:, None, None, None, None] * bm


def _gravity(d):
    f = [0.0] * d
    f[-1] = -2700.0 * 9.81
    return f


def _system_inputs(case, seed):
    """Every coefficient of a coupled PDE: A per element, the others per
    element or per quadrature point, and the state u it is applied to."""
    sides = _sides(case)
    d, n = len(sides), case["eq"]
    E, N = int(np.prod(sides)), int(np.prod([s + 1 for s in sides]))
    gen = _generator(seed)
    lead = (E, 1 << d) if case["expanded"] else (E,)

    def rnd(*shape):
        return torch.rand(shape, dtype=torch.float64, device=_dev(), generator=gen) - 0.5

    c = {}
    if n == 1:
        c["A"] = rnd(E, d, d) + 2.0 * torch.eye(d, dtype=torch.float64, device=_dev())
        c["B"], c["C"], c["D"], c["X"], c["Y"] = rnd(*lead, d), rnd(*lead, d), rnd(*lead) + 1.0, rnd(*lead, d), rnd(*lead)
    else:
        c["A"] = rnd(E, n, d, n, d) + 2.0 * torch.eye(n * d, dtype=torch.float64, device=_dev()).reshape(n, d, n, d)
        c["B"], c["C"], c["D"] = rnd(*lead, n, d, n), rnd(*lead, n, n, d), rnd(*lead, n, n)
        c["X"], c["Y"] = rnd(*lead, n, d), rnd(*lead, n)
    return sides, c, torch.randn(N * n, dtype=torch.float64, device=_dev(), generator=gen)


def _loads(case, seed):
    """Conductivity per element and unit point loads on random nodes of the
    top face."""
    sides = _sides(case)
    gen = _generator(seed)
    kap = _kappa(dict(case, field="ln"), sides, gen)
    plane = (sides[0] + 1) * (sides[1] + 1)
    nodes = sides[2] * plane + torch.randperm(plane, device=_dev(), generator=gen)[:case["rhs"]]
    B = torch.zeros((plane * (sides[2] + 1), case["rhs"]), dtype=torch.float64, device=_dev())
    B[nodes, torch.arange(case["rhs"], device=_dev())] = 1.0
    return sides, kap, B


def _batch_sides(case):
    rng = np.random.default_rng(case["sizes"])
    return [(int(n), int(n)) for n in rng.integers(case["lo"], case["hi"] + 1, size=case["count"])]


def _train_inputs(case, seed):
    """The level's coefficient (per element), an error field and the
    network's weights."""
    nodes = _sides(case)
    sides = tuple(n - 1 for n in nodes)
    gen = _generator(seed)
    kap = torch.exp(case["sigma"] * _random_field(sides, case["corr"], gen))
    e = _random_field(nodes, case["corr"], gen)
    e[:nodes[0] * nodes[1]] = 0.0
    return nodes, sides, kap, e, RL.init_params(int(seed) % (1 << 31))


def _domain(sides):
    return R.Rectangle(*sides) if len(sides) == 2 else R.Brick(*sides)


def _options(o, case):
    o.setTolerance(case["tol"])
    if "method" in case:
        o.setSolverMethod(getattr(R.SolverOptions, case["method"]))
        # the methods that PASO does not have stop on the true residual
        o.setTrueResidualCriterion(case["method"] in ("PCG_PLAIN", "PCG_MIXED", "FCG_LEARNED"))
    if case.get("prec") in ("JACOBI", "GAUSS_SEIDEL", "ILU0"):
        o.setPreconditioner(getattr(R.SolverOptions, case["prec"]))


def _constrained_axis(case):
    return 0 if case.get("field") == "one" else len(_sides(case)) - 1


def _operator(dom, kap, q):
    E, Q, d = dom.getNumElements(), dom.getNumQuadraturePoints(), dom.getDim()
    op = dom.newOperator(1)
    op.assemble({"A": R.Coefficient(kap, (d, d), E, Q, dom.device, isotropic=True)}, None)
    op.nullifyRowsAndCols(q, q, 1.0)
    return op


def prepare(case, seed):
    kind = case["kind"]
    if kind == "poisson":
        sides = _sides(case)
        gen = _generator(seed)
        kap, src = _kappa(case, sides, gen), _source(sides, gen)
        dom = _domain(sides)
        pde = R.LinearPDE(dom)
        if case["sym"]:
            pde.setSymmetryOn()
        pde.setValue(A=R.kronecker_scaled(kap), Y=src, q=dom.whereZero(_constrained_axis(case)))
        _options(pde.getSolverOptions(), case)
        if case["prec"] == "NETWORK":
            net = RL.LearnedPreconditioner(tuple(n // 8 + 1 for n in sides),
                                           params=np.load(_WEIGHTS, allow_pickle=False))
            pde.getOperator().setLearnedPreconditioner(net)
        return {"kind": kind, "pde": pde, "coef": {"A": R.kronecker_scaled(kap), "Y": src}}
    if kind == "advection":
        sides, kap, vel, react, src = _advection_inputs(case, seed)
        dom = _domain(sides)
        pde = R.LinearPDE(dom)
        _options(pde.getSolverOptions(), case)
        pde.setValue(q=dom.whereZero(len(sides) - 1))
        return {"kind": kind, "pde": pde, "coef": {"A": R.kronecker_scaled(kap), "C": vel, "D": react, "Y": src}}
    if kind == "elasticity":
        sides, lam, mu = _lame_inputs(case, seed)
        d = len(sides)
        dom = _domain(sides)
        pde = R.LinearPDE(dom, numEquations=d)
        pde.setSymmetryOn()
        _options(pde.getSolverOptions(), case)
        pde.setValue(q=dom.whereZero(d - 1).repeat_interleave(d))
        return {"kind": kind, "pde": pde, "coef": {"A": _lame_tensor(lam, mu, d), "Y": _gravity(d)}}
    if kind == "system":
        sides, coef, u = _system_inputs(case, seed)
        return {"kind": kind, "pde": R.LinearPDE(_domain(sides), numEquations=case["eq"]), "coef": coef, "u": u}
    if kind == "many_rhs":
        sides, kap, B = _loads(case, seed)
        dom = _domain(sides)
        q = dom.whereZero(2)
        o = R.SolverOptions()
        o.setSymmetryOn()
        _options(o, case)
        return {"kind": kind, "op": _operator(dom, kap, q), "B": B, "options": o}
    if kind == "batch":
        gen = _generator(seed)
        ops, rhs = [], []
        for sides in _batch_sides(case):
            kap, src = _kappa(dict(case, field="ln"), sides, gen), _source(sides, gen)
            dom = _domain(sides)
            q = dom.whereZero(0)
            E, Q = dom.getNumElements(), dom.getNumQuadraturePoints()
            op = dom.newOperator(1)
            f = torch.zeros(op.size, dtype=torch.float64, device=dom.device)
            op.assemble({"A": R.Coefficient(kap, (2, 2), E, Q, dom.device, isotropic=True),
                         "Y": R.Coefficient(src, (), E, Q, dom.device)}, f)
            op.nullifyRowsAndCols(q, q, 1.0)
            ops.append(op)
            rhs.append(torch.where(q > 0, torch.zeros_like(f), f))
        solver = RB.BatchSolver(ops)
        o = R.SolverOptions()
        o.setSymmetryOn()
        _options(o, case)
        return {"kind": kind, "solver": solver, "b": solver.join(rhs), "options": o}
    nodes, sides, kap, e, params = _train_inputs(case, seed)
    dom = _domain(sides)
    op = _operator(dom, kap, dom.whereZero(2))
    net = RL.LearnedPreconditioner(nodes, training=True, params=params)
    dinv, logk = RL.level_inputs(op)
    return {"kind": kind, "net": net, "op": op, "r": op * e, "e": e, "dinv": dinv, "logk": logk}


def run(state):
    kind = state["kind"]
    if kind in ("poisson", "advection", "elasticity"):
        state["pde"].setValue(**state["coef"])
        return state["pde"].getSolution()
    if kind == "system":
        state["pde"].setValue(**state["coef"])
        op, rhs = state["pde"].getSystem()
        return [rhs, op * state["u"]]
    if kind == "many_rhs":
        return RB.solve_many(state["op"], state["B"], state["options"])[0]
    if kind == "batch":
        x, _ = state["solver"].solve(state["b"], state["options"])
        return state["solver"].split(x)
    loss, grads = state["net"].gradients(state["r"], state["dinv"], state["logk"], state["e"], op=state["op"])
    return [loss, grads]


# ------------------------------------------------------------------- bounds


def work(case):
    """Coefficients, masks and right-hand sides in, solutions out; a solve
    has at least to form and apply its operator once."""
    kind = case["kind"]
    if kind == "batch":
        E = sum(a * b for a, b in _batch_sides(case))
        N = sum((a + 1) * (b + 1) for a, b in _batch_sides(case))
        return {"bytes": 8.0 * (9 * N + 2 * N), "flops": 2.0 * 9 * N + 0.0 * E}
    sides = _sides(case)
    d = len(sides)
    if kind == "train":
        return {"bytes": 4.0 * 2 * 332064 + 8.0 * 4 * float(np.prod(sides)),
                "flops": 3.0 * _network_flops(sides)}
    E, N, slots = float(np.prod(sides)), float(np.prod([s + 1 for s in sides])), 3.0 ** d
    if kind == "poisson":
        return {"bytes": 8.0 * (2 * E + 2 * N), "flops": 2.0 * slots * N + 2.0 * 4 ** d * E}
    if kind == "advection":
        return {"bytes": 8.0 * (2 * E + (d + 1) * 2 ** d * E + 2 * N), "flops": 2.0 * slots * N + 2.0 * 2 ** d * 4 ** d * E}
    if kind == "elasticity":
        return {"bytes": 8.0 * (d ** 4 * E + 2 * d * N), "flops": 2.0 * d * d * (slots * N + 4 ** d * E)}
    if kind == "system":
        n = case["eq"]
        pt = 2 * n * n * d + n * n + n * d + n
        return {"bytes": 8.0 * ((n * n * d * d + pt * (2 ** d if case["expanded"] else 1)) * E + 3 * n * N),
                "flops": 2.0 * n * n * (slots * N + (2 ** d if case["expanded"] else 1) * 4 ** d * E)}
    K = case["rhs"]
    return {"bytes": 8.0 * (slots * N + 2 * K * N), "flops": 2.0 * slots * N * K}


def _network_flops(nodes):
    v = [float(np.prod([(n + 3) // 4 * 4 // s for n in nodes])) for s in (1, 2, 4)]
    return 2.0 * 27 * (v[0] * (2 * 16 + 16 * 16 + 48 * 16 + 16) + v[1] * (16 * 32 + 32 * 32 + 96 * 32) +
                       v[2] * (32 * 64 + 64 * 64))


# ------------------------------------------------------- 64-bit expectations


class _Elements:
    """Q1 elements of the unit square / cube, `n` unknowns per node (node
    major): gather to and scatter from element vectors (E, 2^d * n)."""

    def __init__(self, sides, n=1):
        self.sides, self.n, self.d = tuple(sides), n, len(sides)
        self.p = 1 << self.d
        self.E = int(np.prod(sides))
        self.h = [1.0 / s for s in sides]
        self.vol = float(np.prod(self.h))
        self.shape = tuple(s + 1 for s in sides)[::-1]
        self.N = int(np.prod(self.shape))
        g = [0.5 - 0.5 / math.sqrt(3.0), 0.5 + 0.5 / math.sqrt(3.0)]
        phi = torch.zeros((self.p, self.p), dtype=torch.float64)
        grad = torch.zeros((self.p, self.p, self.d), dtype=torch.float64)
        for q in range(self.p):
            x = [g[(q >> a) & 1] for a in range(self.d)]
            for a in range(self.p):
                f = [x[k] if (a >> k) & 1 else 1.0 - x[k] for k in range(self.d)]
                phi[q, a] = float(np.prod(f))
                for k in range(self.d):
                    grad[q, a, k] = (1.0 if (a >> k) & 1 else -1.0) / self.h[k] * float(np.prod(f[:k] + f[k + 1:]))
        self.phi, self.grad = phi.to(_dev()), grad.to(_dev())
        self.w = self.vol / self.p

    def corner(self, v, a):
        """The view of node array v (z, y, x, ...) at local node a of every element."""
        return v[tuple(slice((a >> (self.d - 1 - k)) & 1, ((a >> (self.d - 1 - k)) & 1) + self.sides[self.d - 1 - k])
                       for k in range(self.d))]

    def gather(self, u):
        u = u.reshape(self.shape + (self.n, -1))
        c = torch.stack([self.corner(u, a) for a in range(self.p)], dim=self.d)
        return c.reshape(self.E, self.p * self.n, -1)

    def scatter(self, ue):
        K = ue.shape[-1]
        ue = ue.reshape(self.sides[::-1] + (self.p, self.n, K))
        y = torch.zeros(self.shape + (self.n, K), dtype=torch.float64, device=ue.device)
        for a in range(self.p):
            self.corner(y, a).add_(ue.select(self.d, a))
        return y.reshape(self.N * self.n, K)

    def laplace(self):
        return self.w * torch.einsum("qai,qbi->ab", self.grad, self.grad)


class _Operator:
    """Sum of element operators with homogeneous constraints: terms are
    (coefficient per element, matrix) or (None, matrix per element)."""

    def __init__(self, el, terms, fixed):
        self.el, self.terms = el, terms
        self.free = (~fixed).to(torch.float64)[:, None]

    def full(self, u):
        ue = self.el.gather(u)
        y = None
        for c, M in self.terms:
            if c is None:
                t = torch.stack([(M * ue[:, None, :, k]).sum(-1) for k in range(ue.shape[-1])], dim=-1)
            else:
                t = c[:, None, None] * torch.matmul(M, ue)
            y = t if y is None else y + t
        return self.el.scatter(y)

    def __call__(self, u):
        return self.free * self.full(self.free * u)

    def diagonal(self):
        d = 0
        for c, M in self.terms:
            m = torch.diagonal(M, dim1=-2, dim2=-1)
            d = d + (m if c is None else c[:, None] * m)
        d = self.el.scatter(d[..., None])
        return torch.where(self.free > 0, d, torch.ones_like(d))


def _cg(A, b, rounds=6, inner=1e-5, most=6000):
    """A x = b (each column) by Jacobi-CG with residual replacement, as
    accurately as 64 bits hold it."""
    dinv = 1.0 / A.diagonal()
    x = torch.zeros_like(b)
    bn = torch.linalg.norm(b, dim=0).clamp_min(1e-300)
    last = math.inf
    for _ in range(rounds):
        r = b - A(x)
        worst = (torch.linalg.norm(r, dim=0) / bn).max().item()
        if worst < 3e-15 or worst > 0.5 * last:
            break
        last = worst
        e = torch.zeros_like(b)
        z = dinv * r
        p = z.clone()
        rz = (r * z).sum(0)
        stop = inner * inner * (r * r).sum(0)
        for k in range(most):
            q = A(p)
            al = rz / (p * q).sum(0).clamp_min(1e-300)
            e += al * p
            r -= al * q
            z = dinv * r
            rn = (r * z).sum(0)
            p = z + (rn / rz.clamp_min(1e-300)) * p
            rz = rn
            if k % 25 == 24 and bool(((r * r).sum(0) <= stop).all()):
                break
        x = x + e
    return x


def _bicgstab(A, b, rounds=8, inner=1e-4, most=3000):
    dinv = 1.0 / A.diagonal()
    x = torch.zeros_like(b)
    bn = torch.linalg.norm(b).item()
    last = math.inf
    for _ in range(rounds):
        r = b - A(x)
        worst = torch.linalg.norm(r).item() / bn
        if worst < 3e-15 or worst > 0.5 * last:
            break
        last = worst
        stop = inner * torch.linalg.norm(r)
        e = torch.zeros_like(b)
        rt, p, v = r.clone(), torch.zeros_like(b), torch.zeros_like(b)
        rho = al = om = torch.ones((), dtype=torch.float64, device=b.device)
        for k in range(most):
            rho1 = (rt * r).sum()
            p = r + (rho1 / rho) * (al / om) * (p - om * v)
            rho = rho1
            ph = dinv * p
            v = A(ph)
            al = rho / (rt * v).sum()
            s = r - al * v
            sh = dinv * s
            t = A(sh)
            om = (t * s).sum() / (t * t).sum()
            e += al * ph + om * sh
            r = s - om * t
            if k % 10 == 9 and bool(torch.linalg.norm(r) <= stop):
                break
        if not bool(torch.isfinite(e).all()):
            break
        x = x + e
    return x


def _fixed_plane(el, axis):
    m = torch.zeros(el.shape, dtype=torch.bool, device=_dev())
    m.select(el.d - 1 - axis, 0).fill_(True)
    return m.reshape(-1).repeat_interleave(el.n)


def _load(el, src):
    """Right-hand side of a source that is constant on each element (E, n)."""
    s = src.reshape(el.E, 1, el.n).expand(el.E, el.p, el.n) * (el.vol / el.p)
    return el.scatter(s.reshape(el.E, el.p * el.n, 1))


def exact(case, seed):
    kind = case["kind"]
    if kind == "poisson":
        sides = _sides(case)
        gen = _generator(seed)
        kap, src = _kappa(case, sides, gen), _source(sides, gen)
        el = _Elements(sides)
        A = _Operator(el, [(kap, el.laplace())], _fixed_plane(el, _constrained_axis(case)))
        return _cg(A, A.free * _load(el, src)).reshape(-1)
    if kind == "advection":
        sides, kap, vel, react, src = _advection_inputs(case, seed)
        el = _Elements(sides)
        M = kap[:, None, None] * el.laplace()
        M = M + el.w * torch.einsum("qa,eqi,qbi->eab", el.phi, vel, el.grad)
        M = M + el.w * torch.einsum("qa,eq,qb->eab", el.phi, react, el.phi)
        A = _Operator(el, [(None, M)], _fixed_plane(el, el.d - 1))
        return _bicgstab(A, A.free * _load(el, src)).reshape(-1)
    if kind == "elasticity":
        sides, lam, mu = _lame_inputs(case, seed)
        d = len(sides)
        el = _Elements(sides, d)
        G = el.grad
        same = torch.eye(d, dtype=torch.float64, device=_dev())
        kl = el.w * torch.einsum("qak,qbm->akbm", G, G)
        km = el.w * (torch.einsum("qaj,qbj,km->akbm", G, G, same) + torch.einsum("qam,qbk->akbm", G, G))
        m = el.p * d
        A = _Operator(el, [(lam, kl.reshape(m, m)), (mu, km.reshape(m, m))], _fixed_plane(el, d - 1))
        f = torch.tensor(_gravity(d), dtype=torch.float64, device=_dev()).expand(el.E, d)
        return _cg(A, A.free * _load(el, f)).reshape(-1, d)
    if kind == "system":
        return _exact_system(case, seed)
    if kind == "many_rhs":
        sides, kap, B = _loads(case, seed)
        el = _Elements(sides)
        return _cg(_Operator(el, [(kap, el.laplace())], _fixed_plane(el, 2)), B)
    if kind == "batch":
        gen = _generator(seed)
        out = []
        for sides in _batch_sides(case):
            kap, src = _kappa(dict(case, field="ln"), sides, gen), _source(sides, gen)
            el = _Elements(sides)
            A = _Operator(el, [(kap, el.laplace())], _fixed_plane(el, 0))
            out.append(_cg(A, A.free * _load(el, src)).reshape(-1))
        return out
    return _exact_train(case, seed)


def _exact_system(case, seed):
    sides, c, u = _system_inputs(case, seed)
    el = _Elements(sides, case["eq"])
    n, d = el.n, el.d
    full = {"A": (n, d, n, d), "B": (n, d, n), "C": (n, n, d), "D": (n, n), "X": (n, d), "Y": (n,)}
    c = {k: v.reshape((el.E, -1 if v.numel() == el.E * el.p * int(np.prod(full[k])) and case["expanded"] and k != "A" else 1)
                      + full[k]).expand((el.E, el.p) + full[k]) for k, v in c.items()}
    ue = el.gather(u).reshape(el.E, el.p, n)
    uq = torch.einsum("qb,ebm->eqm", el.phi, ue)
    gq = torch.einsum("qbl,ebm->eqml", el.grad, ue)
    flux = torch.einsum("eqkjml,eqml->eqkj", c["A"], gq) + torch.einsum("eqkjm,eqm->eqkj", c["B"], uq)
    val = torch.einsum("eqkml,eqml->eqk", c["C"], gq) + torch.einsum("eqkm,eqm->eqk", c["D"], uq)

    def test(fl, va):
        t = torch.einsum("qaj,eqkj->eak", el.grad, fl) + torch.einsum("qa,eqk->eak", el.phi, va)
        return el.scatter(el.w * t.reshape(el.E, el.p * n, 1)).reshape(-1)

    return [test(c["X"], c["Y"]), test(flux, val)]


def _exact_train(case, seed):
    """The 3-level U-Net (16, 32, 64 channels, 3x3x3) and its energy loss
    1 - (r.z)^2 / ((r.e)(z.A z)) by autograd on the CPU in 64 bits."""
    F = torch.nn.functional
    nodes, sides, kap, e, params = _train_inputs(case, seed)
    el = _Elements(sides)
    A = _Operator(el, [(kap, el.laplace())], _fixed_plane(el, 2))
    fixed = 1.0 - A.free

    def apply_a(v):
        return (A(v[:, None]) + fixed * v[:, None])[:, 0]

    r = apply_a(e)
    diag = A.diagonal()[:, 0]
    aref = sum(8.0 * el.vol / (9.0 * h * h) for h in el.h)
    un = r / diag
    s = 1.0 / torch.sqrt(torch.mean(un * un))
    n0, n1, n2 = nodes
    x = torch.zeros((1, 16) + tuple((n + 3) // 4 * 4 for n in (n2, n1, n0)), dtype=torch.float64)
    x[0, 0, :n2, :n1, :n0] = (s * un).reshape(n2, n1, n0).cpu()
    x[0, 1, :n2, :n1, :n0] = torch.log10(diag / aref).reshape(n2, n1, n0).cpu()
    p = torch.as_tensor(params, dtype=torch.float64).clone().requires_grad_(True)
    W, o = [], 0
    for cin, cout, _ in RL.LAYERS:
        w = p[o:o + 27 * cin * cout].reshape(cout, 3, 3, 3, cin).permute(0, 4, 1, 2, 3)
        o += 27 * cin * cout
        W.append((w, p[o:o + cout]))
        o += cout

    def conv(l, t):
        t = F.conv3d(t, W[l][0], W[l][1], padding=1)
        return torch.relu(t) if RL.LAYERS[l][2] else t

    s1 = conv(1, conv(0, x))
    s2 = conv(3, conv(2, F.avg_pool3d(s1, 2)))
    a3 = conv(5, conv(4, F.avg_pool3d(s2, 2)))
    a4 = conv(6, torch.cat([F.interpolate(a3, scale_factor=2, mode="nearest"), s2], dim=1))
    y = conv(8, conv(7, torch.cat([F.interpolate(a4, scale_factor=2, mode="nearest"), s1], dim=1)))
    z = y[0, 0, :n2, :n1, :n0].reshape(-1) / s.cpu()
    zd = z.detach().to(r.device)
    az = apply_a(zd)
    rz, zaz, re = torch.dot(r, zd), torch.dot(zd, az), torch.dot(r, e)
    dz = -2.0 * rz / (re * zaz) * r + 2.0 * rz * rz / (re * zaz * zaz) * az
    z.backward(dz.cpu())
    return [float(1.0 - rz * rz / (re * zaz)), p.grad]
