"""Which kernels a solve takes (rg_matrix_solve_route, rg_batch_solve_route) on
both sides of each limit, and the way back from a one-launch solve whose
workgroups stop waiting for one another (a poll limit of one, set by the
host): every kernel ends, and the launch sequence gives the bits it gives when
it is asked for."""
import ctypes
import threading

import numpy as np
import pytest
import torch

import oracle as O
import ripley_hip as R
from gpu_helpers import to_dev
from ripley_hip import _lib, core
from ripley_hip import batch as RB
from test_gpu_march import _system as elastic_system
from test_gpu_resident import SIZES, _batch, _problem, _solve

pytestmark = pytest.mark.gpu

LAUNCHES, ONE_LAUNCH, ABANDONED, MARCH, UNIT_INVERSE = 1, 2, 4, 8, 16


def route(handle, batch=False):
    r = ctypes.c_int(-1)
    f = _lib.load().rg_batch_solve_route if batch else _lib.load().rg_matrix_solve_route
    assert f(handle, ctypes.byref(r)) == 0
    return r.value


class poll_limit:
    """The context's poll limit within a block (0: the default)."""

    def __init__(self, ctx, polls):
        self.ctx, self.polls = ctx, polls

    def __enter__(self):
        assert _lib.load().rg_context_set_poll_limit(self.ctx.handle, self.polls) == 0

    def __exit__(self, *a):
        assert _lib.load().rg_context_set_poll_limit(self.ctx.handle, 0) == 0


def options(method, interval=0, tol=1e-8, true_res=False):
    o = R.SolverOptions()
    o.setSolverMethod(getattr(R.SolverOptions, method))
    o.setTolerance(tol)
    o.setCheckInterval(interval)
    o.setTrueResidualCriterion(true_res)
    return o


@pytest.mark.parametrize("dim,ne", SIZES)
@pytest.mark.parametrize("method", ["PCG", "PCG_PLAIN", "MINRES", "BICGSTAB"])
def test_small_systems_take_one_launch(dim, ne, method):
    op, ptr, idx, val, b = _problem(dim, ne, False)
    assert route(op.handle) == 0
    x, o = _solve(op, b, method, true_res=True)
    assert o.hasConverged() and route(op.handle) == ONE_LAUNCH
    r = b - O.spmv(1, ptr, idx, val, x)
    assert np.linalg.norm(r) <= 1e-8 * (1 + 1e-6) * np.linalg.norm(b)
    op, _, _, _, b = _problem(dim, ne, False)
    op.solve(to_dev(b), options(method, 8))
    assert route(op.handle) == LAUNCHES


def _cube(dim, ne):
    dom = R.Rectangle(*ne) if dim == 2 else R.Brick(*ne)
    E, Q = dom.getNumElements(), 1 << dim
    op = dom.newOperator(1, symmetric=True)
    rhs = torch.zeros(op.size, dtype=torch.float64, device="cuda")
    op.assemble({"A": R.Coefficient(1.0, (dim, dim), E, Q, dom.device, isotropic=True),
                 "Y": R.Coefficient(1.0, (), E, Q, dom.device)}, rhs)
    q = dom.whereZero(dim - 1)
    op.nullifyRowsAndCols(q, q, 1.0)
    return op, torch.where(q > 0, torch.zeros_like(rhs), rhs)


# the sizes of test_capacity_edges
@pytest.mark.parametrize("method,dim,n,fits", [("PCG", 3, 70, True), ("PCG", 3, 76, False), ("PCG_PLAIN", 3, 70, True),
                                               ("MINRES", 3, 62, True), ("MINRES", 3, 66, False),
                                               ("BICGSTAB", 3, 62, True), ("BICGSTAB", 3, 66, False),
                                               ("PCG", 2, 700, True), ("PCG", 2, 740, False)])
def test_capacity(method, dim, n, fits):
    op, b = _cube(dim, (n,) * dim if dim == 2 else (n, n - 1, n - 3))
    op.solve(b, options(method))
    assert bool(route(op.handle) & ONE_LAUNCH) == fits and bool(route(op.handle) & LAUNCHES) != fits


def test_other_preconditioners_and_methods_launch():
    op, _, _, _, b = _problem(3, (10, 9, 11), True)
    o = options("PCG")
    o.setNumSweeps(2)
    op.solve(to_dev(b), o)
    assert route(op.handle) == LAUNCHES
    op.solve(to_dev(b), options("PCG_MIXED"))
    assert route(op.handle) == LAUNCHES


# grids of several workgroups
MANY = [(2, (97, 61)), (3, (11, 11, 11)), (3, (30, 23, 17))]


@pytest.mark.parametrize("dim,ne", MANY)
@pytest.mark.parametrize("method", ["PCG", "PCG_PLAIN", "MINRES", "BICGSTAB"])
def test_an_abandoned_launch_leaves_the_solve_to_the_sequence(dim, ne, method):
    op, _, _, _, b = _problem(dim, ne, True)
    want = op.solve(to_dev(b), options(method, 32))
    fresh, _, _, _, _ = _problem(dim, ne, True)
    with poll_limit(fresh.ctx, 1):
        o = options(method)
        got = fresh.solve(to_dev(b), o)
        assert o.hasConverged() and route(fresh.handle) == ABANDONED | LAUNCHES
        assert torch.equal(got, want)
    # one more try at the next solve; kept if it goes through
    assert torch.allclose(fresh.solve(to_dev(b), options(method)), want, rtol=0, atol=1e-6 * want.abs().max().item())
    assert route(fresh.handle) == ONE_LAUNCH
    # two in a row: the matrix stays with the sequence
    with poll_limit(fresh.ctx, 1):
        for expected in (ABANDONED | LAUNCHES, ABANDONED | LAUNCHES, LAUNCHES):
            assert torch.equal(fresh.solve(to_dev(b), options(method)), want)
            assert route(fresh.handle) == expected
    fresh.solve(to_dev(b), options(method))
    assert route(fresh.handle) == LAUNCHES


@pytest.mark.parametrize("shapes", [[(97, 61), (200, 131), (30, 30)], [(20, 21, 19), (11, 11, 11)]])
@pytest.mark.parametrize("method", ["PCG_PLAIN", "PCG_MIXED"])
def test_an_abandoned_batch_launch(shapes, method):
    ops, _, rhs = _batch(shapes, len(shapes))
    solver = RB.BatchSolver(ops)
    solver.set_tile(2)
    b = solver.join(rhs)
    one, _ = solver.solve(b, options(method))
    assert route(solver.handle, True) == ONE_LAUNCH
    want, _ = solver.solve(b, options(method, 32))
    assert route(solver.handle, True) == LAUNCHES
    with poll_limit(solver.ctx, 1):
        got, diags = solver.solve(b, options(method))
        assert route(solver.handle, True) == ABANDONED | LAUNCHES and all(d["converged"] for d in diags)
        assert torch.equal(got, want)
    again, _ = solver.solve(b, options(method))
    assert route(solver.handle, True) == ONE_LAUNCH and torch.equal(again, one)


# the shapes of test_gpu_march, and ones whose tiles do not fill the chip or
# whose storage is full
@pytest.mark.parametrize("ne,method,sym,march", [((66, 65, 64), "PCG", True, True), ((150, 60, 31), "PCG_PLAIN", True, True),
                                                 ((47, 170, 36), "PCG", True, True), ((84, 83, 82), "PCG_MIXED", True, True),
                                                 ((66, 65, 64), "PCG_MIXED", True, False), ((64, 63, 66), "PCG", True, False),
                                                 ((8, 8, 3600), "PCG", True, False), ((66, 65, 64), "PCG", False, False)])
def test_marching_product(ne, method, sym, march):
    op, b = elastic_system(ne, sym, 1)
    o = options(method)
    o.setIterMax(3)
    o.setAcceptanceConvergenceFailureOn()
    op.solve(b, o)
    assert bool(route(op.handle) & MARCH) == march


@pytest.mark.parametrize("ne,unit", [((64, 65, 63), True), ((30, 23, 17), False)])
@pytest.mark.parametrize("method", ["PCG", "PCG_PLAIN"])
def test_unit_inverse(ne, unit, method):
    op, b = _cube(3, ne)
    op.solve(b, options(method, 32))
    assert bool(route(op.handle) & UNIT_INVERSE) == unit


def test_inverse_that_is_not_one_is_read():
    # an off-diagonal entry above its row's diagonal one
    n = 600
    dom = R.Rectangle(n, n)
    ix = np.arange(n * n)
    n0 = (ix % n) + (n + 1) * (ix // n)
    s = np.exp(np.random.default_rng(3).standard_normal((n * n, 4)))
    op = dom.newOperator(1)
    op.addElementBlocks(np.stack([n0, n0 + 1, n0 + n + 1, n0 + n + 2], axis=1).astype(np.int32),
                        s[:, :, None] * (np.eye(4) + 0.8)[None] * s[:, None, :])
    o = options("PCG", 32)
    o.setIterMax(3)
    o.setAcceptanceConvergenceFailureOn()
    op.solve(torch.ones(op.size, dtype=torch.float64, device="cuda"), o)
    assert route(op.handle) == LAUNCHES


def test_threads_with_their_own_contexts(monkeypatch):
    # cooperative launches of several streams take turns on the GPU: each
    # solve goes through in one launch, with the bits it has alone
    jobs = []
    for dim, ne in MANY:
        ctx = core.Context(0)
        monkeypatch.setattr(core, "get_context", lambda device=0, ctx=ctx: ctx)
        op, _, _, _, b = _problem(dim, ne, True)
        jobs.append((op, to_dev(b), torch.cuda.Stream()))
    monkeypatch.undo()
    alone = [op.solve(b, options("PCG")) for op, b, _ in jobs]
    torch.cuda.synchronize()
    got = [[] for _ in jobs]

    def work(k):
        op, b, s = jobs[k]
        with torch.cuda.stream(s):
            for _ in range(8):
                got[k].append((op.solve(b, options("PCG")), route(op.handle)))
            s.synchronize()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for x, runs in zip(alone, got):
        assert len(runs) == 8 and all(r == ONE_LAUNCH and torch.equal(y, x) for y, r in runs)
