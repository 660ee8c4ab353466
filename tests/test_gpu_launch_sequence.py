"""The launch sequences of the Krylov methods (a check_interval selects them;
without one, systems this small are solved in one launch) to convergence
against the oracle, at small and odd sizes, with the bars of the solves' other
parity tests; and both routes on matrices that are indefinite or break the
recurrence down."""
import numpy as np
import pytest
import torch

import oracle as O
import ripley_hip as R
from gpu_helpers import grid, to_dev
from test_gpu_minres import _reaction
from test_gpu_parity import _advection_problem, _poisson_problem
from test_gpu_precond import _constrained, _options

pytestmark = pytest.mark.gpu

SIZES = [(2, (1, 9)), (2, (32, 32)), (2, (45, 44)), (3, (2, 1, 3)), (3, (11, 11, 11)), (3, (12, 10, 14))]


@pytest.mark.parametrize("interval", [0, 8])
@pytest.mark.parametrize("dim,ne", SIZES)
@pytest.mark.parametrize("method", ["PCG", "PCG_PLAIN"])
def test_pcg(interval, dim, ne, method):
    op, rhs, ptr, idx, oval, orhs = _poisson_problem(dim, ne)
    opts = R.SolverOptions()
    opts.setSymmetryOn()
    opts.setSolverMethod(getattr(R.SolverOptions, method))
    opts.setCheckInterval(interval)
    x = op.solve(rhs, opts).cpu().numpy()
    xo, dg, _, _ = O.solve(1, ptr, idx, oval.copy(), orhs, tolerance=1e-8, plain=(method == "PCG_PLAIN"))
    assert opts.hasConverged() and dg["converged"] == 1
    assert abs(opts.getDiagnostics("num_iter") - dg["num_iter"]) <= max(2, 0.02 * dg["num_iter"])
    assert np.linalg.norm(orhs - O.spmv(1, ptr, idx, oval, x)) <= 1e-7 * np.linalg.norm(orhs)
    assert np.linalg.norm(x - xo) <= 1e-6 * np.linalg.norm(xo)


@pytest.mark.parametrize("interval", [0, 8])
@pytest.mark.parametrize("method", ["PCG", "PCG_PLAIN", "MINRES"])
def test_true_residual(interval, method):
    op, rhs, ptr, idx, oval, orhs = _poisson_problem(3, (14, 12, 16), sigma=2.0)
    opts = _options("JACOBI", 1, getattr(R.SolverOptions, method))
    opts.setTolerance(1e-9)
    opts.setTrueResidualCriterion(True)
    opts.setCheckInterval(interval)
    x = op.solve(rhs, opts).cpu().numpy()
    assert opts.hasConverged()
    assert np.linalg.norm(orhs - O.spmv(1, ptr, idx, oval, x)) <= 1e-9 * 1.001 * np.linalg.norm(orhs)


@pytest.mark.parametrize("interval", [0, 8])
@pytest.mark.parametrize("dim,ne,sym", [(3, (12, 10, 9), False), (2, (30, 26), True), (2, (1, 9), False),
                                        (3, (11, 11, 11), True)])
def test_minres(interval, dim, ne, sym):
    op, rhs, ptr, idx, oval, orhs = _constrained(dim, ne, 1, sym, seed=12)
    opts = _options("JACOBI", 1, R.SolverOptions.MINRES)
    opts.setTolerance(1e-9)
    opts.setCheckInterval(interval)
    x = op.solve(rhs, opts).cpu().numpy()
    xo, dg, _, _ = O.solve(1, ptr, idx, oval.copy(), orhs, tolerance=1e-9, method="MINRES")
    assert opts.hasConverged() and dg["converged"] == 1
    assert abs(opts.getDiagnostics("num_iter") - dg["num_iter"]) <= max(3, 0.05 * dg["num_iter"])
    assert np.linalg.norm(orhs - O.spmv(1, ptr, idx, oval, x)) <= 1e-8 * np.linalg.norm(orhs)
    assert np.linalg.norm(x - xo) <= 1e-6 * np.linalg.norm(xo)


@pytest.mark.parametrize("interval", [0, 8])
@pytest.mark.parametrize("dim,ne", [(2, (24, 20)), (3, (10, 9, 8)), (2, (1, 9)), (2, (45, 44)), (3, (11, 11, 11))])
def test_bicgstab(interval, dim, ne):
    op, rhs, ptr, idx, oval, orhs = _advection_problem(dim, ne, 9)
    opts = R.SolverOptions()
    opts.setTolerance(1e-9)
    opts.setCheckInterval(interval)
    x = op.solve(rhs, opts).cpu().numpy()
    xo, dg, _, _ = O.solve(1, ptr, idx, oval.copy(), orhs, tolerance=1e-9, method="BICGSTAB")
    assert opts.hasConverged() and dg["converged"] == 1
    assert abs(opts.getDiagnostics("num_iter") - dg["num_iter"]) <= max(3, 0.05 * dg["num_iter"])
    assert np.linalg.norm(orhs - O.spmv(1, ptr, idx, oval, x)) <= 1e-8 * np.linalg.norm(orhs)
    assert np.linalg.norm(x - xo) <= 1e-6 * np.linalg.norm(xo)


@pytest.mark.parametrize("interval", [0, 8])
@pytest.mark.parametrize("method", ["PCG", "PCG_PLAIN", "MINRES", "BICGSTAB"])
def test_indefinite(interval, method):
    # a negative reaction term: indefinite, positive main diagonal
    op, rhs, ptr, idx, oval, orhs = _reaction(-60.0)
    M = O.csr_to_dense(1, ptr, idx, oval)
    ev = np.linalg.eigvalsh(M)
    assert ev.min() < 0 < ev.max()
    opts = _options("JACOBI", 1, getattr(R.SolverOptions, method))
    opts.setTolerance(1e-10)
    opts.setTrueResidualCriterion(True)
    opts.setCheckInterval(interval)
    x = op.solve(rhs, opts).cpu().numpy()
    assert opts.hasConverged()
    # ||x - xs|| <= ||A^-1|| ||r||
    xs = np.linalg.solve(M, orhs)
    assert np.linalg.norm(x - xs) <= 1.001e-10 * np.linalg.norm(orhs) / np.abs(ev).min()


def _pairs(ne):
    """Nodes coupled two by two along x: [[1, 1/2], [1/2, -1]].  With b = (1,
    -1) per pair the start residual is (-1/2, -1/2), so r.M^-1 r = 0 in exact
    arithmetic and in floating point."""
    dom, _ = grid(2, ne)
    n0 = ne[0] + 1
    assert n0 % 2 == 0
    op = dom.newOperator(1)
    nodes, em = [], []
    pair = np.array([[1.0, 0.5], [0.5, -1.0]])
    for y in range(ne[1]):
        for x in range(0, n0, 2):
            b = x + n0 * y
            nodes.append([b, b + 1, b + n0, b + n0 + 1])
            e = np.zeros((4, 4))
            e[:2, :2] = pair
            if y == ne[1] - 1:
                e[2:, 2:] = pair
            em.append(e)
    op.addElementBlocks(np.asarray(nodes, dtype=np.int32), np.asarray(em))
    return op, to_dev(np.tile([1.0, -1.0], op.size // 2))


@pytest.mark.parametrize("ne", [(7, 5), (7, 700)])
@pytest.mark.parametrize("method", ["PCG", "PCG_PLAIN", "MINRES"])
def test_breakdown_is_reported_alike(ne, method):
    # one workgroup and many; PCG and its textbook form divide by r.M^-1 r
    got = []
    for interval in (0, 8):
        op, b = _pairs(ne)
        o = R.SolverOptions()
        o.setSolverMethod(getattr(R.SolverOptions, method))
        o.setCheckInterval(interval)
        with pytest.raises(R.PasoException) as e:
            op.solve(b, o)
        got.append((e.value.args, o.getDiagnostics("num_iter")))
    assert got[0] == got[1]
    if method != "MINRES":
        assert "fatal break down" in str(got[0][0])
