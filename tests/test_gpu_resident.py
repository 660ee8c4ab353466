"""The one-launch Krylov solves (systems that fit in the chip's registers) at
the edges of their tiling, against the oracle's PASO restatement: one tile, a
few tiles, tiles cut by the grid's end, thin grids, the largest grids that
still fit and the first that does not; full and symmetric storage.  Bars: the
oracle's iteration count within 2 % (at least 2), its solution within 1e-6, as
for every solve; the FP64 residual is checked beside them."""
import numpy as np
import pytest
import torch

import oracle as O
import ripley_hip as R
from gpu_helpers import dirichlet_mask, gpu_assemble, grid, to_dev

pytestmark = pytest.mark.gpu

# nodes: 24 and 60 (far fewer than threads), 1-tile sizes, several tiles, and
# sides that no tile side divides
SIZES = [(2, (5, 3)), (2, (1, 700)), (2, (44, 43)), (2, (45, 45)), (2, (97, 61)), (2, (200, 131)),
         (3, (2, 1, 3)), (3, (10, 9, 11)), (3, (11, 11, 11)), (3, (3, 2, 250)), (3, (30, 23, 17))]


def _problem(dim, ne, sym, bs=1):
    rng = np.random.default_rng(sum(ne) + 100 * dim)
    dom, length = grid(dim, ne)
    E = dom.getNumElements()
    A = np.exp(0.7 * rng.standard_normal(E))[:, None, None] * np.eye(dim)[None]
    Y = rng.uniform(0.5, 1.5, E)
    op, rhs = gpu_assemble(dom, 1, symmetric=sym, A=A, Y=Y)
    q = dirichlet_mask(dom, dim - 1)
    op.nullifyRowsAndCols(to_dev(q), to_dev(q), 1.0)
    ptr, idx, val, orhs = O.assemble(dim, ne, length, A=A, Y=Y)
    O.nullify(1, ptr, idx, val, q, q, 1.0)
    b = np.where(q > 0, 0.0, orhs)
    return op, ptr, idx, val, b


def _solve(op, b, method, tol=1e-8, true_res=False):
    o = R.SolverOptions()
    o.setSolverMethod(getattr(R.SolverOptions, method))
    o.setTolerance(tol)
    o.setTrueResidualCriterion(true_res)
    return op.solve(to_dev(b), o).cpu().numpy(), o


@pytest.mark.parametrize("dim,ne", SIZES)
@pytest.mark.parametrize("sym", [False, True])
@pytest.mark.parametrize("method", ["PCG", "PCG_PLAIN", "MINRES"])
def test_symmetric_methods_match_the_oracle(dim, ne, sym, method):
    op, ptr, idx, val, b = _problem(dim, ne, sym)
    x, o = _solve(op, b, method)
    xo, dg, _, _ = O.solve(1, ptr, idx, val.copy(), b, tolerance=1e-8)
    assert o.hasConverged()
    assert np.linalg.norm(x - xo) <= 1e-6 * np.linalg.norm(xo)
    r = b - O.spmv(1, ptr, idx, val, x)
    assert np.linalg.norm(r) <= 1e-6 * np.linalg.norm(b)
    if method == "PCG":
        n = o.getDiagnostics("num_iter")
        assert abs(n - dg["num_iter"]) <= max(2, 0.02 * dg["num_iter"])


@pytest.mark.parametrize("dim,ne", SIZES)
def test_bicgstab_solves(dim, ne):
    rng = np.random.default_rng(11 + sum(ne))
    dom, length = grid(dim, ne)
    E = dom.getNumElements()
    c = {"A": np.exp(0.5 * rng.standard_normal(E))[:, None, None] * np.eye(dim)[None],
         "C": 2.0 * rng.standard_normal((E, dim)), "D": rng.uniform(1.0, 2.0, E), "Y": rng.standard_normal(E)}
    op, rhs = gpu_assemble(dom, 1, **c)
    q = dirichlet_mask(dom, dim - 1)
    op.nullifyRowsAndCols(to_dev(q), to_dev(q), 1.0)
    ptr, idx, val, orhs = O.assemble(dim, ne, length, **c)
    O.nullify(1, ptr, idx, val, q, q, 1.0)
    b = np.where(q > 0, 0.0, orhs)
    x, o = _solve(op, b, "BICGSTAB", tol=1e-10, true_res=True)
    assert o.hasConverged()
    r = b - O.spmv(1, ptr, idx, val, x)
    assert np.linalg.norm(r) <= 2e-10 * np.linalg.norm(b)


# the largest cube / square of each method's capacity (256 tiles of 512 x rows
# per thread nodes) and the first beyond: the same solution to the tolerance
@pytest.mark.parametrize("method,dim,n", [("PCG", 3, 70), ("PCG", 3, 76), ("PCG_PLAIN", 3, 70), ("MINRES", 3, 62),
                                          ("MINRES", 3, 66), ("BICGSTAB", 3, 62), ("BICGSTAB", 3, 66),
                                          ("PCG", 2, 700), ("PCG", 2, 740)])
def test_capacity_edges(method, dim, n):
    ne = (n,) * dim if dim == 2 else (n, n - 1, n - 3)
    dom, _ = grid(dim, ne)
    E, Q = dom.getNumElements(), 1 << dim
    g = torch.Generator(device="cuda").manual_seed(n)
    kap = torch.exp(torch.randn(E, dtype=torch.float64, device="cuda", generator=g) * 0.5)

    def system():
        op = dom.newOperator(1, symmetric=method != "BICGSTAB")
        rhs = torch.zeros(op.size, dtype=torch.float64, device="cuda")
        op.assemble({"A": R.Coefficient(kap, (dim, dim), E, Q, dom.device, isotropic=True),
                     "Y": R.Coefficient(1.0, (), E, Q, dom.device)}, rhs)
        q = dom.whereZero(dim - 1)
        op.nullifyRowsAndCols(q, q, 1.0)
        return op, torch.where(q > 0, torch.zeros_like(rhs), rhs)

    op, b = system()
    o = R.SolverOptions()
    o.setSolverMethod(getattr(R.SolverOptions, method))
    o.setTrueResidualCriterion(True)
    x = op.solve(b, o)
    op2, r = system()
    op2.MatrixVector(-1.0, x, 1.0, r)
    assert o.hasConverged()
    assert (torch.linalg.norm(r) / torch.linalg.norm(b)).item() <= 1e-8


def test_repeats_are_bit_identical_and_streams_do_not_matter():
    op, ptr, idx, val, b = _problem(3, (30, 23, 17), True)
    x1, _ = _solve(op, b, "PCG")
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        x2, _ = _solve(op, b, "PCG")
    assert np.array_equal(x1, x2)


@pytest.mark.parametrize("dim,ne", [(2, (44, 43)), (2, (97, 61)), (3, (10, 9, 11)), (3, (30, 23, 17))])
@pytest.mark.parametrize("method", ["PCG", "PCG_PLAIN", "MINRES", "BICGSTAB"])
def test_iteration_limits_match_the_launch_sequence(dim, ne, method):
    # a check_interval selects the launch sequence; after k iterations both
    # hold the same iterate but for the rounding of their sums
    for k in (1, 2, 3, 4, 9, 17):
        got = []
        for interval in (0, 4):
            op, _, _, _, b = _problem(dim, ne, True)
            o = R.SolverOptions()
            o.setSolverMethod(getattr(R.SolverOptions, method))
            o.setTolerance(1e-12)
            o.setIterMax(k)
            o.setAcceptanceConvergenceFailureOn()
            o.setCheckInterval(interval)
            got.append((op.solve(to_dev(b), o).cpu().numpy(), o.getDiagnostics("num_iter"), o.hasConverged()))
        assert got[0][1:] == got[1][1:]
        assert np.linalg.norm(got[0][0] - got[1][0]) <= 1e-11 * np.linalg.norm(got[1][0])


@pytest.mark.parametrize("method", ["PCG", "PCG_PLAIN", "MINRES", "BICGSTAB"])
def test_special_right_hand_sides(method):
    # zero, one that a multiple of the start vector solves at once, and the
    # iterates of a system whose solution is reached in one step
    dom, _ = grid(3, (6, 5, 7))
    op, _ = gpu_assemble(dom, 1, symmetric=True, D=np.ones(dom.getNumElements()))
    q = np.ones(op.size)
    op.nullifyRowsAndCols(to_dev(q), to_dev(q), 2.0)     # the matrix is 2 I
    b = np.random.default_rng(1).standard_normal(op.size)
    o = R.SolverOptions()
    o.setSolverMethod(getattr(R.SolverOptions, method))
    assert np.array_equal(op.solve(to_dev(0 * b), o).cpu().numpy(), 0 * b)
    x = op.solve(to_dev(b), o).cpu().numpy()
    assert o.hasConverged() and np.allclose(x, 0.5 * b, rtol=1e-14, atol=0)


def _batch(shapes, seed, spread=0.7):
    rng = np.random.default_rng(seed)
    ops, vals, rhs = [], [], []
    for ne in shapes:
        dim = len(ne)
        dom, length = grid(dim, ne)
        E = dom.getNumElements()
        A = np.exp(spread * rng.standard_normal(E))[:, None, None] * np.eye(dim)[None]
        op, b = gpu_assemble(dom, 1, A=A, Y=rng.uniform(0.5, 1.5, E))
        q = to_dev(dirichlet_mask(dom, 0))
        op.nullifyRowsAndCols(q, q, 1.0)
        ops.append(op)
        rhs.append(torch.where(q > 0, torch.zeros_like(b), b))
        vals.append(op.exportCSR())
    return ops, vals, rhs


# one tile each, many tiles, more tiles than the chip holds at once, one
# system larger than all others, and the smallest grids
BATCHES = [[(5, 3)], [(54, 54), (55, 55), (56, 54)], [(300, 290), (40, 700), (3, 3), (120, 64)],
           [(260, 250)] * 6 + [(64, 64)] * 9, [(10, 11, 9)] * 3, [(40, 33, 37), (5, 4, 3), (1, 1, 900), (24, 24, 24)]]


@pytest.mark.parametrize("shapes", BATCHES, ids=lambda s: "%d systems" % len(s))
@pytest.mark.parametrize("method", ["PCG_PLAIN", "PCG_MIXED"])
def test_batches_match_the_launch_sequence(shapes, method):
    from ripley_hip import batch as RB
    ops, vals, rhs = _batch(shapes, len(shapes))
    solver = RB.BatchSolver(ops)
    b = solver.join(rhs)
    got = []
    for interval in (0, 8):
        o = R.SolverOptions()
        o.setSolverMethod(getattr(R.SolverOptions, method))
        o.setTolerance(1e-9)
        o.setCheckInterval(interval)
        x, diags = solver.solve(b, o)
        assert all(d["converged"] for d in diags)
        got.append(solver.split(x))
    for (ptr, idx, val), x, y, f in zip(vals, got[0], got[1], rhs):
        f = f.cpu().numpy()
        r = f - O.spmv(1, ptr, idx, val, x.cpu().numpy())
        assert np.linalg.norm(r) <= 1e-9 * (1 + 1e-6) * np.linalg.norm(f)
        assert torch.linalg.norm(x - y) <= 1e-6 * torch.linalg.norm(y)


def test_batch_limits_zero_sides_and_reuse():
    from ripley_hip import batch as RB
    ops, vals, rhs = _batch([(30, 30), (200, 90), (9, 9)], 5)
    solver = RB.BatchSolver(ops)
    o = R.SolverOptions()
    o.setSolverMethod(R.SolverOptions.PCG_PLAIN)
    o.setAcceptanceConvergenceFailureOn()
    o.setIterMax(7)
    rhs[2] = torch.zeros_like(rhs[2])
    b = solver.join(rhs)
    x7, diags = solver.solve(b, o)
    assert [d["num_iter"] for d in diags] == [7, 7, 0]
    assert [d["converged"] for d in diags] == [False, False, True]
    o.setCheckInterval(7)
    y7, _ = solver.solve(b, o)
    assert torch.linalg.norm(x7 - y7) <= 1e-11 * torch.linalg.norm(y7)
    o.setCheckInterval(0)
    o.setIterMax(100000)
    x, diags = solver.solve(b, o)
    again, _ = solver.solve(b, o)
    assert all(d["converged"] for d in diags) and torch.equal(x, again)
    assert torch.count_nonzero(solver.split(x)[2]) == 0


# iterations whose streams exceed the L2s: the PCGs' update kernels leave the
# Jacobi inverse unread where it is 1 to rounding (diffusion after PASO's
# balance) and read it where it is not (element matrices whose off-diagonal
# entries exceed a diagonal one); the one-launch solve always reads it
@pytest.mark.parametrize("unit", [True, False])
@pytest.mark.parametrize("method", ["PCG", "PCG_PLAIN"])
def test_unread_jacobi_inverse(unit, method):
    rng = np.random.default_rng(3)
    got = []
    if unit:
        dom, _ = grid(3, (64, 65, 63))
        A = np.exp(0.7 * rng.standard_normal(dom.getNumElements()))[:, None, None] * np.eye(3)[None]
        make = lambda: gpu_assemble(dom, 1, symmetric=True, A=A)[0]
    else:
        n = 600
        dom, _ = grid(2, (n, n))
        ix = np.arange(n * n)
        n0 = (ix % n) + (n + 1) * (ix // n)
        nodes = np.stack([n0, n0 + 1, n0 + n + 1, n0 + n + 2], axis=1).astype(np.int32)
        s = np.exp(1.0 * rng.standard_normal((n * n, 4)))
        em = s[:, :, None] * (np.eye(4) + 0.8)[None] * s[:, None, :]

        def make():
            op = dom.newOperator(1)
            op.addElementBlocks(nodes, em)
            return op
    b = rng.standard_normal(dom.getNumNodes())
    for interval in (0, 32):
        op = make()
        if unit:
            q = to_dev(dirichlet_mask(dom, 2))
            op.nullifyRowsAndCols(q, q, 1.0)
        o = R.SolverOptions()
        o.setSolverMethod(getattr(R.SolverOptions, method))
        o.setTolerance(1e-9)
        o.setCheckInterval(interval)
        got.append((op.solve(to_dev(b), o), o.getDiagnostics("num_iter")))
        assert o.hasConverged()
    assert abs(got[0][1] - got[1][1]) <= max(2, 0.02 * got[1][1])
    assert torch.linalg.norm(got[0][0] - got[1][0]) <= 1e-7 * torch.linalg.norm(got[1][0])
