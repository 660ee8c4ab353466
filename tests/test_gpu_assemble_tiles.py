"""The gather assembly at the edges of its tiles (64 / n^2 nodes per wave along
x, two node lines per block along y and z, four along y in 2-D) against the
oracle: coefficients per element (closed-form integrals, of the 2-point and the
one-point rule), on quadrature points (Gauss sum) and mixed, full and symmetric storage, written into zeroed values
and added to present ones.  Bar: |d a_ij| <= 1e-13 max_j |a_ij|, as for every
assembly."""
import numpy as np
import pytest

import oracle as O
import ripley_hip as R
from gpu_helpers import entrywise_ok, gpu_assemble, grid, to_dev

pytestmark = pytest.mark.gpu

SHAPES = [(1, 2, (63, 4)), (1, 2, (64, 3)), (2, 2, (15, 1)), (3, 2, (7, 6)), (4, 2, (3, 4)),
          (1, 3, (64, 1, 2)), (2, 3, (16, 2, 1)), (3, 3, (6, 1, 1)), (3, 3, (7, 2, 3)), (4, 3, (4, 2, 2))]


def _tensor(rng, n, dim, lead, name):
    pt = {"A": (n, dim, n, dim), "B": (n, dim, n), "C": (n, n, dim), "D": (n, n), "X": (n, dim), "Y": (n,)}[name]
    if n == 1:
        pt = tuple(d for d, k in zip(pt, {"A": (0, 1, 0, 1), "B": (0, 1, 0), "C": (0, 0, 1), "D": (0, 0),
                                          "X": (0, 1), "Y": (0,)}[name]) if k)
    return rng.standard_normal(lead + pt)


@pytest.mark.parametrize("n,dim,ne", SHAPES)
@pytest.mark.parametrize("expanded", [(), ("B", "C", "D", "X", "Y"), ("A", "B", "C", "D", "X", "Y")])
def test_tile_edges(n, dim, ne, expanded):
    rng = np.random.default_rng(100 * n + 10 * dim + ne[0] + len(expanded))
    length = tuple(0.7 + 0.3 * d for d in range(dim))
    dom, _ = grid(dim, ne, length)
    E, Q = dom.getNumElements(), 1 << dim
    c = {k: _tensor(rng, n, dim, (E, Q) if k in expanded else (E,), k) for k in "ABCDXY"}
    op, rhs = gpu_assemble(dom, n, **c)
    ptr, _, val = op.exportCSR()
    _, _, oval, orhs = O.assemble(dim, ne, length, n=n, expanded=expanded, **c)
    ok, worst = entrywise_ok(n, ptr, val, oval)
    assert ok, worst
    assert np.max(np.abs(rhs.cpu().numpy() - orhs)) <= 1e-13 * np.abs(orhs).max()


@pytest.mark.parametrize("n,dim,ne", SHAPES)
def test_one_point_rule(n, dim, ne):
    rng = np.random.default_rng(31 * n + dim + ne[0])
    length = tuple(0.7 + 0.3 * d for d in range(dim))
    dom, _ = grid(dim, ne, length)
    E = dom.getNumElements()
    c = {k: _tensor(rng, n, dim, (E,), k) for k in "ABCDXY"}
    op, rhs = gpu_assemble(dom, n, reduced=True, **c)
    ptr, _, val = op.exportCSR()
    _, _, oval, orhs = O.assemble(dim, ne, length, n=n, reduced=True, **c)
    ok, worst = entrywise_ok(n, ptr, val, oval)
    assert ok, worst
    assert np.max(np.abs(rhs.cpu().numpy() - orhs)) <= 1e-13 * np.abs(orhs).max()


@pytest.mark.parametrize("n,dim,ne", SHAPES)
@pytest.mark.parametrize("expanded", [(), ("D",)])
def test_symmetric_storage_and_second_assembly(n, dim, ne, expanded):
    rng = np.random.default_rng(7 * n + dim + ne[0])
    dom, length = grid(dim, ne)
    E, Q = dom.getNumElements(), 1 << dim
    A = rng.standard_normal((E, n * dim, n * dim))
    A = (A + A.transpose(0, 2, 1)).reshape((E, n, dim, n, dim) if n > 1 else (E, dim, dim))
    D = rng.standard_normal(((E, Q) if expanded else (E,)) + (n, n))
    D = D + np.swapaxes(D, -1, -2)
    D = D if n > 1 else D[..., 0, 0]
    op, _ = gpu_assemble(dom, n, symmetric=True, A=A, D=D)
    ptr, _, val = op.exportCSR()
    _, _, oval, _ = O.assemble(dim, ne, length, n=n, expanded=expanded, A=A, D=D)
    ok, worst = entrywise_ok(n, ptr, val, oval)
    assert ok, worst
    shape = {"A": (n, dim, n, dim) if n > 1 else (dim, dim), "D": (n, n) if n > 1 else ()}
    op.assemble({k: R.Coefficient(to_dev(v), shape[k], E, Q, dom.device) for k, v in (("A", A), ("D", D))}, None)
    ok, worst = entrywise_ok(n, ptr, op.exportCSR()[2], 2 * oval)
    assert ok, worst


# grids whose lines are short against a wave (whole lines per tile) and sides
# just over a multiple of the nodes per wave (the staged sums' own tile)
TILES = [(1, 2, (1, 40)), (1, 2, (20, 33)), (2, 2, (4, 30)), (3, 2, (1, 20)), (4, 2, (1, 9)),
         (1, 3, (3, 2, 9)), (1, 3, (3, 70, 1)), (1, 3, (30, 3, 5)), (1, 3, (65, 5, 3)), (2, 3, (2, 5, 6)),
         (2, 3, (16, 4, 5)), (3, 3, (2, 3, 4)), (3, 3, (7, 5, 4)), (4, 3, (1, 3, 4))]


@pytest.mark.parametrize("n,dim,ne", TILES)
@pytest.mark.parametrize("expanded", [(), ("B", "C", "D", "X", "Y"), ("A", "B", "C", "D", "X", "Y")])
def test_other_tiles(n, dim, ne, expanded):
    test_tile_edges(n, dim, ne, expanded)


# D alone on quadrature points: staged whole, one barrier
@pytest.mark.parametrize("n,dim,ne", SHAPES + TILES)
def test_mass_matrix_on_points(n, dim, ne):
    rng = np.random.default_rng(17 * n + dim + ne[0])
    length = tuple(0.7 + 0.3 * d for d in range(dim))
    dom, _ = grid(dim, ne, length)
    D = _tensor(rng, n, dim, (dom.getNumElements(), 1 << dim), "D")
    op, _ = gpu_assemble(dom, n, D=D)
    ptr, _, val = op.exportCSR()
    _, _, oval, _ = O.assemble(dim, ne, length, n=n, expanded=("D",), D=D)
    ok, worst = entrywise_ok(n, ptr, val, oval)
    assert ok, worst


@pytest.mark.parametrize("n,dim,ne", TILES)
def test_other_tiles_symmetric_and_one_point(n, dim, ne):
    test_symmetric_storage_and_second_assembly(n, dim, ne, ("D",))
    test_one_point_rule(n, dim, ne)
