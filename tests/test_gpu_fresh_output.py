"""The colour substitutions write every row of their output before anything
reads it: what the output buffer held before (here NaN) does not reach the
result."""
import numpy as np
import pytest
import torch

import ripley_hip as R
from gpu_helpers import dirichlet_mask, gpu_assemble, grid, to_dev
from ripley_hip import _lib
from ripley_hip.core import _ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["GAUSS_SEIDEL", "ILU0"])
@pytest.mark.parametrize("dim,ne,n", [(2, (30, 26), 1), (3, (12, 10, 9), 1), (3, (5, 5, 4), 3)])
def test_output_buffer_contents_do_not_matter(prec, dim, ne, n):
    import ctypes
    rng = np.random.default_rng(5)
    dom, _ = grid(dim, ne)
    E = dom.getNumElements()
    A = rng.uniform(1, 2, (E, n * dim))[:, :, None] * np.eye(n * dim)[None]
    op, _ = gpu_assemble(dom, n, A=A.reshape((E, n, dim, n, dim) if n > 1 else (E, dim, dim)),
                         D=np.broadcast_to(np.eye(n) + 0.1, (E, n, n)).copy() if n > 1 else np.ones(E))
    q = to_dev(dirichlet_mask(dom, dim - 1, n))
    op.nullifyRowsAndCols(q, q, 1.0)
    b = to_dev(rng.standard_normal(op.size))
    o = R.SolverOptions()
    o.setPreconditioner(getattr(R.SolverOptions, prec))
    opt = o._rg_options()
    out = []
    for fill in (0.0, float("nan")):
        x = torch.full((op.size,), fill, dtype=torch.float64, device="cuda")
        op._bind()
        assert _lib.load().rg_matrix_solve_preconditioner(op.handle, ctypes.byref(opt), _ptr(x), _ptr(b)) == 0
        out.append(x)
    assert bool(torch.isfinite(out[0]).all()) and torch.equal(out[0], out[1])
