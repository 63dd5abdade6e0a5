"""The two-kernel CG iteration (sliced-ELL, stream and block stream SpMV)
against the three-kernel one (lanes-per-row SpMV) and a direct solve."""

import numpy as np
import pytest
import scipy.sparse as sps
import scipy.sparse.linalg as spla

from dolfinx_amd import la, problems, solvers
from dolfinx_amd._lib import DfxError
from dolfinx_amd.mesh import CellType

pytestmark = pytest.mark.gpu


def system(kind):
    if kind == "q1":      # sliced ELL, an odd number of rows
        p = problems.scalar_problem((12, 10, 8), CellType.hexahedron, kappa="exp_normal", c=0.3,
                                    f="normal", seed=2)
        return problems.assemble_system(p)
    if kind == "p3":      # stream kernel
        return problems.assemble_system(problems.p3_problem((5, 4, 3), seed=2))
    if kind == "p2":      # 3 x 3 blocks
        return problems.assemble_system(problems.elasticity_problem((5, 3, 4), seed=2))
    # 3 x 3 blocks in rows longer than the small chunk holds (342 blocks)
    n = 350
    rng = np.random.default_rng(1)
    D = rng.uniform(-1, 1, (3 * n, 3 * n)) / (6 * n)
    D = D + D.T + np.eye(3 * n)
    A = la.MatrixCSR(np.arange(n + 1) * n, np.tile(np.arange(n), n), bs=3)
    A.data = D.reshape(n, 3, n, 3).transpose(0, 2, 1, 3).ravel()
    return A, la.Vector.from_array(rng.standard_normal(3 * n))


@pytest.mark.parametrize("jacobi", [True, False])
@pytest.mark.parametrize("kind", ["q1", "p3", "p2", "long"])
def test_pairs(kind, jacobi):
    A, b = system(kind)
    n = A.shape[0]
    kw = dict(rtol=1e-11, max_it=20000, jacobi=jacobi, classic=True)
    x = la.Vector(n)
    r = solvers.cg(A, b, x, check_every=7, **kw)
    assert r.converged and r.true_rel_residual <= 2e-11
    ref = spla.spsolve(A.to_scipy().tocsc(), b.array)
    # |x - ref| <= cond |residual|; the systems' conditions are below 1e5
    assert np.linalg.norm(x.array - ref) <= 2e-6 * np.linalg.norm(ref)
    # the count and the iterates do not depend on how often the host looks
    for every, graph in ((1, False), (64, False), (5, True)):
        y = la.Vector(n)
        s = solvers.cg(A, b, y, check_every=every, graph=graph, **kw)
        assert s.iterations == r.iterations and np.array_equal(y.array, x.array)
    if kind != "long":
        A.set_lanes(4)
        y = la.Vector(n)
        s = solvers.cg(A, b, y, **kw)
        assert abs(s.iterations - r.iterations) <= max(2, r.iterations // 50)
        assert np.linalg.norm(x.array - y.array) <= 2e-6 * np.linalg.norm(ref)
        A.set_lanes(0)
    with pytest.raises(DfxError, match="exceeded max iterations"):
        solvers.cg(A, b, la.Vector(n), rtol=1e-30, max_it=3, jacobi=jacobi, classic=True)
    # from a nonzero guess, and from the solution of b = 0
    y = la.Vector.from_array(x.array)
    assert solvers.cg(A, b, y, rtol=1e-3, classic=True, jacobi=jacobi).true_rel_residual <= 1e-10
    z = la.Vector(n)
    assert solvers.cg(A, la.Vector(n), z, classic=True, jacobi=jacobi).iterations == 0


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_large_blocks(dtype):
    """3 x 3 blocks whose values pass the line of the two-kernel iteration in
    FP64 (175 MB) and not in FP32, against the residual on the host."""
    n, half = 30000, 40
    c = np.arange(n)[:, None] + np.arange(-half, half + 1)[None, :]
    on = (c >= 0) & (c < n)
    rp, cols = np.concatenate([[0], np.cumsum(on.sum(1))]), c[on].astype(np.int32)
    rng = np.random.default_rng(2)
    B = np.full((len(cols), 3, 3), -0.5 / (6 * half))
    B[cols == np.repeat(np.arange(n), np.diff(rp))] = np.diag([1.0, 2.0, 3.0])
    A = la.MatrixCSR(rp, cols, bs=3, dtype=dtype)
    A.data = B.ravel()
    b = rng.standard_normal(3 * n).astype(dtype)
    x = la.Vector(3 * n, dtype)
    rtol = 1e-10 if dtype == np.float64 else 1e-5
    r = solvers.cg(A, la.Vector.from_array(b), x, rtol=rtol)
    S = sps.bsr_matrix((B.astype(dtype).astype(np.float64), cols, rp), shape=(3 * n, 3 * n))
    res = b.astype(np.float64) - S @ x.array.astype(np.float64)
    # the recurrence's residual, and the rounding of 30 iterations on x
    assert r.converged and r.iterations < 30
    assert np.linalg.norm(res) <= (2 * rtol + 100 * np.finfo(dtype).eps) * np.linalg.norm(b)
