"""The cooperative CG with its rows in LDS and, for rows that do not fit
there, read from memory: against a direct solve and the classic path."""

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from dolfinx_amd import la, solvers

pytestmark = pytest.mark.gpu


def ragged(n, longest, dtype):
    """Symmetric, strictly diagonally dominant (condition below 3): rows of 1
    to about `longest` entries in a band, every 37th row its diagonal alone."""
    rng = np.random.default_rng(n + longest)
    half = (longest - 1) // 2
    i = np.arange(n)
    rows, cols, vals = [i], [i], [np.ones(n)]
    for d in range(1, half + 1):
        a = i[:n - d]
        a = a[(a % 37 != 5) & ((a + d) % 37 != 5)]
        w = rng.uniform(-1, 1, a.size) / (4 * half)
        rows += [a, a + d]
        cols += [a + d, a]
        vals += [w, w]
    S = sp.csr_matrix((np.concatenate(vals), (np.concatenate(rows), np.concatenate(cols))),
                      shape=(n, n))
    if longest % 2 == 0:  # one row of exactly `longest` entries
        length = np.diff(S.indptr)
        p = int(np.argmax(length[:n - longest]))
        more = [q for q in range(p + half + 1, n) if q % 37 != 5][:longest - length[p]]
        E = sp.csr_matrix((np.full(len(more), 0.1 / longest), ([p] * len(more), more)), (n, n))
        S = (S + E + E.T).tocsr()
        assert np.diff(S.indptr).max() == longest
    S.sort_indices()
    A = la.MatrixCSR(S.indptr.astype(np.int64), S.indices.astype(np.int32), dtype=dtype)
    A.data = S.data.astype(dtype)
    return A, S.astype(dtype).astype(np.float64)


# rows per workgroup: one per thread up to 16,384 rows, then two; beside the
# kernel's own arrays an LDS of 160 KiB holds 63 (FP64) or 106 (FP32) entries
# per thread: 64 (and 32 with two rows) would fill it to the last byte
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,longest", [(1, 1), (255, 15), (257, 17), (700, 33), (511, 63),
                                       (511, 64), (600, 65), (600, 105), (600, 106), (600, 107), (16384, 15),
                                       (16385, 31), (16385, 32), (20000, 35),
                                       (65536, 17)])
def test_coop_rows(n, longest, dtype):
    A, S = ragged(n, longest, dtype)
    b = np.random.default_rng(3).standard_normal(n).astype(dtype)
    ref = spla.spsolve(S.tocsc(), b.astype(np.float64))
    rtol = 1e-12 if dtype == np.float64 else 1e-6
    out = []
    for classic in (False, True):
        x = la.Vector(n, dtype=dtype)
        r = solvers.cg(A, la.Vector.from_array(b), x, rtol=rtol, max_it=500, classic=classic)
        assert r.cooperative == (0 if classic else 1)
        # |x - ref| <= |A^-1| |residual| <= 2 rtol |b|, plus the rounding of the
        # recurrence (30 iterations at most of a well-conditioned system)
        eps = np.finfo(dtype).eps
        err = np.linalg.norm(x.array.astype(np.float64) - ref)
        assert err <= (2 * rtol + 200 * eps) * np.linalg.norm(b)
        out.append(r.iterations)
    assert abs(out[0] - out[1]) <= 1
