"""SpMV kernels at the edges of their chunks, pairs, row groups and column
encodings, against scipy in FP64."""

import numpy as np
import pytest
import scipy.sparse as sps

from dolfinx_amd import la, solvers

pytestmark = pytest.mark.gpu


def banded(nrows, ncols, offsets, keep, seed):
    """Pattern with the columns r + offset of each row r that exist, each kept
    with probability keep; random values."""
    rng = np.random.default_rng(seed)
    c = np.arange(nrows)[:, None] + np.asarray(offsets)[None, :]
    on = (c >= 0) & (c < ncols) & (rng.random(c.shape) < keep)
    rp = np.concatenate([[0], np.cumsum(on.sum(1))])
    return rp, c[on].astype(np.int32), rng.standard_normal(int(rp[-1]))


def check(rp, cols, vals, ncols, dtype, seed=1):
    A = la.MatrixCSR(rp, cols, ncols=ncols, dtype=dtype)
    A.data = vals
    rng = np.random.default_rng(seed)
    n = len(rp) - 1
    x, y0 = rng.standard_normal(ncols).astype(dtype), rng.standard_normal(n).astype(dtype)
    y = la.Vector.from_array(y0)
    A.mult(la.Vector.from_array(x), y)
    S = sps.csr_matrix((vals.astype(dtype).astype(np.float64), cols, rp), shape=(n, ncols))
    ref = y0.astype(np.float64) + S @ x.astype(np.float64)
    # one rounding per product and per addition, whatever their order
    size = abs(S) @ abs(x.astype(np.float64)) + abs(y0)
    bound = (np.diff(rp) + 3) * np.finfo(dtype).eps * size
    assert (np.abs(y.array - ref) <= bound).all()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("offsets,keep", [
    (range(0, 1), 1.0),                        # one entry per row: 256 rows a block
    (range(-3, 4), 1.0),
    (range(-40, 41), 0.5),                     # odd and even lengths, empty rows none
    (range(-2, 3), 0.2),                       # empty rows, odd first entries
    (range(0, 2047), 1.0), (range(0, 2049), 1.0),   # one row fills or exceeds a chunk
    (range(0, 4096), 1.0),
    ((-70000, -1, 0, 1, 70000), 0.9),          # columns too far apart for 16 bits
])
def test_stream(dtype, offsets, keep):
    wide = max(offsets) > 60000
    n = 150001 if wide else (9 if max(offsets) > 2000 else 1037)
    rp, cols, vals = banded(n, n + (2100 if max(offsets) > 2000 else 0), offsets, keep, 5)
    check(rp, cols, vals, n + (2100 if max(offsets) > 2000 else 0), dtype)


@pytest.mark.parametrize("dtype,n", [(np.float32, (1 << 18) + 37), (np.float64, (1 << 20) + 1)])
@pytest.mark.parametrize("offsets,keep", [
    # 32, 27 and 16 entries at most, columns in up to four bands
    ([-40000, -39999] + list(range(-13, 15)) + [39999, 40000], 1.0),
    (sorted([b + i for b in (-30000, 0, 30000) for i in range(-4, 5)]), 0.97),
    ([-17, -16, -1, 0, 1, 17], 0.4),           # empty rows
    ([-90000, -60000, -30000, 0, 30000], 0.9),  # five bands: no windows, stream kernel
])
def test_row_lanes(dtype, n, offsets, keep):
    rp, cols, vals = banded(n, n, offsets, keep, 7)
    check(rp, cols, vals, n, dtype)


def test_row_lanes_rectangular():
    """Fewer columns than rows; the last rows are empty."""
    rp, cols, vals = banded((1 << 18) + 5, 1 << 18, range(0, 5), 1.0, 3)
    check(rp, cols, vals, 1 << 18, np.float32)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [1, 255, 257, (1 << 18) + 3])
def test_no_entries(dtype, n):
    """Rows without any entry: the product adds nothing, whatever the kernel,
    and CG of b = 0 stops at once with x as it was."""
    def matrix():
        return la.MatrixCSR(np.zeros(n + 1, np.int64), np.zeros(0, np.int32), dtype=dtype)

    rng = np.random.default_rng(n)
    x = la.Vector.from_array(rng.standard_normal(n).astype(dtype))
    y0 = rng.standard_normal(n).astype(dtype)
    A = matrix()
    for lanes in (0, 1, 2, 64):
        A.set_lanes(lanes)
        y = la.Vector.from_array(y0)
        A.mult(x, y)
        assert np.array_equal(y.array, y0)
    A.autotune()
    y = la.Vector.from_array(y0)
    A.mult(x, y)
    assert np.array_equal(y.array, y0)
    S = la.MatrixCSR.shared(A, dtype)
    S.mult(x, y)
    assert np.array_equal(y.array, y0)
    for classic in (False, True):
        z = la.Vector.from_array(y0)
        r = solvers.cg(matrix(), la.Vector(n, dtype), z, classic=classic)
        assert r.converged and r.iterations == 0 and np.array_equal(z.array, y0)
