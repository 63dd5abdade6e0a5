"""SpMV kernels at the edges of their chunks, pairs, row groups and column
encodings, against scipy in FP64."""

import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sps

from dolfinx_amd import _lib, la, solvers

pytestmark = pytest.mark.gpu


def banded(nrows, ncols, offsets, keep, seed, empty=0):
    """Pattern with the columns r + offset of each row r that exist, each kept
    with probability keep (every `empty`-th row without any); random values."""
    rng = np.random.default_rng(seed)
    c = np.arange(nrows)[:, None] + np.asarray(offsets)[None, :]
    on = (c >= 0) & (c < ncols) & (rng.random(c.shape) < keep)
    if empty:
        on[::empty] = False
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


SPACED = {16: range(-320, 320, 40), 27: range(-520, 521, 40)}
BANDS = {27: sorted([b + 40 * i for b in (-30000, 0, 30000) for i in range(-4, 5)]),
         32: [-60000, -30000] + list(range(-420, 420, 30)) + [30000, 30040]}


@pytest.mark.parametrize("dtype,n", [(np.float32, (1 << 18) + 37), (np.float64, (1 << 20) + 1)])
@pytest.mark.parametrize("offsets,keep,empty,rows", [
    (BANDS[32], 1.0, 0, True), (BANDS[27], 0.995, 0, True), (SPACED[27], 1.0, 5, True),
    (SPACED[16], 1.0, 3, np.float32),         # FP64 rows of 16 stay on the stream
    (range(-1, 2), 1.0, 0, False), (range(-13, 14), 1.0, 0, False),  # few lines per row
    ([-10000, -100, -1, 0, 1, 100, 10000], 1.0, 0, False),
    (SPACED[27], 0.5, 0, False),              # the same columns never side by side
])
def test_row_lane_choice(dtype, n, offsets, keep, empty, rows):
    """Large matrices whose gathers touch half the lines in row order are
    served by the row-lane kernel (its bits differ from the stream's), others
    of any size by the stream."""
    rp, cols, vals = banded(n, n, offsets, keep, 13, empty)
    A = la.MatrixCSR(rp, cols, dtype=dtype)
    A.data = vals
    x = la.Vector.from_array(np.random.default_rng(1).standard_normal(n).astype(dtype))
    y = product(A, x)
    A.set_lanes(1)
    assert np.array_equal(product(A, x), y) == (rows not in (True, dtype))
    S = sps.csr_matrix((vals.astype(dtype).astype(np.float64), cols, rp), shape=(n, n))
    xd = x.array.astype(np.float64)
    assert (np.abs(y - S @ xd) <= 35 * np.finfo(dtype).eps * (abs(S) @ abs(xd))).all()


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


def product(A, x):
    y = la.Vector(A.shape[0], A.dtype)
    A.mult(x, y)
    return y.array


def test_kernel_of_a_large_matrix():
    """set_lanes(1) and the autotuner reach the row-block stream on a matrix
    that the row-lane kernel serves by default (the bits of its first rows are
    those of a smaller matrix, which the stream serves), and a copy of the
    pattern in the other precision takes the kernel of its own size rule."""
    n, cut = (1 << 18) + 37, 100000
    rp, cols, vals = banded(n, n, range(-520, 521, 40), 0.995, 7)
    A = la.MatrixCSR(rp, cols, dtype=np.float32)
    A.data = vals
    B = la.MatrixCSR(rp[:cut + 1], cols[:rp[cut]], ncols=n, dtype=np.float32)
    B.data = vals[:rp[cut]]
    x = la.Vector.from_array(np.random.default_rng(1).standard_normal(n).astype(np.float32))
    rows, few = product(A, x), product(B, x)[:cut - 256]
    A.set_lanes(1)
    assert np.array_equal(product(A, x)[:cut - 256], few)
    assert not np.array_equal(rows[:cut - 256], few)
    assert A.autotune()[0] in (0, 1, 2, 4, 8, 16, 32, 64)
    A.set_lanes(0)
    assert np.array_equal(product(A, x), rows)
    # FP64 rows of this length need 2^20 rows: 8 lanes per row (27 entries)
    D = la.MatrixCSR.shared(A, np.float64)
    D.data = vals
    xd = la.Vector.from_array(x.array.astype(np.float64))
    default = product(D, xd)
    D.set_lanes(8)
    assert np.array_equal(default, product(D, xd))


def test_shared_pattern_of_the_other_precision():
    """FP32 values on a large FP64 pattern: the autotuner times the row-lane
    kernel too and its choice gives the same product."""
    n = (1 << 20) + 1
    rp, cols, vals = banded(n, n, range(-520, 521, 40), 1.0, 11)
    A = la.MatrixCSR.shared(la.MatrixCSR(rp, cols), np.float32)
    A.data = vals
    x = la.Vector.from_array(np.random.default_rng(1).standard_normal(n).astype(np.float32))
    S = sps.csr_matrix((vals.astype(np.float32).astype(np.float64), cols, rp), shape=(n, n))
    xd = x.array.astype(np.float64)
    bound = 30 * np.finfo(np.float32).eps * (abs(S) @ abs(xd))
    assert (np.abs(product(A, x) - S @ xd) <= bound).all()
    assert A.autotune()[0] == 0  # (38 us; 2 to 64 lanes per row 60 or more)
    assert (np.abs(product(A, x) - S @ xd) <= bound).all()


@pytest.mark.parametrize("dtype,n", [(np.float32, (1 << 18) + 37), (np.float64, (1 << 20) + 37)])
def test_cg_through_the_row_lane_kernel(dtype, n):
    """CG whose product is the row-lane kernel (its partial sums and stop flag;
    an odd number of groups, the last of 37 rows): rows of 27 scattered entries
    with every fifth its diagonal alone, which the sliced-ELL copy would pad by
    a quarter. The residual is checked on the host, the iterations against the
    stream's, and the no-allocation solve where it takes the size."""
    rp, cols, _ = banded(n, n, range(-520, 521, 40), 1.0, 3)
    row = np.repeat(np.arange(n), np.diff(rp))
    on = (row % 5 != 0) | (cols == row)       # (40 k keeps the remainder: symmetric)
    row, cols = row[on], cols[on]
    rp = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))])
    vals = np.where(cols == row, 1.0 + row % 3, -0.5 / 26).astype(dtype)
    b = np.random.default_rng(5).standard_normal(n).astype(dtype)
    S = sps.csr_matrix((vals.astype(np.float64), cols, rp), shape=(n, n))
    rtol = 1e-10 if dtype == np.float64 else 1e-5
    A = la.MatrixCSR(rp, cols, dtype=dtype)
    A.data = vals
    bv, its, ys = la.Vector.from_array(b), [], []

    def solve(name):
        x, opts, res = la.Vector(n, dtype), _lib.CGOpts(200, rtol, 1, 7, 0, 0), _lib.CGResult()
        _lib.call(name, A.handle, bv.handle, x.handle, C.byref(opts), C.byref(res))
        r = b.astype(np.float64) - S @ x.array.astype(np.float64)
        assert np.linalg.norm(r) <= (2 * rtol + 100 * np.finfo(dtype).eps) * np.linalg.norm(b)
        return res.iterations

    for lanes in (0, 1):
        A.set_lanes(lanes)
        its.append(solve("dfx_cg_solve"))
        ys.append(product(A, bv))
        if n <= 1 << 20:
            its.append(solve("dfx_cg_solve_noalloc"))
    assert max(its) - min(its) <= 1 and 3 < its[0] < 60
    assert not np.array_equal(*ys)            # (two kernels)
