"""Batched CG at the edges of its 256-row chunks and of the 16 entries per row
that are loaded together, with systems joining between steps."""

import numpy as np
import pytest

from dolfinx_amd import la, serve

pytestmark = pytest.mark.gpu


def band_matrix(n, half, seed):
    """Symmetric band matrix with unit diagonal and row sums of |off-diagonal|
    at most 1/2: eigenvalues in [1/2, 3/2], condition number at most 3."""
    rng = np.random.default_rng(seed)
    D = np.eye(n)
    for k in range(1, min(half, n - 1) + 1):
        v = rng.uniform(-1.0, 1.0, n - k) / (4.0 * half)
        D[np.arange(n - k), np.arange(k, n)] = v
        D[np.arange(k, n), np.arange(n - k)] = v
    band = np.abs(np.subtract.outer(np.arange(n), np.arange(n))) <= half
    rp = np.concatenate([[0], np.cumsum(band.sum(1))])
    cols = np.nonzero(band)[1]
    A = la.MatrixCSR(rp, cols)
    A.data = D[band]
    return D, A


def solve(systems, joins_at):
    """Solutions with system i joining before step joins_at[i]."""
    B = serve.BatchSolver(len(systems), sum(len(b) for _, _, b in systems))
    held, slots = [], {}
    for step in range(60):
        for i, (_, A, b) in enumerate(systems):
            if joins_at[i] == step:
                bv, x = la.Vector.from_array(b), la.Vector(len(b))
                held.append((i, bv, x))
                slots[i] = B.add(A, bv, x, rtol=1e-12)
        B.step(3)
        done = B.status(list(slots.values()))[0]
        if len(slots) == len(systems) and done.all():
            break
    assert B.status(list(slots.values()))[1].all()
    return {i: x.array for i, _, x in held}


@pytest.mark.parametrize("half", [0, 7, 8, 20])  # rows of 1, 15, 17 and 41 entries
def test_chunk_edges(half):
    sizes = [1, 63, 64, 255, 256, 257, 511, 513, 1030]
    rng = np.random.default_rng(half)
    systems = [(*band_matrix(n, half, n), rng.standard_normal(n)) for n in sizes]
    together = solve(systems, [0] * len(sizes))
    late = solve(systems, [i % 3 for i in range(len(sizes))])
    for i, (D, A, b) in enumerate(systems):
        ref = np.linalg.solve(D, b)
        # |x - ref| <= cond (rtol + rounding) |ref|, cond <= 3
        assert np.linalg.norm(together[i] - ref) <= 1e-11 * np.linalg.norm(ref)
        assert np.array_equal(late[i], together[i])
        assert np.array_equal(solve([systems[i]], [0])[0], together[i])


def test_matrix_without_entries():
    """No diagonal and no entries: every product is zero, the solve stops at
    max_it without converging."""
    A = la.MatrixCSR(np.zeros(301, np.int64), np.zeros(0, np.int32))
    B = serve.BatchSolver(1, 300)
    b, x = la.Vector.from_array(np.ones(300)), la.Vector(300)
    slot = B.add(A, b, x, rtol=1e-8, max_it=2)
    B.step(4)
    done, conv, its, _ = B.status([slot])
    assert done[0] == 1 and conv[0] == 0 and its[0] == 2
