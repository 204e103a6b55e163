"""Plain CRS rows (the zero-allocation solve's matrix, format 9): a wave takes
the entries of its 64 rows a tile of 512 at a time and hands the products to the
rows' threads."""
import time

import numpy as np
import pytest

import ogs5_amd as ox
from devbuf import DevArray

pytestmark = pytest.mark.gpu


def _solve(n, ptr, col, val, b, **kw):
    dev = [DevArray(a) for a in (ptr.astype(np.int32), col.astype(np.int32), val, b)]
    x = DevArray(np.zeros(n))
    t = time.perf_counter()
    info, _ = ox.solve_crs_noalloc(n, *(d.ptr for d in dev), x.ptr, **kw)
    t = time.perf_counter() - t
    got = x.get()
    for d in dev + [x]:
        d.free()
    return got, info, t


# lengths of 64 rows: a tile exactly, one entry more and less, half a tile, a row
# across three tiles and one of a tile, a slice that ends in a short one
@pytest.mark.parametrize("lengths", [
    [8] * 64, [8] * 63 + [9], [8] * 63 + [7], [4] * 64, [4] * 63 + [5],
    [1] * 30 + [1400] + [1] * 33, [512] + [1] * 63, [1] * 63 + [40], [28, 1, 900] * 40 + [3]])
@pytest.mark.parametrize("method", [ox.CG, ox.BICGSTAB])
def test_row_lengths(lengths, method):
    """One row longer than 27 entries keeps the solve to separate launches.  The
    sums are CSparseMatrix::multiVec's: products rounded, added left to right."""
    n = 3000
    rng = np.random.default_rng(len(lengths))
    want = np.resize(lengths, n)
    want[-1] = max(want[-1], 29)
    rows, cols = [], []
    for i, k in enumerate(want):  # a symmetric pattern of at least these lengths
        rows.append(np.full(k, i))
        cols.append(rng.integers(0, n, k))
    r, c = np.concatenate(rows), np.concatenate(cols)
    key = np.unique(np.concatenate([r * n + c, c * n + r, np.arange(n) * (n + 1)]))
    row, col = key // n, key % n
    off = -1.0 / (1.0 + np.abs(row - col))
    val = np.where(row == col, 1.0, off)
    val[row == col] = 1.5 - np.bincount(row, np.where(row == col, 0.0, off), n)
    ptr = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))])
    b = rng.standard_normal(n)
    x, info, _ = _solve(n, ptr, col, val, b, tol=1e-12, max_iter=500, method=method)
    assert info["converged"] == 1
    res = np.linalg.norm(b - np.bincount(row, val * x[col], n))
    assert res <= 1e-11 * np.linalg.norm(b)  # the recurrence's stop, and rounding
    again, _, _ = _solve(n, ptr, col, val, b, tol=1e-12, max_iter=500, method=method)
    assert np.array_equal(x, again)


def test_long_rows_of_a_large_system():
    """Rows of 27 entries past the resident sizes.  33 us per iteration; lines of
    the matrix loaded once per entry took 211."""
    s = 61
    n = s ** 3
    o = np.array([-1, 0, 1])
    off = (o[:, None, None] * s * s + o[None, :, None] * s + o).ravel()
    cols = np.arange(n)[:, None] + off
    have = (cols >= 0) & (cols < n)
    val = np.broadcast_to(np.where(off == 0, 27.0, -1.0), cols.shape)[have]
    ptr = np.concatenate([[0], np.cumsum(have.sum(1))])
    b = np.random.default_rng(1).standard_normal(n)
    args = (n, ptr, cols[have], np.ascontiguousarray(val), b)
    for _ in range(2):
        x, info, t = _solve(*args, tol=1e-30, max_iter=100)
    assert info["iterations"] == 100
    print(f"{t * 1e4:.1f} us per iteration")
    assert t < 100 * 120e-6
