"""The COO solve's product at the edges of its row split: mean row lengths on
both sides of each lane count, a dense row among short ones, empty rows, and
systems with fewer triplets than the sort area needs for a second direction;
against numpy's solve."""
import numpy as np
import pytest

from sbs_amd import capi
from sbs_amd.linear import PCGJacobiSolver

pytestmark = pytest.mark.gpu


def band(n, half, rng):
    r = np.repeat(np.arange(n), 2 * half + 1)
    c = r + np.tile(np.arange(-half, half + 1), n)
    ok = (c >= 0) & (c < n)
    r, c = r[ok], c[ok]
    lo, hi = np.minimum(r, c), np.maximum(r, c)
    v = np.where(r == c, 2.0 * half + 2.0, -1.0 + 0.5 * np.sin(lo * 7.0 + hi * 3.0))
    p = rng.permutation(len(r))
    return r[p], c[p], v[p]


def solve(n, r, c, v, b, precision):
    dt = np.float32 if precision == 32 else np.float64
    bufs = [capi.DeviceArray.from_numpy(a) for a in (b.astype(dt), np.zeros(n, dt), v.astype(dt), r.astype(np.int32),
                                                     c.astype(np.int32))]
    s = PCGJacobiSolver(n, max_iter=4 * n + 50, tolerance=1e-4 if precision == 32 else 1e-10, precision=precision)
    s.Solve(n, bufs[0], bufs[1], bufs[2], len(v), bufs[3], bufs[4])
    s.Solve(n, bufs[0], bufs[1], bufs[2], len(v), bufs[3], bufs[4])   # the host's looks follow the first count
    x = bufs[1].download(dt, (n,)).astype(np.float64)
    s.close()
    return x


# mean entries per row around 1, 2 | 8 | 16 | 32 | 64 | 128 | 256, where the lanes double
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("n,half", [(1, 0), (255, 0), (257, 3), (300, 4), (300, 7), (513, 8), (400, 16), (700, 33),
                                    (600, 70), (700, 140)])
def test_row_lengths(gpu, n, half, precision):
    rng = np.random.default_rng(n + half)
    r, c, v = band(n, half, rng)
    A = np.zeros((n, n))
    np.add.at(A, (r, c), v)
    b = rng.normal(size=n)
    x = solve(n, r, c, v, b, precision)
    # strictly diagonally dominant by at least 2: |A^-1| <= 1/2.  The solve
    # stops at |r| < tol or at |r.z| = sum r^2 / d < 1e-15, where |r| is below
    # sqrt(1e-15 max d); rounding adds cond(A) units
    u = np.finfo(np.float32 if precision == 32 else np.float64).eps
    stop = max(1e-4 if precision == 32 else 1e-10, np.sqrt(1e-15 * np.diag(A).max()))
    bound = stop / 2 + 50 * u * np.linalg.cond(A) * np.linalg.norm(x)
    assert np.linalg.norm(x - np.linalg.solve(A, b)) <= bound


@pytest.mark.parametrize("n", [64, 1000])
def test_dense_row_and_empty_rows(gpu, n):
    """Row and column 0 full, a diagonal elsewhere but on the last rows, whose
    right-hand side is 0 (a missing diagonal counts as 1)."""
    m = n - 5
    r = np.concatenate([np.arange(m), np.zeros(m - 1, int), np.arange(1, m)])
    c = np.concatenate([np.arange(m), np.arange(1, m), np.zeros(m - 1, int)])
    v = np.concatenate([np.r_[float(n), np.full(m - 1, 2.0)], np.full(2 * (m - 1), 0.5)])
    A = np.zeros((n, n))
    np.add.at(A, (r, c), v)
    b = np.r_[np.linspace(-1, 1, m), np.zeros(5)]
    x = solve(n, r, c, v, b, 64)
    assert np.all(x[m:] == 0)
    # |r| stops below sqrt(1e-15 n) (see above); the smallest eigenvalue is over 1
    assert np.linalg.norm(x[:m] - np.linalg.solve(A[:m, :m], b[:m])) <= np.sqrt(1e-15 * n)


def test_fewer_triplets_than_rows(gpu):
    """Too few triplets for a second direction in the sort's area: the
    direction is formed in place."""
    n = 5000
    r = np.arange(0, 40)
    b = np.zeros(n)
    b[:40] = np.arange(1, 41)
    x = solve(n, r, r, np.full(40, 4.0), b, 64)
    assert np.allclose(x, b / 4.0, rtol=1e-12, atol=0)
