"""The 64 x 64 tile factorization on the GPU (LU in LDS with pivoting inside the
tile, by panels of four columns, its triangular inverses, the last tile's solve),
through solve_tau00_matrix, against LAPACK.

Sizes at the edges of the tile and of its panels, every kind of right-hand-side
count.  Tolerance: the backward error of LU with partial
pivoting is a small multiple of n eps here (no growth: random matrices and
matrices near 1), so the forward error is held to 8 n eps cond(M)."""
import numpy as np
import pytest

from lsms_amd import capi

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def matrix(kind, n, k, rng):
    """Rows of the 64-tiles (counted from the end, where the solver keeps the
    central block) scrambled, so that pivots are anywhere in their tile; the
    central k rows among themselves only."""
    if kind == "ties":  # entries of equal magnitude: every search ties
        m = rng.choice([-1.0, 1.0], size=(n, n)) + 1j * rng.choice([-1.0, 1.0], size=(n, n))
        m = np.where(rng.random((n, n)) < 0.15, m, 0.0) + 4.0 * np.eye(n)
    else:
        m = (rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))) * (0.3 / np.sqrt(n)) + np.eye(n)
    # solver order: non-central rows k..n-1 first, then the central rows 0..k-1
    order = np.concatenate([np.arange(k, n), np.arange(k)])
    pad = -n % 64
    for lo in range(0, n + pad, 64):
        idx = np.arange(max(lo - pad, 0), min(lo + 64 - pad, n))
        for part in (idx[idx < n - k], idx[idx >= n - k]):
            rows = order[part]
            m[rows] = m[rng.permutation(rows)]
    return m


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("kind", ["near1", "ties"])
@pytest.mark.parametrize("n,k", [(1, 1), (8, 8), (9, 4), (16, 16), (63, 16), (64, 1), (64, 64),
                                 (65, 9), (71, 16), (72, 32), (127, 33), (128, 17), (200, 50)])
def test_tile_solve(ctx, kind, n, k):
    rng = np.random.default_rng(1000 * n + k)
    m = matrix(kind, n, k, rng)
    t = rng.normal(size=(k, k)) + 1j * rng.normal(size=(k, k))
    tau, info = ctx.solve_tau00_matrix(m, t)
    rhs = np.zeros((n, k), dtype=complex)
    rhs[:k] = t
    ref = np.linalg.solve(m, rhs)[:k]
    assert info == 0
    assert np.linalg.norm(tau - ref) <= 8 * n * EPS * np.linalg.cond(m) * np.linalg.norm(ref)


@pytest.mark.parametrize("col", [0, 7, 8, 40, 63])
def test_zero_pivot_position(ctx, col):
    """A zero column of the first tile: info names it (1-based, solver order)."""
    n, k = 128, 16
    rng = np.random.default_rng(col)
    m = matrix("near1", n, k, rng)
    m[:, k + col] = 0.0
    _, info = ctx.solve_tau00_matrix(m, np.eye(k, dtype=complex))
    assert info == col + 1


@pytest.mark.parametrize("n,k", [(3, 2), (4, 4), (5, 1), (61, 3), (67, 4), (68, 5), (69, 8)])
def test_panel_edges(ctx, n, k):
    """Sizes on both sides of a panel of four columns."""
    test_tile_solve(ctx, "near1", n, k)
    test_tile_solve(ctx, "ties", n, k)
