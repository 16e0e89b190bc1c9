"""Iterations in one launch: rows of 6 to 9 entries (8 and 9 are left to the launches, on either side), some of them
missing, in one workgroup and in several, against the same solve from launches, bit for bit."""
import os

import numpy as np
import pytest

import alien_amd as aa

pytestmark = pytest.mark.gpu

OFFSETS = {6: (-40, -1, 1, 37, 41), 7: (-37, -5, -1, 1, 5, 37), 8: (-41, -37, -5, -1, 1, 5, 37), 9: (-41, -37, -5, -1, 1, 5, 37, 41)}


def matrix(n, width):
    """Diagonally dominant (the symmetric part too: |row sum| and |column sum| of the off-diagonals < 9); every
    third row lacks its first entry, every fifth one its last."""
    d = np.array(sorted((0, *OFFSETS[width])))
    row, k = np.repeat(np.arange(n), len(d)), np.tile(np.arange(len(d)), n)
    col = row + d[k]
    keep = (col >= 0) & (col < n) & ~((row % 3 == 0) & (k == 0)) & ~((row % 5 == 0) & (k == len(d) - 1))
    row, col = row[keep], col[keep].astype(np.int32)
    ro = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))]).astype(np.int32)
    vals = np.where(row == col, 9.0, -0.5 - 0.5 * ((row + col) % 7) / 7)
    return ro, col, vals


@pytest.fixture(scope="module")
def contexts():
    os.environ["ALIEN_HIP_CG_RESIDENT"] = "0"  # read when a context is created
    launches = aa.Context()
    del os.environ["ALIEN_HIP_CG_RESIDENT"]
    with aa.Context() as resident, launches:
        yield launches, resident


@pytest.mark.parametrize("special", [None, np.inf, -0.0])
@pytest.mark.parametrize("n", [50, 1000, 1025, 1386, 2047, 2048, 2049, 5000])
@pytest.mark.parametrize("width", list(OFFSETS))
def test_width(contexts, width, n, special):
    ro, cols, vals = matrix(n, width)
    b = np.random.default_rng(n).standard_normal(n)
    if special is not None:
        b[n // 2] = special
    for precond in (aa.PREC_DIAG, aa.PREC_CHEB):
        for mode in (aa.MODE_GRAPH, aa.MODE_MIXED):
            print("case", width, n, special, precond, mode, flush=True)
            # (the matrix is not symmetric: a fixed number of steps, not a converged solve, is compared)
            (x, r), (gx, gr) = (aa.solve_csr(c, ro, cols, vals, b, solver=aa.CG, precond=precond, mode=mode, tol=1e-11,
                                             max_iter=40, poll_every=4) for c in contexts)
            np.testing.assert_array_equal(gx, x)
            assert all(np.array_equal(gr[k], r[k], equal_nan=True) for k in ("iterations", "status", "error"))
