"""Mixed CG's q = A p on symmetric values, read at their mirrors, against the general form, bit for bit.

The matrix ends in a block of its own whose right-hand side is 0: the iterates stay 0 there, so that one entry of
it, one FP32 step off its mirror, sends the same solve through the general form.
"""
import numpy as np
import pytest

import alien_amd as aa

pytestmark = pytest.mark.gpu

TAIL = 7000


def system(n, offsets, skew):
    d = np.array(sorted({0, *offsets, *(-o for o in offsets)}))
    row = np.repeat(np.arange(n), len(d))
    col = row + np.tile(d, n)
    keep = (col >= 0) & (col < n)
    row, col = row[keep], col[keep]
    vals = np.where(row == col, 7.0, -1.0 + 0.25 * ((row + col) % 5) / 5)
    cut = n - TAIL
    vals[(row < cut) != (col < cut)] = 0.0
    if skew:
        k = np.flatnonzero((row == n - 50) & (col == n - 50 - offsets[0]))[0]
        vals[k] = np.nextafter(np.float32(vals[k]), np.float32(0))
    ro = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))]).astype(np.int32)
    b = np.random.default_rng(n).standard_normal(n)
    b[cut:] = 0
    return ro, col.astype(np.int32), vals, b


@pytest.mark.parametrize("offsets", [(1, 61, 3001), (2, 61, 3001), (1, 64, 6400)])
@pytest.mark.parametrize("n", [(1 << 19) + 64, (1 << 19) + 128, 530001])
def test_same_bits_as_the_general_form(ctx, n, offsets):
    print("case", n, offsets, flush=True)
    got = []
    for skew in (False, True):
        ro, cols, vals, b = system(n, offsets, skew)
        x, r = aa.solve_csr(ctx, ro, cols, vals, b, solver=aa.CG, precond=aa.PREC_DIAG, mode=aa.MODE_MIXED, layout=aa.LAYOUT_RBDIA,
                            tol=1e-11, max_iter=400)
        assert r["status"] == 1
        got.append((x, r["iterations"]))
    assert got[0][1] == got[1][1]
    np.testing.assert_array_equal(got[0][0], got[1][0])
    q = np.add.reduceat(vals * got[0][0][cols], ro[:-1])
    assert np.linalg.norm(b - q) <= 2e-11 * np.linalg.norm(b)


def test_new_values_are_looked_at_again(ctx):
    """A kept matrix whose values become nonsymmetric and symmetric again."""
    n, offsets = 530001, (1, 61, 3001)
    ro, cols, sym, b = system(n, offsets, False)
    skewed = system(n, offsets, True)[2]
    kw = dict(solver=aa.CG, precond=aa.PREC_DIAG, mode=aa.MODE_MIXED, tol=1e-11, max_iter=400)
    with aa.Matrix(ctx, ro, cols, sym) as M:
        want = M.solve(b, **kw)[0]
        for vals in (skewed, sym, 2 * sym):
            M.update_values(vals)
            x = M.solve(b, **kw)[0]
            scale = vals[0] / sym[0] # a power of two: the iterates' bits but for the exponent
            np.testing.assert_array_equal(x * scale, want)
