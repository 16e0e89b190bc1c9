"""CSR and 2x2-block CSR products whose rows' entries are staged through LDS, at the edges of their tiles, runs and
grids: bit for bit the oracle's sequential sums (so no tolerance)."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from gpu_util import call, dev, empty, host, p  # noqa: E402


def lengths(case, rows):
    """Entries per row; `rows`: rows per workgroup."""
    rng = np.random.default_rng(11)
    if case == "one":
        return np.array([1])
    if case == "empty":
        return np.zeros(rows + 1, int)
    if case == "short of a block":
        return rng.integers(0, 9, rows - 1)
    if case == "a block and a row":
        return np.full(rows + 1, 8)  # whole tiles of 2048 entries, then one row
    if case == "rows over several tiles":
        n = rng.integers(0, 5, 2 * rows + 7)
        n[[0, rows - 1, rows, 2 * rows + 6]] = [4999, 2048, 2049, 5001]
        return n
    if case == "at the walk's line":  # 64 a row on average: staged; one entry more: walked
        n = np.full(2 * rows, 64)
        n[rows] += 1
        return n
    if case == "walked":
        return rng.integers(60, 140, rows + 3)
    assert case == "grid in XCD chunks"
    return rng.integers(0, 3, 4 * 512 * rows + 5)


CASES = ["one", "empty", "short of a block", "a block and a row", "rows over several tiles", "at the walk's line", "walked",
         "grid in XCD chunks"]


def matrix(case, rows, per_entry):
    rng = np.random.default_rng(12)
    n = lengths(case, rows)
    ro = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    cols = rng.integers(0, len(n), ro[-1]).astype(np.int32)
    return ro, cols, rng.standard_normal(per_entry * len(cols)), rng.standard_normal(len(n) * (2 if per_entry == 4 else 1))


@pytest.mark.parametrize("case", CASES)
def test_csr_products(ctx, case):
    ro, cols, vals, x = matrix(case, 256, 1)
    n = len(ro) - 1
    print("case csr", case, n, len(cols), flush=True)
    ref = orc.spmv(ro, cols, vals, x)
    d = [dev(ro), dev(np.append(cols, np.int32(0))), dev(np.append(vals, 0.0))]
    y, y2, out = empty(n), empty(n), empty(1)
    call("alien_hip_spmv_csr_f64", ctx.h, n, *map(p, d), p(dev(x)), p(y))
    np.testing.assert_array_equal(host(y, ctx)[:n], ref)
    call("alien_hip_spmv_dot_csr_f64", ctx.h, n, *map(p, d), p(dev(x)), p(y2), p(out))
    np.testing.assert_array_equal(host(y2, ctx)[:n], ref)
    # n additions of rounded products: |error| <= (n + 1) eps sum |x_i y_i|
    assert abs(host(out, ctx)[0] - np.dot(x, ref)) <= (n + 1) * 2.0**-52 * np.dot(np.abs(x), np.abs(ref))
    v32, x32 = vals.astype(np.float32), x.astype(np.float32)
    y32 = empty(n, torch.float32)
    call("alien_hip_spmv_csr_f32", ctx.h, n, p(d[0]), p(d[1]), p(dev(np.append(v32, np.float32(0)))), p(dev(x32)), p(y32))
    acc = np.zeros(n, np.float32)  # entry j of every row in turn: the sequential sum in FP32
    for j in range(int(np.diff(ro).max(initial=0))):
        i = np.flatnonzero(np.diff(ro) > j)
        acc[i] = acc[i] + v32[ro[i] + j] * x32[cols[ro[i] + j]]
    np.testing.assert_array_equal(host(y32, ctx)[:n], acc)


@pytest.mark.parametrize("case", CASES)
def test_block_products(ctx, case):
    ro, cols, vals, x = matrix(case, 128, 4)
    n = len(ro) - 1
    print("case bsr2", case, n, len(cols), flush=True)
    y = empty(2 * n)
    call("alien_hip_spmv_bsr2_f64", ctx.h, n, p(dev(ro)), p(dev(np.append(cols, np.int32(0)))), p(dev(np.append(vals, [0.0] * 4))), p(dev(x)), p(y))
    np.testing.assert_array_equal(host(y, ctx)[:2 * n], orc.spmv_bsr(ro, cols, vals, x))
