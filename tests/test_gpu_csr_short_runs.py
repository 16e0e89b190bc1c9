"""CSR and 2x2-block CSR products of workgroups with few entries (walked, or staged in as many rounds as they have entries
for), at the lines between the forms: bit for bit the oracle's sequential sums (so no tolerance)."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from gpu_util import call, dev, empty, host, p  # noqa: E402

RUNS = [0, 1, 255, 256, 257, 512, 513, 1024, 1025, 2049]  # entries of one workgroup


def matrix(rows, per_entry):
    """A workgroup of `rows` rows for each of RUNS, then a last one that is not full."""
    rng = np.random.default_rng(21)
    lens = np.concatenate([np.bincount(rng.integers(0, rows, run), minlength=rows) for run in RUNS] + [np.array([3, 0, 1])])
    ro = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    n = len(lens)
    return ro, rng.integers(0, n, ro[-1]).astype(np.int32), rng.standard_normal(per_entry * ro[-1]), rng.standard_normal(
        n * (2 if per_entry == 4 else 1))


def in_turn(ro, n, add):
    """add(rows, entries): entry j of every row in turn, the sequential sums."""
    lens = np.diff(ro)
    for j in range(int(lens.max())):
        i = np.flatnonzero(lens > j)
        add(i, ro[i] + j)


def test_csr():
    import alien_amd as aa
    ro, cols, vals, x = matrix(256, 1)
    n = len(ro) - 1
    print("case csr short runs", n, len(cols), flush=True)
    with aa.Context() as c:
        ref = orc.spmv(ro, cols, vals, x)
        y, y2, out = empty(n), empty(n), empty(1)
        a = [p(dev(ro)), p(dev(cols)), p(dev(vals)), p(dev(x))]
        call("alien_hip_spmv_csr_f64", c.h, n, *a, p(y))
        np.testing.assert_array_equal(host(y, c)[:n], ref)
        call("alien_hip_spmv_dot_csr_f64", c.h, n, *a, p(y2), p(out))
        np.testing.assert_array_equal(host(y2, c)[:n], ref)
        v32, x32 = vals.astype(np.float32), x.astype(np.float32)
        acc = np.zeros(n, np.float32)

        def add(i, k):
            acc[i] = acc[i] + v32[k] * x32[cols[k]]

        in_turn(ro, n, add)
        y32 = empty(n, torch.float32)
        call("alien_hip_spmv_csr_f32", c.h, n, a[0], a[1], p(dev(v32)), p(dev(x32)), p(y32))
        np.testing.assert_array_equal(host(y32, c)[:n], acc)


@pytest.mark.parametrize("kind", [np.float64, np.float32])
def test_blocks(kind):
    import alien_amd as aa
    ro, cols, vals, x = matrix(128, 4)
    vals, x = vals.astype(kind), x.astype(kind)
    n = len(ro) - 1
    print("case bsr2 short runs", n, len(cols), kind.__name__, flush=True)
    acc, v, x2 = np.zeros((n, 2), kind), vals.reshape(-1, 2, 2), x.reshape(-1, 2)  # v[block, column, row]

    def add(i, k):
        for u in range(2):
            acc[i] = acc[i] + v[k, u] * x2[cols[k], u][:, None]

    in_turn(ro, n, add)
    f32 = kind is np.float32
    y = empty(2 * n, torch.float32 if f32 else torch.float64)
    with aa.Context() as c:
        call("alien_hip_spmv_bsr2_f32" if f32 else "alien_hip_spmv_bsr2_f64", c.h, n, p(dev(ro)), p(dev(cols)), p(dev(vals)),
             p(dev(x)), p(y))
        np.testing.assert_array_equal(host(y, c)[:2 * n], acc.reshape(-1))
