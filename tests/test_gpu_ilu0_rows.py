"""ILU(0) factorisation in one launch, a wavefront per row (matrices whose rows update more than their pivots), against one
launch per level, bit for bit: rows of up to 64 entries and more, columns' rows wider than a wavefront, rows without lower
or without upper entries, several rows a ticket, every wait given up; and matrices at the line between the two kernels."""
import numpy as np
import pytest

import alien_amd as aa
from test_gpu_ilu0_sync import banded

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from gpu_util import call, dev, host, p  # noqa: E402

ENV = {"launches": {"ALIEN_HIP_ILU_SYNC_FREE": "0"}, "one launch": {}, "gives up": {"ALIEN_HIP_ILU_SF_SPINS": "0"}}
DEFAULTS = {"ALIEN_HIP_ILU_SYNC_FREE": "1", "ALIEN_HIP_ILU_SF_SPINS": "65536"}


def wide(n, width, seed):
    """Bands of `width` neighbours on each side, some missing: rows of up to 2 width + 1 entries."""
    return banded(n, tuple(range(-width, width + 1)), seed)


def mixed(n, share, seed):
    """7-point-like rows, `share` of them with a second entry beside the far one: the latter are not plain."""
    rng = np.random.default_rng(seed)
    rows = {}
    for i in range(n):
        c = [i + o for o in (-60, -8, -1, 0, 1, 8, 60)]
        if rng.random() < share:
            c += [i - 59, i + 7]
        rows[i] = sorted({j for j in c if 0 <= j < n})
    cols = np.concatenate([rows[i] for i in range(n)]).astype(np.int32)
    ro = np.concatenate([[0], np.cumsum([len(rows[i]) for i in range(n)])]).astype(np.int32)
    row = np.repeat(np.arange(n), np.diff(ro))
    vals = -rng.random(len(cols)) - 1e-3
    vals[row == cols] = 12.0
    return ro, cols, vals


CASES = {
    "9-point": lambda: banded(4000, (-51, -50, -49, -1, 0, 1, 49, 50, 51), 1),
    "27 entries": lambda: banded(6000, tuple(a + b + c for a in (-400, 0, 400) for b in (-20, 0, 20) for c in (-1, 0, 1)), 2),
    "63 entries": lambda: wide(700, 31, 3),
    "65 entries": lambda: wide(700, 32, 4),
    "150 entries": lambda: wide(600, 75, 5),
    "few rows": lambda: wide(5, 2, 6),
    "diagonal blocks": lambda: banded(3000, (-2, -1, 0, 1, 2), 7),
    "several rows a ticket": lambda: banded(120000, (-12001, -12000, -11999, 0, 11999, 12000, 12001), 8),
    "a tenth not plain": lambda: mixed(5000, 0.1, 9),
    "a sixth not plain": lambda: mixed(5000, 0.17, 10),
}


@pytest.mark.parametrize("case", list(CASES))
def test_rows(monkeypatch, case):
    ro, cols, vals = CASES[case]()
    n = len(ro) - 1
    dcol = aa.host_dcol(ro, cols)
    lp, lr = aa.group_by_level(*aa.host_levels(ro, cols, dcol, False))
    lp = np.ascontiguousarray(lp, np.int32)
    A = [dev(ro), dev(cols), dev(dcol)]
    got = {}
    try:
        for name, env in ENV.items():
            for k, v in DEFAULTS.items():
                monkeypatch.setenv(k, env.get(k, v))
            with aa.Context() as c:  # the variables are read when a context is created
                print("case", case, name, n, len(lp) - 1, int(np.diff(ro).max()), flush=True)
                lu = dev(vals)
                call("alien_hip_ilu0_factor_f64", c.h, n, *map(p, A), p(lu), len(lp) - 1, aa._capi.iptr(lp),
                     p(dev(lr.astype(np.int32))))
                got[name] = host(lu, c)
    finally:
        for k, v in DEFAULTS.items():
            monkeypatch.setenv(k, v)
        aa.Context().close()
    for name in ("one launch", "gives up"):
        np.testing.assert_array_equal(got[name], got["launches"], err_msg=name)
