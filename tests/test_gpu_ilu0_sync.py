"""ILU(0) factorisation and sweeps in one launch each, against one launch per level, through the C entry points: bit for
bit (the same operations in the same order), on patterns with and without updates of strictly-upper entries, schedules
whose levels are smaller than a wavefront, and outputs that share memory."""
import numpy as np
import pytest

import alien_amd as aa

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from gpu_util import call, dev, empty, host, p  # noqa: E402


def banded(n, offsets, seed):
    """Rows with a random subset of the offsets, values in [-1, 0), diagonally dominant."""
    rng = np.random.default_rng(seed)
    row, col = [], []
    for o in offsets:
        i = np.arange(max(0, -o), min(n, n - o))
        i = i if o == 0 else i[rng.random(len(i)) < 0.8]
        row.append(i)
        col.append(i + o)
    row, col = np.concatenate(row), np.concatenate(col)
    order = np.lexsort((col, row))
    row, col = row[order], col[order].astype(np.int32)
    vals = -rng.random(len(col)) - 1e-3
    vals[row == col] = np.bincount(row, -vals)[row[row == col]] + 1.0
    return np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))]).astype(np.int32), col, vals


CASES = {
    "chain": lambda: banded(300, (-1, 0, 1), 1),  # one row a level
    "fill": lambda: banded(5000, (-70, -69, -2, -1, 0, 1, 2, 69, 70), 2),  # upper entries are updated
    "wide": lambda: banded(20000, (-900, -899, -898, -1, 0, 898, 899, 900), 3),
    "grid 7-point": lambda: aa.gen_csr(aa.GEN_CONVDIFF7, 21, 18, 19),
    "one chunk": lambda: banded(64, (-9, 0, 9), 4),
    "a row over": lambda: banded(65, (-9, -3, 0, 3, 9), 5),
}


@pytest.fixture(scope="module")
def contexts():
    import os
    runs = {"launches": {"ALIEN_HIP_ILU_SYNC_FREE": "0"}, "sync": {}, "gives up": {"ALIEN_HIP_ILU_SF_SPINS": "0"}}
    yield runs
    os.environ.update({"ALIEN_HIP_ILU_SYNC_FREE": "1", "ALIEN_HIP_ILU_SF_SPINS": "65536"})
    aa.Context().close()
    del os.environ["ALIEN_HIP_ILU_SYNC_FREE"], os.environ["ALIEN_HIP_ILU_SF_SPINS"]


@pytest.mark.parametrize("case", list(CASES))
def test_factor_and_solve(monkeypatch, contexts, case):
    ro, cols, vals = CASES[case]()
    n = len(ro) - 1
    dcol = aa.host_dcol(ro, cols)
    lower, upper = (aa.group_by_level(*aa.host_levels(ro, cols, dcol, u)) for u in (False, True))
    y = np.random.default_rng(9).standard_normal(n)
    A = [dev(ro), dev(cols), dev(dcol)]
    sched = []
    for ptr, rows in (lower, upper):
        ptr = np.ascontiguousarray(ptr, np.int32)
        sched.append((len(ptr) - 1, ptr, dev(rows.astype(np.int32))))
    (nl, lp, lr), (nu, up, ur) = sched
    got = {}
    for name, env in contexts.items():
        for k, v in {"ALIEN_HIP_ILU_SYNC_FREE": "1", "ALIEN_HIP_ILU_SF_SPINS": "65536", **env}.items():
            monkeypatch.setenv(k, v)
        with aa.Context() as c:  # the variables are read when a context is created
            print("case", case, name, n, nl, nu, flush=True)
            lu = dev(vals)
            call("alien_hip_ilu0_factor_f64", c.h, n, *map(p, A), p(lu), nl, aa._capi.iptr(lp), p(lr))
            got[name, "lu"] = host(lu, c)
            # y, t and x apart; x in y's place; t in y's place; x in t's place
            for form in ("apart", "x is y", "t is y", "x is t"):
                dy, t, x = dev(y), empty(n), empty(n)
                x = dy if form == "x is y" else x
                t = dy if form == "t is y" else t
                x = t if form == "x is t" else x
                call("alien_hip_ilu0_solve_f64", c.h, n, *map(p, A), p(lu), nl, aa._capi.iptr(lp), p(lr), nu,
                     aa._capi.iptr(up), p(ur), p(dy), p(t), p(x))
                got[name, form] = host(x, c)[:n]
    for (name, what), v in got.items():
        np.testing.assert_array_equal(v, got["launches", what], err_msg=name + " " + what)
    for form in ("x is y", "t is y", "x is t"):
        np.testing.assert_array_equal(got["sync", form], got["sync", "apart"])


def test_under_capture():
    """In a graph captured on the context's stream, replayed with eager work between: the eager result each time."""
    ro, cols, vals = CASES["fill"]()
    n = len(ro) - 1
    dcol = aa.host_dcol(ro, cols)
    (lp, lr), (up, ur) = (aa.group_by_level(*aa.host_levels(ro, cols, dcol, u)) for u in (False, True))
    s = torch.cuda.Stream()
    with aa.Context(s.cuda_stream) as c:
        d = [dev(a) for a in (ro, cols, dcol, vals, lr.astype(np.int32), ur.astype(np.int32), np.random.default_rng(3).random(n))]
        lu, t, x = empty(len(cols)), empty(n), empty(n)
        ptr = lambda a: aa._capi.C.c_void_p(a.data_ptr())  # noqa: E731

        def work():
            L = aa.lib()
            aa.check(L.alien_hip_copy_f64(c.h, len(cols), ptr(d[3]), ptr(lu)))
            aa.check(L.alien_hip_ilu0_factor_f64(c.h, n, ptr(d[0]), ptr(d[1]), ptr(d[2]), ptr(lu), len(lp) - 1, aa._capi.iptr(lp), ptr(d[4])))
            aa.check(L.alien_hip_ilu0_solve_f64(c.h, n, ptr(d[0]), ptr(d[1]), ptr(d[2]), ptr(lu), len(lp) - 1, aa._capi.iptr(lp), ptr(d[4]),
                                                len(up) - 1, aa._capi.iptr(up), ptr(d[5]), ptr(d[6]), ptr(t), ptr(x)))

        with torch.cuda.stream(s):
            work()
            s.synchronize()
            want = x.clone()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=s):
                work()
            for k in range(3):
                x.zero_()
                g.replay()
                s.synchronize()
                assert torch.equal(x, want)
                work()  # eager between replays
                s.synchronize()
                assert torch.equal(x, want)
