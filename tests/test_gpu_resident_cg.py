"""CG whose iterations run in one launch with the system in registers, against the same solve from launches, bit for
bit: at the edges of its forms (one workgroup, one and two rows per lane, and past the last)."""
import threading

import numpy as np
import pytest

import alien_amd as aa
import oracle as orc

pytestmark = pytest.mark.gpu


def matrix(n, offsets=(-1, 1, -37, 37)):
    """5-point-like SPD matrix of any size: the offsets that are in range, -1 each, and a diagonal of 5 (eigenvalues in
    [1, 9]). Only dependence on n is through the ends: odd sizes, last bundles of any length."""
    d = sorted({o for o in offsets if abs(o) < n} | {0})
    row = np.repeat(np.arange(n), len(d))
    col = row + np.tile(d, n)
    keep = (col >= 0) & (col < n)
    row, col = row[keep], col[keep].astype(np.int32)
    ro = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))]).astype(np.int32)
    return ro, col, np.where(row == col, 5.0, -1.0)


@pytest.fixture(scope="module")
def contexts():
    import os
    made = {}
    for name, env in (("launches", {"ALIEN_HIP_CG_RESIDENT": "0"}), ("resident", {}),
                      ("gives up", {"ALIEN_HIP_CG_RESIDENT_SPINS": "0"})):
        os.environ.update(env)  # read when a context is created
        made[name] = aa.Context()
        for k in env:
            del os.environ[k]
    yield made
    for c in made.values():
        c.close()


SIZES = [1, 2, 63, 65, 255, 257, 1023, 1025, 2048, 2049, 4097, 32769, 65600, 131073, 262144, 262145, 524288, 524289]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("precond", ["diag", "cheb"])
def test_resident_cg(contexts, n, precond):
    ro, cols, vals = matrix(n)
    b = np.random.default_rng(n).standard_normal(n)
    kw = dict(solver=aa.CG, precond=aa.PREC_DIAG if precond == "diag" else aa.PREC_CHEB, poll_every=4)
    for mode in (aa.MODE_FUSED, aa.MODE_GRAPH, aa.MODE_MIXED):
        got = {c: aa.solve_csr(contexts[c], ro, cols, vals, b, mode=mode, tol=1e-11, max_iter=500, **kw)
               for c in ("launches", "resident", "gives up")}
        x, r = got["launches"]
        print("case resident", n, precond, mode, r["iterations"], got["gives up"][1]["iterations"], flush=True)
        assert r["status"] == 1
        np.testing.assert_array_equal(got["resident"][0], x)
        assert all(got["resident"][1][k] == r[k] for k in ("iterations", "status", "error", "outer", "value"))
        # begun again after the wait given up: another recurrence to the same residual; the smallest
        # eigenvalue is 1 or more, so either error is at most its residual
        assert got["gives up"][1]["status"] == 1
        assert np.linalg.norm(got["gives up"][0] - x) <= 2.1e-11 * np.linalg.norm(b)


def test_max_iter_and_breakdown(contexts):
    ro, cols, vals = matrix(5000)
    b = np.ones(5000)
    for k in (1, 2, 7):
        r = aa.solve_csr(contexts["resident"], ro, cols, vals, b, solver=aa.CG, precond=aa.PREC_DIAG, mode=aa.MODE_GRAPH,
                         tol=1e-30, max_iter=k)[1]
        assert (r["iterations"], r["status"], r["error"]) == (k, 0, 0)
    # p.q = 0 in the third step: a zero residual in exact arithmetic, the identity's solve continued past its end
    ro, cols = np.arange(3000 + 1, dtype=np.int32), np.arange(3000, dtype=np.int32)
    got = {name: aa.solve_csr(c, ro, cols, np.full(3000, 2.0), np.ones(3000), solver=aa.CG, precond=aa.PREC_DIAG,
                              mode=aa.MODE_GRAPH, tol=0.0, max_iter=9) for name, c in contexts.items() if name != "gives up"}
    print({k: v[1] for k, v in got.items()}, flush=True)
    for key in ("iterations", "status", "error"):
        assert got["resident"][1][key] == got["launches"][1][key]
    np.testing.assert_array_equal(got["resident"][0], got["launches"][0])


def test_not_finite(contexts):
    ro, cols, vals = matrix(70000)
    b = np.ones(70000)
    b[12345] = np.inf
    for mode in (aa.MODE_GRAPH, aa.MODE_MIXED):
        got = [aa.solve_csr(contexts[c], ro, cols, vals, b, solver=aa.CG, precond=aa.PREC_DIAG, mode=mode, tol=1e-8,
                            max_iter=20)[1] for c in ("launches", "resident")]
        assert got[0]["status"] == got[1]["status"] and got[0]["iterations"] == got[1]["iterations"]


def test_two_threads(contexts):
    """Solves of two contexts at once: each takes its turn on the device."""
    ro, cols, vals = aa.gen_csr(aa.GEN_POISSON7, 56)
    b = orc.spmv(ro, cols, vals, aa.uniform01(3, len(ro) - 1))
    kw = dict(solver=aa.CG, precond=aa.PREC_DIAG, mode=aa.MODE_GRAPH, tol=1e-10, max_iter=1000)
    alone = aa.solve_csr(contexts["resident"], ro, cols, vals, b, **kw)[0]
    out = {}

    def work(k):
        with aa.Context() as c:
            out[k] = [aa.solve_csr(c, ro, cols, vals, b, **kw)[0] for _ in range(5)]

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(3):
        for x in out[k]:
            np.testing.assert_array_equal(x, alone)
