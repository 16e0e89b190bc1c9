"""ILU(0) of full 7-point matrices in pencils of grid lines: the solves are the launch-per-level ones bit for bit (the
same factor and sweeps, so no tolerance), at the edges of the pencils and of the rule that picks them."""
import numpy as np
import pytest

import alien_amd as aa
import oracle as orc

pytestmark = pytest.mark.gpu


def matrix(case, dims):
    """Nonsymmetric 7-point matrix with random values, diagonally dominant; or one that is almost such a matrix."""
    ro, cols, vals = aa.gen_csr(aa.GEN_POISSON7, *dims)
    rng = np.random.default_rng(sum(dims))
    vals = np.where(vals < 0, -rng.random(len(vals)) - 0.1, 7.7)
    n, nx = len(ro) - 1, dims[0]
    row = np.repeat(np.arange(n), np.diff(ro))
    if case == "entry missing":  # the entry count is the full one's: the last row's first entry, moved to a wrap below
        case, drop = "wrap", ro[n - 1]
    else:
        drop = np.flatnonzero((row == n // 2) & (cols > row))[-1]
    if case == "wrap":  # row (0, 1, 0) also reads the end of the line before it
        keep = np.arange(len(cols)) != drop
        row, cols, vals = np.append(row[keep], nx), np.append(cols[keep], nx - 1), np.append(vals[keep], -0.25)
        o = np.lexsort((cols, row))
        row, cols, vals = row[o], cols[o].astype(np.int32), vals[o]
        ro = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))]).astype(np.int32)
    return ro, cols, vals


CASES = [("full", d) for d in [(2, 2, 2), (8, 8, 8), (9, 7, 17), (3, 16, 9), (64, 8, 24), (50, 33, 40), (130, 17, 15)]]
CASES += [("wrap", (9, 10, 11)), ("entry missing", (9, 10, 11)), ("full", (2, 70, 90))]  # the last: too thin


@pytest.mark.parametrize("case,dims", CASES, ids=["%s %dx%dx%d" % ((c,) + d) for c, d in CASES])
def test_pencil_ilu0_equals_level_launches(monkeypatch, case, dims):
    ro, cols, vals = matrix(case, dims)
    b = orc.spmv(ro, cols, vals, aa.uniform01(3, len(ro) - 1))
    defaults = {"ALIEN_HIP_ILU_SYNC_FREE": "1", "ALIEN_HIP_ILU_SF_SPINS": "65536"}
    envs = {"levels": {"ALIEN_HIP_ILU_SYNC_FREE": "0"}, "pencils": {}, "every wait given up": {"ALIEN_HIP_ILU_SF_SPINS": "0"}}
    kw = dict(precond=aa.PREC_ILU0, ilu_schedule=0, tol=1e-30, max_iter=3, poll_every=1)
    runs = {}
    try:
        for name, env in envs.items():
            for k, v in defaults.items():
                monkeypatch.setenv(k, env.get(k, v))
            c = aa.Context()  # the variables are read when a context is created
            try:
                for mode in (aa.MODE_REFERENCE, aa.MODE_GRAPH, aa.MODE_MIXED):
                    print("case pencil", case, dims, name, mode, flush=True)
                    runs[name, mode] = aa.solve_csr(c, ro, cols, vals, b, solver=aa.BICGS, mode=mode, **kw)[0]
                # the factor in CSR order: FILU0's exact factor
                runs[name, "filu0"] = aa.solve_csr(c, ro, cols, vals, b, solver=aa.BICGS, mode=aa.MODE_FUSED,
                                                   **dict(kw, precond=aa.PREC_FILU0, filu_solver_niter=2))[0]
            finally:
                c.close()
    finally:
        for k, v in defaults.items():
            monkeypatch.setenv(k, v)
        aa.Context().close()
    for (name, mode), x in runs.items():
        np.testing.assert_array_equal(x, runs["levels", mode], err_msg="%s %s" % (name, mode))
