"""GRAPH-mode BiCGStab that its first block solves (the capture beside it is broken off) or does not: FUSED mode's iterates, bit
for bit, and the same again on the same context."""
import numpy as np
import pytest

import alien_amd as aa
import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precond", [aa.PREC_DIAG, aa.PREC_ILU0, aa.PREC_CHEB])
@pytest.mark.parametrize("edge", [6, 40])
def test_first_block(ctx, edge, precond):
    ro, cols, vals = aa.gen_csr(aa.GEN_POISSON7, edge)
    x = aa.uniform01(7, len(ro) - 1)
    b = orc.spmv(ro, cols, vals, x)
    for off, tol, first in ((1e-6, 1e-5, True), (1.0, 1e-10, False)):  # off: the first guess's relative error
        x0 = x * (1.0 + off * np.cos(np.arange(len(x))))
        for mode in (aa.MODE_GRAPH, aa.MODE_MIXED):
            kw = dict(x0=x0, solver=aa.BICGS, precond=precond, tol=tol, max_iter=200, poll_every=8)
            print("case", edge, precond, off, mode, flush=True)
            got = [aa.solve_csr(ctx, ro, cols, vals, b, mode=mode, **kw) for _ in range(2)]
            for gx, r in got:
                assert r["status"] == 1 and (r["iterations"] <= 1) == first
                np.testing.assert_array_equal(gx, got[0][0])
            if mode == aa.MODE_GRAPH:
                fx, fr = aa.solve_csr(ctx, ro, cols, vals, b, mode=aa.MODE_FUSED, **kw)
                np.testing.assert_array_equal(got[0][0], fx)
                assert got[0][1]["iterations"] == fr["iterations"]
