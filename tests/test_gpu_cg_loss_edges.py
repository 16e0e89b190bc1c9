"""k-step CG loss of the learned preconditioner: sizes at the edges of its reductions and row batches.

A dot product's partials (one per 256 rows) are summed by their consumers up to 64 of them, by a finalize launch
beyond; rows are read in batches of 8 (4 in the reverse pass); weight gradients are formed per 256 rows, 8 workgroups
(2 from 256 row blocks on) sharing each. Oracle and bounds are those of the CG loss on a 10^3 grid (FP32 vectors
and FP64 dots against the FP64 oracle with the same bf16 rounding): 1e-4 on the loss, 2e-3 on the gradient.
"""
import numpy as np
import pytest

import alien_amd as aa
from oracle import gnn_oracle as go

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with aa.Context() as c:
        yield c


def say(*a):
    print(*a, flush=True)


def grid(*dims):
    return aa.gen_csr(aa.GEN_LOGNORMAL7, *dims, params=[1.0, 1.0, 1.0, 1.0], seed=3)


def wide_rows(n, half, seed):
    """Symmetric, diagonally dominant, up to 2 half + 1 entries a row (9 or more: past one batch)."""
    rng = np.random.default_rng(seed)
    a = np.zeros((n, n))
    for i in range(n):
        j = rng.integers(0, n, half)
        a[i, j] -= rng.uniform(0.1, 1.0, half)
    a = np.tril(a, -1)
    a = a + a.T
    a[np.arange(n), np.arange(n)] = 1.1 * np.abs(a).sum(1) + 0.5
    ro = np.concatenate([[0], np.cumsum((a != 0).sum(1))]).astype(np.int32)
    cols = np.nonzero(a)[1].astype(np.int32)
    return ro, cols, a[a != 0]


SYSTEMS = {
    "n2": lambda: grid(2, 1, 1),
    "n255": lambda: grid(17, 15, 1),
    "n257": lambda: grid(257, 1, 1),
    "n2049": lambda: grid(683, 3, 1),     # 9 row blocks: a second group of 8
    "n16384": lambda: grid(64, 16, 16),   # 64 partials
    "n16640": lambda: grid(65, 16, 16),   # 65
    "n65536": lambda: grid(64, 32, 32),   # 256 row blocks: weight gradients in groups of 32 columns
    "wide": lambda: wide_rows(300, 9, 1),
}


@pytest.mark.parametrize("k", [1, 4])
@pytest.mark.parametrize("which", list(SYSTEMS))
def test_cg_loss_at_edges_matches_oracle(ctx, which, k):
    ro, cols, vals = SYSTEMS[which]()
    n = len(ro) - 1
    k = min(k, n // 2)  # CG ends in n steps: the loss is log(rounding) from there on
    th = go.init_params(0)
    th = (th + 0.05 * np.random.default_rng(6).standard_normal(len(th))).astype(np.float32)
    V = np.random.default_rng(12).choice([-1.0, 1.0], size=(n, 4)).astype(np.float32)
    say("cg loss", which, "n", n, "k", k)
    L, (lc, lp), grad = aa.gnn_loss_grad(ctx, ro, cols, vals, th, V, beta=0.1, cg_steps=k)
    again = aa.gnn_loss_grad(ctx, ro, cols, vals, th, V, beta=0.1, cg_steps=k)
    assert again[0] == L and np.array_equal(again[2], grad)
    g = go.Graph(ro, cols, vals)
    Lo, go_grad, Gh = go.cg_total_loss_and_grad(g, th, V.astype(np.float64), k=k, beta=0.1, bf=True)
    assert L == pytest.approx(Lo, rel=1e-4, abs=1e-5)
    rel = np.linalg.norm(grad - go_grad) / np.linalg.norm(go_grad)
    say("  grad rel err", rel)
    assert rel < 2e-3
