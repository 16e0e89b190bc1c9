"""Dot products finished in their own launch (up to 1024 workgroups of 1024 elements) against the two-launch form.

A stream capture takes the two-launch form: its replays have to give the eager call's bits, at the edges of a
workgroup, of a group of 32 workgroups and of the range. Against exactly rounded sums the error is at most that of
the longest chain of additions, 4 per lane, 6 + 4 per workgroup and 6 + 16 + n / 2^20 in the second stage: 48 rounding
errors of 2^-53 of the sum of magnitudes.
"""
import ctypes
import math
import threading

import numpy as np
import pytest
import torch

import alien_amd as aa

pytestmark = pytest.mark.gpu

GROUP = 32 * 1024
SIZES = [0, 1, 1023, 1024, 1025, GROUP, GROUP + 1, 1024 * 1024 - 1, 1024 * 1024, 1024 * 1024 + 1]


def ptr(t):
    return ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("kind", ["f64", "f32", "axpy"])
@pytest.mark.parametrize("n", SIZES)
def test_eager_equals_captured(n, kind):
    rng = np.random.default_rng(n)
    dt = np.float32 if kind == "f32" else np.float64
    hx, hy = (rng.standard_normal(max(n, 1)).astype(dt) for _ in range(2))
    stream = torch.cuda.Stream()
    with aa.Context(stream=stream.cuda_stream) as ctx, torch.cuda.stream(stream):
        L = aa.lib()
        x, y0 = torch.from_numpy(hx).cuda(), torch.from_numpy(hy).cuda()
        y, out = y0.clone(), torch.zeros(2, dtype=torch.float64, device="cuda")
        stream.synchronize()

        def call(slot):
            res = ctypes.c_void_p(out.data_ptr() + 8 * slot)
            if kind == "axpy":
                aa.check(L.alien_hip_axpy_dot_f64(ctx.h, n, ctypes.c_double(0.5), ptr(x), ptr(y), res))
            else:
                aa.check(getattr(L, "alien_hip_dot_" + kind)(ctx.h, n, ptr(x), ptr(y), res))

        call(0)
        stream.synchronize()
        eager = out[0].item()
        hy1 = y.cpu().numpy()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            call(1)
        for _ in range(3):
            y.copy_(y0)
            graph.replay()
            stream.synchronize()
            assert out[1].item() == eager
            y.copy_(y0)
            out[0] = -1
            call(0) # eager work between the replays
            stream.synchronize()
            assert out[0].item() == eager
    a, b = (hy1, hy1) if kind == "axpy" else (hx, hy)
    terms = (a[:n].astype(np.float64) * b[:n].astype(np.float64))
    assert abs(eager - math.fsum(terms)) <= 48 * 2.0**-53 * math.fsum(np.abs(terms))


def test_threads_read_back_their_own_scalars():
    """Solves whose every scalar the host reads, on three threads with a context each: the bits of one thread."""
    ro, cols, vals = aa.gen_csr(aa.GEN_POISSON7, 17, 13, 11)
    rhs = [aa.uniform01(k, len(ro) - 1) for k in range(3)]

    def solve(k):
        with aa.Context() as c:
            x, r = aa.solve_csr(c, ro, cols, vals, rhs[k], solver=aa.CG, precond=aa.PREC_DIAG, mode=aa.MODE_REFERENCE,
                                tol=1e-10, max_iter=1000)
            return x, r["iterations"]

    want = [solve(k) for k in range(3)]
    got = [None] * 3

    def work(k):
        for _ in range(3):
            got[k] = solve(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for (x, it), (gx, git) in zip(want, got):
        assert it == git and np.array_equal(x, gx)
