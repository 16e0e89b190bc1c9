"""The context's workspace of the ILU(0) entry points. A captured graph holds the caller's arrays only, so it replays rightly
after a larger system has gone through the context, and after the context is gone; the workspace grows under queued work; two
threads may call on one context."""
import ctypes
import threading

import numpy as np
import pytest

import alien_amd as aa

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from gpu_util import dev, empty  # noqa: E402
from test_gpu_ilu0_sync import CASES  # noqa: E402


def ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def system(case):
    """(run(context), lu, x): factorisation of the case's matrix and one solve, on arrays of their own."""
    ro, cols, vals = CASES[case]()
    n = len(ro) - 1
    dcol = aa.host_dcol(ro, cols)
    (lp, lr), (up, ur) = (aa.group_by_level(*aa.host_levels(ro, cols, dcol, u)) for u in (False, True))
    lp, up = (np.ascontiguousarray(a, np.int32) for a in (lp, up))
    A = [dev(ro), dev(cols), dev(dcol)]
    v, lr, ur, y = dev(vals), dev(lr.astype(np.int32)), dev(ur.astype(np.int32)), dev(np.random.default_rng(n).random(n))
    lu, t, x = empty(len(cols)), empty(n), empty(n)

    def run(c):
        L, a = aa.lib(), [ptr(q) for q in A]
        aa.check(L.alien_hip_copy_f64(c.h, len(cols), ptr(v), ptr(lu)))
        aa.check(L.alien_hip_ilu0_factor_f64(c.h, n, *a, ptr(lu), len(lp) - 1, aa._capi.iptr(lp), ptr(lr)))
        aa.check(L.alien_hip_ilu0_solve_f64(c.h, n, *a, ptr(lu), len(lp) - 1, aa._capi.iptr(lp), ptr(lr), len(up) - 1,
                                            aa._capi.iptr(up), ptr(ur), ptr(y), ptr(t), ptr(x)))

    return run, lu, x


def test_graph_outlives_the_workspace():
    print("case graph of a small system, eager larger one, context closed", flush=True)
    (small, lu, x), (large, _, xl) = system("fill"), system("wide")
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        with aa.Context(s.cuda_stream) as c:
            small(c)
            s.synchronize()
            want, want_lu = x.clone(), lu.clone()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=s):
                small(c)
            large(c)
            s.synchronize()
            want_large = xl.clone()
            for _ in range(3):
                x.zero_()
                g.replay()
                large(c)
                s.synchronize()
                assert torch.equal(x, want) and torch.equal(lu, want_lu) and torch.equal(xl, want_large)
        for _ in range(3):
            x.zero_()
            lu.zero_()
            g.replay()
            s.synchronize()
            assert torch.equal(x, want) and torch.equal(lu, want_lu)


def test_larger_system_while_the_stream_is_busy():
    """The workspace grows without a wait for the stream, under a smaller system's launches that are still to run."""
    print("case small and larger system behind 400 copies", flush=True)
    (small, lu, x), (large, _, xl) = system("fill"), system("wide")
    s = torch.cuda.Stream()
    with torch.cuda.stream(s), aa.Context(s.cuda_stream) as c:
        with aa.Context(s.cuda_stream) as other:
            small(other)
            large(other)
            s.synchronize()
            want, want_lu, want_large = x.clone(), lu.clone(), xl.clone()
        x.zero_()
        xl.zero_()
        a = torch.zeros(1 << 28, dtype=torch.float64, device="cuda")
        b = torch.empty_like(a)
        s.synchronize()
        for _ in range(400):  # 2 GiB each: 0.3 s in all
            b.copy_(a)
        copied = torch.cuda.Event()
        copied.record(s)
        small(c)
        large(c)
        assert not copied.query()
        s.synchronize()
        assert torch.equal(x, want) and torch.equal(lu, want_lu) and torch.equal(xl, want_large)


def test_two_threads_on_one_context():
    """Calls of two threads on one context: its stream runs them whole, one after the other."""
    print("case two threads, one context", flush=True)
    systems = [system("fill"), system("wide")]
    with aa.Context() as c:
        want = []
        for run, lu, x in systems:
            run(c)
            c.synchronize()
            want.append((lu.clone(), x.clone()))
        torch.cuda.synchronize()
        same = [True, True]

        def work(k):
            run, lu, x = systems[k]
            s = torch.cuda.Stream()
            for _ in range(20):
                run(c)
                c.synchronize()
                with torch.cuda.stream(s):
                    same[k] = same[k] and torch.equal(lu, want[k][0]) and torch.equal(x, want[k][1])
                s.synchronize()

        threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert same == [True, True]
