"""Eigendecompositions on a device that other work shares.

A wait that runs out
twice in a row (forced by a limit of zero) makes the context's next two
calls go without the resident reduction, the third tries it again; seen from
the launches of the chip-wide kernel that does its columns instead.

A context whose stream has a long (one-workgroup) kernel queued before its
decomposition does not keep another context's from running meanwhile."""
import ctypes
import threading
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


class Solver:
    """eigendecompositions on a context of its own (made in the thread that
    uses it: a context makes its stream torch's current one there)"""

    def __init__(self, n):
        from itg import _lib
        self.lib, self.n = _lib, n
        self.c = _lib.Context(0)
        A = np.random.default_rng(n).standard_normal((n, n))
        self.A = A + A.T
        self.ref = np.linalg.eigvalsh(self.A)[::-1]

    def load(self):
        import torch
        n = self.n
        self.dA = torch.from_numpy(self.A.ravel().copy()).to("cuda:0")
        self.w = torch.empty(n, device="cuda:0", dtype=torch.float64)
        self.U = torch.empty(n * n, device="cuda:0", dtype=torch.float64)
        torch.cuda.current_stream().synchronize()

    def run(self):
        lib, n = self.lib, self.n
        k, te, dc = ctypes.c_int64(), ctypes.c_double(), ctypes.c_double()
        self.c.check(lib.lib().itg_eigh_trunc(self.c.ptr, lib.F64, n, lib.ptr(self.dA),
                                              lib.ptr(self.w), lib.ptr(self.U), 0, -1.0, 0, 1,
                                              ctypes.byref(k), ctypes.byref(te), ctypes.byref(dc)))
        self.c.sync()

    def solve(self):
        self.load()
        self.run()
        tol = 8 * self.n * EPS * abs(self.ref).max()
        assert abs(self.w.cpu().numpy() - self.ref).max() <= tol

    def columns(self):
        """columns that one decomposition leaves to the chip-wide kernel"""
        self.c.timing([self.lib.K_TRD_SYMV])
        self.solve()
        got = self.c.timing_report(self.lib.K_TRD_SYMV)["launches"]
        self.c.timing()
        return got


def _in_thread(f):
    out = []

    def go():
        try:
            out.append(f())
        except BaseException as e:
            out.append(e)
    t = threading.Thread(target=go)
    t.start()
    t.join()
    if isinstance(out[0], BaseException):
        raise out[0]
    return out[0]


def test_run_outs_are_remembered(monkeypatch):
    from itg import _lib
    _lib.ctx()

    def work():
        s = Solver(260)
        before = [s.columns()]
        monkeypatch.setenv("ITG_TRD_WAIT_MS", "0")
        outs = [s.columns() for _ in range(2)]
        monkeypatch.delenv("ITG_TRD_WAIT_MS")
        after = [s.columns() for _ in range(4)]
        return before, outs, after

    before, outs, after = _in_thread(work)
    m = outs[0]
    assert m > 0 and before == [0] and outs == [m, m]
    assert after == [m, m, 0, 0]


def test_other_contexts_queue():
    import torch
    from itg import _lib
    _lib.ctx()
    torch.cuda._sleep(1000)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    torch.cuda._sleep(5000000)
    torch.cuda.synchronize()
    per_s = int(5000000 / (time.perf_counter() - t0))
    queued, times = threading.Event(), {}

    def independent(s, sleeper):
        # streams share a few hardware queues: one that runs beside `sleeper`
        for _ in range(8):
            torch.cuda.synchronize()
            with torch.cuda.stream(sleeper):
                torch.cuda._sleep(per_s // 10)
            st = torch.cuda.Stream()
            torch.cuda.set_stream(st)
            s.c.bind_stream(st.cuda_stream)
            x = torch.ones(8, device="cuda:0")
            st.synchronize()
            if not sleeper.query():
                return True
        return False

    def busy(s):
        s.load()
        torch.cuda._sleep(2 * per_s)
        queued.set()
        s.run()
        times["busy"] = time.perf_counter()

    def both():
        a = Solver(300)
        a.solve()
        stream_a = torch.cuda.current_stream()

        def other():
            b = Solver(300)
            if not independent(b, stream_a):
                return False
            b.solve()
            b.load()

            def run_a():
                torch.cuda.set_stream(stream_a)
                busy(a)
            t = threading.Thread(target=run_a)
            t.start()
            queued.wait()
            time.sleep(0.2)   # the other thread is at its reduction
            b.run()
            times["other"] = time.perf_counter()
            t.join()
            return True
        return _in_thread(other)

    if not _in_thread(both):
        pytest.skip("no two streams on hardware queues of their own")
    # the other one took milliseconds of the queued two seconds (less if the
    # clock rose since they were counted out)
    assert times["other"] < times["busy"] - 0.25
