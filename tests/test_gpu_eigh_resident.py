"""Eigendecompositions whose tridiagonalisation runs in workgroups that keep
the matrix in registers: sizes around its first one, around a workgroup's 16
(12, 14) rows and around each 512 columns at which one kernel hands over to the next;
the start over without it when a wait runs out; several threads at once.
Bounds: eigenvalues, U^T U - I and A U - U w within 8 n eps ||A||_2 of a
backward stable reduction (eps = 2^-52)."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


def _matrix(n, kind):
    rng = np.random.default_rng(n)
    if kind == "full":
        A = rng.standard_normal((n, n))
    elif kind == "deficient":
        B = rng.standard_normal((n, max(1, n // 3)))
        A = B @ B.T
    elif kind == "arrow":   # zero columns below the subdiagonal but the first
        A = np.diag(rng.standard_normal(n))
        A[:, 0] = rng.standard_normal(n)
    else:
        A = np.exp(-rng.uniform(0, 30, n))[:, None] * rng.standard_normal((n, n))
        A = A @ A.T
    return A + A.T


def _solve(A):
    from itg import ops
    n = len(A)
    w, U, k, _, _ = ops.eigh_trunc(ops.to_device(np.ravel(A, order="F")), n)
    assert k == n
    return ops.to_host(w), np.reshape(ops.to_host(U), (n, n), order="F")


def _check(A, w, U):
    n = len(A)
    ref = np.linalg.eigvalsh(A)[::-1]
    tol = 8 * n * EPS * abs(ref).max()
    assert abs(w - ref).max() <= tol
    assert abs(U.T @ U - np.eye(n)).max() <= 8 * n * EPS
    assert abs(A @ U - U * w).max() <= tol


@pytest.mark.parametrize("kind", ["full", "deficient", "arrow", "graded"])
@pytest.mark.parametrize("n", [199, 200, 201, 207, 208, 209, 255, 256, 300, 511, 512, 513, 529, 700,
                               1023, 1024, 1025])
def test_sizes(n, kind):
    A = _matrix(n, kind)
    _check(A, *_solve(A))


@pytest.mark.parametrize("n", [1537, 2049, 2560, 2561, 2569, 2580, 3072, 3073, 3300,
                               3584, 3585, 3650])
def test_large(n):
    A = _matrix(n, "graded" if n == 2560 else "full")
    _check(A, *_solve(A))


@pytest.mark.parametrize("n", [300, 1100])
def test_wait_runs_out(n, monkeypatch):
    monkeypatch.setenv("ITG_TRD_WAIT_MS", "0")
    A = _matrix(n, "full")
    _check(A, *_solve(A))


def test_threads():
    """four host threads, each with a context and a stream of its own, reduce
    at the same time (one resident reduction runs at a time on a device)"""
    import ctypes

    import torch
    from itg import _lib
    _lib.ctx()
    As = [_matrix(n, "full") for n in (300, 520, 1030, 400)]
    out = [None] * len(As)

    def work(i):
        c = _lib.Context(0)
        n = len(As[i])
        for _ in range(3):
            A = torch.from_numpy(As[i].ravel().copy()).to("cuda:0")
            w = torch.empty(n, device="cuda:0", dtype=torch.float64)
            U = torch.empty(n * n, device="cuda:0", dtype=torch.float64)
            k, te, dc = ctypes.c_int64(), ctypes.c_double(), ctypes.c_double()
            c.check(_lib.lib().itg_eigh_trunc(c.ptr, _lib.F64, n, _lib.ptr(A), _lib.ptr(w),
                                              _lib.ptr(U), 0, -1.0, 0, 1, ctypes.byref(k),
                                              ctypes.byref(te), ctypes.byref(dc)))
            c.sync()
            out[i] = (w.cpu().numpy(), U.cpu().numpy().reshape(n, n, order="F"))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(len(As))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for A, o in zip(As, out):
        _check(A, *o)
