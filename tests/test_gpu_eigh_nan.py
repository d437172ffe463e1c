"""Eigendecompositions of matrices that hold a NaN: every eigenvalue depends on
it (it sits in the first column, so the whole tridiagonal does), so none may
come out finite. A clean matrix of the same size in the next call is solved
within the usual bound (8 n eps ||A||)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(A):
    from itg import ops
    n = len(A)
    w, U, k, _, _ = ops.eigh_trunc(ops.to_device(np.ravel(A, order="F")), n)
    assert k == n
    return ops.to_host(w)


def _check(n):
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    A = A + A.T
    B = A.copy()
    B[1, 0] = B[0, 1] = np.nan
    print("n = %d with a NaN" % n, flush=True)
    assert not np.isfinite(_solve(B)).any()
    ref = np.linalg.eigvalsh(A)[::-1]
    assert abs(_solve(A) - ref).max() <= 8 * n * 2.0 ** -52 * abs(ref).max()


@pytest.mark.parametrize("n", [2, 3, 5, 16, 17, 33, 63, 64])
def test_one_leaf(n):
    _check(n)


@pytest.mark.parametrize("n", [65, 100, 128, 130, 193, 257, 300, 520, 1030])
def test_merges(n):
    _check(n)
