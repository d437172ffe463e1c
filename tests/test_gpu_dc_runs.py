"""Divide-and-conquer merges above 64 rows whose deflation rotates runs of
nearly equal eigenvalues into one: glued copies of one tridiagonal, multiplets
of every length, a spectrum that falls through the rounding level, and two
values only; sizes around the powers of two at which merges double.
Bounds: eigenvalues, U^T U - I and A U - U w within 8 n eps ||A||_2 of a
backward stable reduction (eps = 2^-52)."""
import numpy as np
import pytest

from test_gpu_eigh_resident import _check, _solve

pytestmark = pytest.mark.gpu


def _matrix(n, kind):
    rng = np.random.default_rng(n)
    if kind == "glued":
        i = np.arange(n)
        e = np.where(i[1:] % 21 == 0, 10.0 ** -(6 + i[1:] // 21 % 10), 1.0)
        return np.diag(abs(i % 21 - 10.0)) + np.diag(e, 1) + np.diag(e, -1)
    Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    if kind == "multiplets":
        w = np.sqrt(np.floor(np.sqrt(2.0 * np.arange(n)))) + 1e-15 * rng.standard_normal(n)
    elif kind == "falling":
        w = np.exp(-60.0 * np.arange(n) / n)
    else:
        w = np.where(np.arange(n) < n // 3, 1.0, 1e-3)
    A = (Q * w) @ Q.T
    return 0.5 * (A + A.T)


@pytest.mark.parametrize("kind", ["glued", "multiplets", "falling", "two"])
@pytest.mark.parametrize("n", [65, 127, 129, 200, 255, 257, 400, 513, 1000, 1300])
def test_runs(n, kind):
    A = _matrix(n, kind)
    _check(A, *_solve(A))
