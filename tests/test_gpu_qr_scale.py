"""QR of matrices so small that the squares of their entries underflow: bounds
relative to the matrix itself, Q^T Q - I within 4 max(m, n) eps (eps = 2^-52)
and QR - A within that of ||A||. Scales 2^-k are exact, so the check is made
on Q, R 2^k and the matrix before scaling. `column`: a matrix of order one with
some columns that small, which count as zero beside the others."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


def _check(A, k):
    """QR of 2^-k A, checked against A"""
    from itg import ops
    m, n = A.shape
    r = min(m, n)
    Q, R = ops.qr(ops.to_device(np.ravel(np.ldexp(A, -k), order="F")), m, n)
    Q = np.reshape(ops.to_host(Q), (m, r), order="F")
    R = np.ldexp(np.reshape(ops.to_host(R), (r, n), order="F"), k)
    tol = 4 * max(m, n) * EPS
    assert abs(Q.T @ Q - np.eye(r)).max() <= tol
    assert abs(Q @ R - A).max() <= tol * np.linalg.norm(A, 2)


SIZES = [(7, 5), (40, 33), (33, 60), (600, 40), (1500, 70), (3000, 40), (5000, 20), (8200, 20)]


@pytest.mark.parametrize("m,n", SIZES)
@pytest.mark.parametrize("k", [500, 512, 530, 600, 900])
def test_scaled(m, n, k):
    _check(np.random.default_rng(m + k).standard_normal((m, n)), k)


@pytest.mark.parametrize("m,n", SIZES)
def test_small_columns(m, n):
    rng = np.random.default_rng(m)
    A = rng.standard_normal((m, n))
    A[:, ::3] = np.ldexp(A[:, ::3], -560)
    A[:, 1::5] = 0.0
    _check(A, 0)
