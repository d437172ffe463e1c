"""Eigendecompositions at the sizes where the tridiagonalisation changes
hands (the one-workgroup tail of 64, 128 and 192 rows, a short first panel
before it, whole panels) and where the divide and conquer does (leaves of 64
rows, a short last leaf). Full-rank, rank-deficient and diagonal matrices,
multiplets, and glued copies of one tridiagonal (runs of nearly equal
eigenvalues at every merge).
Bounds: eigenvalues, U^T U - I and A U - U w within 8 n eps ||A||_2 of a
backward stable reduction (eps = 2^-52)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


@pytest.mark.parametrize("kind", ["full", "deficient", "diagonal", "multiplets",
                                  "glued"])
@pytest.mark.parametrize("n", [2, 3, 17, 31, 32, 33, 63, 64, 65, 100, 127, 128, 129, 160, 191, 192,
                               193, 200, 223, 224, 225, 257, 290])
def test_eigh_sizes(n, kind):
    from itg import ops
    rng = np.random.default_rng(n)
    if kind == "full":
        A = rng.standard_normal((n, n))
        A = A + A.T
    elif kind == "deficient":
        B = rng.standard_normal((n, max(1, n // 3)))
        A = B @ B.T
    elif kind == "diagonal":
        A = np.diag(rng.standard_normal(n))
    elif kind == "multiplets":
        Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
        A = (Q * (1.0 + np.arange(n) // 5 + 1e-15 * rng.standard_normal(n))) @ Q.T
    else:
        i = np.arange(n)
        e = np.where(i[1:] % 21 == 0, 10.0 ** -(6 + i[1:] // 21 % 10), 1.0)
        A = np.diag(abs(i % 21 - 10.0)) + np.diag(e, 1) + np.diag(e, -1)
    A = 0.5 * (A + A.T)
    w, U, k, _, _ = ops.eigh_trunc(ops.to_device(np.ravel(A, order="F")), n)
    w = ops.to_host(w)
    U = np.reshape(ops.to_host(U), (n, n), order="F")
    ref = np.linalg.eigvalsh(A)[::-1]
    tol = 8 * n * EPS * abs(ref).max()
    assert k == n
    assert abs(w - ref).max() <= tol
    assert abs(U.T @ U - np.eye(n)).max() <= 8 * n * EPS
    assert abs(A @ U - U * w).max() <= tol
