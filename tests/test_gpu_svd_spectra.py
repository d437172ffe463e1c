"""SVD over the spectra that decide how the columns are made orthogonal:
flat, decaying past the square root of the precision (the first eigenbasis
resolves the leading columns only), clustered, exactly degenerate and rank
deficient; square, tall and wide, at the smallest preconditioned size and one
off the tile sizes.

Bounds (eps = 2^-52): singular values and U S V^T within 4 (m + n) eps s_1 of
a backward stable computation; V orthogonal to the same multiple; U's columns
orthogonal to the convergence cosine 4 eps sqrt(max(m, n)) plus the rounding
of forming and dividing them, for values above eps times the Frobenius norm
(below it a column is rounding noise). U and V change places if m < n.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


def _spectrum(kind, r):
    i = np.arange(r)
    if kind == "flat":
        return 1.0 - 0.5 * i / r
    if kind == "decay":
        return np.exp(-34.0 * i / r)
    if kind == "cluster":
        return np.exp(-3.0 * (i // 9)) * (1.0 + 1e-13 * (i % 9)) + 1e-14
    if kind == "degenerate":
        return np.where(i < r // 2, 1.0, 1e-7)
    s = np.exp(-5.0 * i / r)
    s[r // 3:] = 0.0
    return s     # rank deficient


@pytest.mark.parametrize("kind", ["flat", "decay", "cluster", "degenerate", "deficient"])
@pytest.mark.parametrize("m,n", [(64, 64), (65, 127), (300, 257), (129, 700), (513, 513)])
def test_svd_spectra(kind, m, n):
    from itg import ops
    r = min(m, n)
    rng = np.random.default_rng(m + n)
    Q1 = np.linalg.qr(rng.standard_normal((m, r)))[0]
    Q2 = np.linalg.qr(rng.standard_normal((n, r)))[0]
    A = (Q1 * _spectrum(kind, r)) @ Q2.T
    U, S, V, k, _, _ = ops.svd_trunc(ops.to_device(np.ravel(A, order="F")), m, n, cutoff=0.0)
    s = ops.to_host(S)
    ref = np.linalg.svd(A, compute_uv=False)
    tol = 4 * (m + n) * EPS
    assert abs(s - ref).max() <= tol * ref[0]
    assert (np.diff(s) <= 0).all()
    U = np.reshape(ops.to_host(U)[: m * k], (m, k), order="F")
    V = np.reshape(ops.to_host(V)[: n * k], (n, k), order="F")
    assert abs((U * s[:k]) @ V.T - A).max() <= tol * ref[0]
    # the factor of the shorter side is a product of rotations; the other
    # one is the columns divided by their norms
    if m < n:
        U, V = V, U
    assert abs(V.T @ V - np.eye(k)).max() <= tol
    live = s[:k] > 2 * EPS * np.linalg.norm(A)
    U = U[:, live]
    cos = 4 * EPS * np.sqrt(max(m, n)) + 4 * np.sqrt(max(m, n)) * EPS
    assert abs(U.T @ U - np.eye(U.shape[1])).max() <= cos


def test_svd_random_square():
    """A dense random matrix: flat spectrum down to a condition of ~n."""
    from itg import ops
    n = 600
    A = np.random.default_rng(5).standard_normal((n, n))
    U, S, V, k, _, _ = ops.svd_trunc(ops.to_device(np.ravel(A, order="F")), n, n, cutoff=0.0)
    s, ref = ops.to_host(S), np.linalg.svd(A, compute_uv=False)
    assert k == n and abs(s - ref).max() <= 8 * n * EPS * ref[0]
    U = np.reshape(ops.to_host(U), (n, n), order="F")
    V = np.reshape(ops.to_host(V), (n, n), order="F")
    assert abs((U * s) @ V.T - A).max() <= 8 * n * EPS * ref[0]
    assert abs(U.T @ U - np.eye(n)).max() <= 8 * np.sqrt(n) * EPS
