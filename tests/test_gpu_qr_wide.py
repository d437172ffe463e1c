"""QR of wide matrices whose last panel of 16 columns is partial: the row count
is no multiple of 16 and there are columns to its right, fewer and more than
the panel's block of 16 has left. Bounds (eps = 2^-52) as for any backward
stable Householder QR: Q^T Q - I and QR - A within 4 max(m, n) eps. Then a gauge
move that meets such matrices: a sum of spin-1 states, whose third site from
the end has 27 rows and more columns."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


@pytest.mark.parametrize("m,n", [(17, 18), (20, 21), (20, 40), (20, 60), (31, 33), (33, 50), (33, 60),
                                 (40, 100), (100, 130), (347, 706), (1000, 1500), (1030, 1100),
                                 (2060, 2100)])
def test_partial_last_panel(m, n):
    from itg import ops
    A = np.random.default_rng(m + n).standard_normal((m, n))
    Q, R = ops.qr(ops.to_device(np.ravel(A, order="F")), m, n)
    Q = np.reshape(ops.to_host(Q), (m, m), order="F")
    R = np.reshape(ops.to_host(R), (m, n), order="F")
    tol = 4 * max(m, n) * EPS
    assert abs(Q.T @ Q - np.eye(m)).max() <= tol
    assert abs(Q @ R - A).max() <= tol * np.linalg.norm(A, 2)
    assert (np.tril(R, -1) == 0.0).all()


def test_orthogonalize_sum_of_spin1_states():
    from itg import mpo
    from itg.itensor import Index
    sites = [Index(3) for _ in range(8)]
    a, b = mpo.random_mps(sites, 20, seed=1), mpo.random_mps(sites, 13, seed=2)
    s = mpo.add(a, b)
    want = mpo.inner(a, a) + 2 * mpo.inner(a, b) + mpo.inner(b, b)
    mpo.orthogonalize(s, 0)
    # a few hundred roundings of values of order one
    assert abs(mpo.inner(s, s) - want) <= 1e-12 * abs(want)
    assert abs(mpo.inner(a, s) - mpo.inner(a, a) - mpo.inner(a, b)) <= 1e-12 * abs(want)
