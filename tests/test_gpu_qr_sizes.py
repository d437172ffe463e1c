"""QR at the edges of its panels: widths and heights one off 16, 512 rows (one
row a thread) and the row counts where a thread takes more rows and fewer
columns at a time (1024, 2048, 4096), wide matrices, zero and dependent
columns. Bounds (eps = 2^-52): Q^T Q - I, QR - A within 4 max(m, n) eps of a
backward stable Householder QR, R upper triangular with the signs of LAPACK's
(R from numpy agrees up to the conditioning, checked on a well conditioned
matrix)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


def _qr(A):
    from itg import ops
    m, n = A.shape
    r = min(m, n)
    Q, R = ops.qr(ops.to_device(np.ravel(A, order="F")), m, n)
    return (np.reshape(ops.to_host(Q), (m, r), order="F"),
            np.reshape(ops.to_host(R), (r, n), order="F"))


@pytest.mark.parametrize("kind", ["random", "dependent"])
@pytest.mark.parametrize("m,n", [(1, 1), (1, 9), (5, 3), (15, 17), (16, 16), (17, 15), (33, 31),
                                 (64, 200), (511, 47), (512, 48), (513, 49), (1025, 33),
                                 (1030, 20), (2049, 35), (2060, 40), (4097, 18), (4110, 37),
                                 (8192, 20), (8193, 20), (300, 300)])
def test_qr_sizes(m, n, kind):
    rng = np.random.default_rng(m + n)
    A = rng.standard_normal((m, n))
    if kind == "dependent":
        A[:, 1::3] = 0.0
        A[:, 2::5] = A[:, :1]
    Q, R = _qr(A)
    tol = 4 * max(m, n) * EPS
    assert abs(Q.T @ Q - np.eye(min(m, n))).max() <= tol
    assert abs(Q @ R - A).max() <= tol * max(1.0, np.linalg.norm(A, 2))
    assert (np.tril(R, -1) == 0.0).all()
    if kind == "random":
        # same sign convention (dlarfg: beta opposite to alpha) as LAPACK
        Rn = np.linalg.qr(A)[1]
        i = np.arange(min(m, n))
        live = abs(Rn[i, i]) > 1e-8 * abs(Rn[0, 0])
        assert (np.sign(R[i, i]) == np.sign(Rn[i, i]))[live].all()
