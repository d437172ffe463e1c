"""The dense diagonal factor of an SVD is built on the device: exactly the
singular values on the diagonal and zeros elsewhere, in every storage type
and for truncated, one-column and wide or tall matrices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float64", "float32", "complex128"])
@pytest.mark.parametrize("m,n,maxdim", [(1, 1, None), (7, 5, None), (5, 7, 3), (64, 65, 1),
                                        (130, 40, None)])
def test_diagonal_factor(dtype, m, n, maxdim):
    from itg import itensor, ops
    rng = np.random.default_rng(m + n)
    A = rng.standard_normal((m, n))
    if dtype == "complex128":
        A = A + 1j * rng.standard_normal((m, n))
    i, j = itensor.Index(m), itensor.Index(n)
    T = itensor.itensor(A, i, j, dtype=dtype).roc()
    U, S, V, spec = itensor.svd(T, [i], maxdim=maxdim)
    k = maxdim or min(m, n)
    assert [x.dim for x in S.inds] == [k, k]
    got = np.reshape(ops.to_host(S.data), (k, k), order="F")
    assert got.dtype == np.dtype(dtype)
    # eigs holds s^2: its root is s up to one rounding each way
    want = np.sqrt(spec.eigs)
    eps = 2.0 ** (-23 if dtype == "float32" else -51)
    assert (got[~np.eye(k, dtype=bool)] == 0).all()
    assert (abs(np.diag(got) - want) <= eps * want).all()
