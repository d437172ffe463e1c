"""SVD of matrices whose squared column norms are subnormal: beyond what the
one-sided method resolves, so the call has to say that it did not converge, not
return without an error. At 2^-200 it still works (singular values within
8 max(m, n) eps ||A||)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _svd(A):
    from itg import ops
    m, n = A.shape
    return ops.to_host(ops.svd_trunc(ops.to_device(np.ravel(A, order="F")), m, n)[1])


@pytest.mark.parametrize("m,n", [(100, 80), (80, 130)])
def test_subnormal_squares(m, n):
    from itg import _lib
    A = np.random.default_rng(m).standard_normal((m, n))
    s = np.linalg.svd(A, compute_uv=False)
    got = np.ldexp(_svd(np.ldexp(A, -200)), 200)
    assert abs(got[:len(s)] - s).max() <= 8 * max(m, n) * 2.0 ** -52 * s[0]
    with pytest.raises(_lib.ITGError, match="did not converge"):
        _svd(np.ldexp(A, -520))
