"""FP64 products on both sides of the rules that choose between the library and
the contraction kernel (tiles for 0.4, 0.5 and 0.75 of the CUs, K of 800 and
1024, 2^29 multiply-adds), as itg_gemm and as a contraction with either order of
the output. Bound: (K + 4) eps |A| |B| + |C0| per entry, as for any sum of K
products (eps = 2^-52)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(256, 4096, 300), (700, 1024, 256), (750, 1030, 256), (704, 640, 799),
                                   (704, 640, 800), (640, 576, 800), (660, 700, 1023), (660, 700, 1024),
                                   (640, 640, 1500), (1024, 1024, 511), (1024, 1024, 512),
                                   (300, 300, 1200)])
@pytest.mark.parametrize("trans", ["NN", "NT", "TN"])
def test_routes(m, n, k, trans):
    from itg import ops
    rng = np.random.default_rng(m + n + k)
    A, B, C0 = rng.standard_normal((m, k)), rng.standard_normal((k, n)), rng.standard_normal((m, n))
    ref = A @ B
    tol = (k + 4) * 2.0 ** -52 * (abs(A) @ abs(B) + abs(C0))
    sA = A if trans[0] == "N" else A.T
    sB = B if trans[1] == "N" else B.T
    up = lambda x: ops.to_device(np.ravel(x, order="F"))
    dA, dB, C = up(sA), up(sB), up(C0)
    ops.gemm(trans[0], trans[1], m, n, k, 2.0, dA, sA.shape[0], dB, sB.shape[0], 0.5, C, m)
    got = np.reshape(ops.to_host(C), (m, n), order="F")
    assert (abs(got - (2.0 * ref + 0.5 * C0)) <= 3 * tol).all()
    la = [1, 2] if trans[0] == "N" else [2, 1]
    lb = [2, 3] if trans[1] == "N" else [3, 2]
    for lc, want in (([1, 3], ref), ([3, 1], ref.T)):
        C, dims = ops.contract(dA, sA.shape, la, dB, sB.shape, lb, lc)
        got = np.reshape(ops.to_host(C), dims, order="F")
        assert (abs(got - want) <= (tol if lc[0] == 1 else tol.T)).all()
