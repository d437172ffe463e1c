"""A matrix with itself, by product and by contraction: exactly symmetric, and
within the a-priori bound |C - A A^T| <= (K + 4) u |A| |A|^T of a K-term sum,
below and above the sizes from which half of it is computed and mirrored
(256 rows; as many 64 x 64 tiles of the band as CUs: 1345 rows on 256), at tile
edges, with a leading dimension, and scaled."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(got, A, alpha, dtype):
    A = A.astype(np.float64)
    u = 2.0 ** (-53 if dtype == "float64" else -24)
    ref = alpha * (A @ A.T)
    bound = (A.shape[1] + 4) * u * abs(alpha) * (abs(A) @ abs(A).T)
    assert (got == got.T).all()
    assert (abs(got - ref) <= bound).all(), (abs(got - ref) / bound).max()


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("n,k", [(255, 40), (256, 1), (257, 700), (640, 130), (1344, 33),
                                 (1345, 33), (1408, 129), (1500, 16), (2049, 47)])
@pytest.mark.parametrize("ta,tb", ["NT", "TN"])
def test_gemm_with_itself(dtype, n, k, ta, tb):
    from itg import ops
    rng = np.random.default_rng(n + k)
    A = rng.standard_normal((n, k)).astype(dtype)
    rows = n if ta == "N" else k
    X = np.zeros((rows + 3, k if ta == "N" else n), dtype=dtype)   # ld = rows + 3
    X[:rows] = A if ta == "N" else A.T
    Xd = ops.to_device(np.ravel(X, order="F"), dtype)
    C = ops.empty(n * n, dtype)
    ops.gemm(ta, tb, n, n, k, -0.5, Xd, rows + 3, Xd, rows + 3, 0.0, C, n)
    _check(np.reshape(ops.to_host(C), (n, n), order="F").astype(np.float64), A, -0.5, dtype)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("dims,keep,order", [((16, 16, 25), (0, 1), 0), ((700, 2, 31), (0, 1), 0),
                                             ((700, 2, 31), (0, 1), 1), ((31, 2, 673), (1, 2), 0),
                                             ((1411, 33), (0,), 1)])
def test_contract_with_itself(dtype, dims, keep, order):
    from itg import ops
    rng = np.random.default_rng(sum(dims))
    T = rng.standard_normal(dims).astype(dtype)
    Td = ops.to_device(np.ravel(T, order="F"), dtype)
    la = [i + 1 for i in range(len(dims))]
    lb = [x + 10 if i in keep else x for i, x in enumerate(la)]
    ka, kb = [la[i] for i in keep], [lb[i] for i in keep]
    lc = kb + ka if order else ka + kb
    C, _ = ops.contract(Td, dims, la, Td, dims, lb, lc)
    gone = [i for i in range(len(dims)) if i not in keep]
    n = int(np.prod([dims[i] for i in keep]))
    A = np.reshape(np.transpose(T, list(keep) + gone), (n, -1), order="F")
    _check(np.reshape(ops.to_host(C), (n, n), order="F").astype(np.float64), A, 1.0, dtype)
