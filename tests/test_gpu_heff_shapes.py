"""The effective-Hamiltonian apply over the shapes that take different W-pass
kernels and products: one row tile and its remainders, two row tiles (chiL
from 200), one to six column tiles of the operator, boundary operators
(wl = 1, wr = 1), more outputs than one launch holds (d = 1, a wide MPO), the
20 x 20 operator on both sides of its size rule, a K-split C4. Against the
four einsum contractions in float64; FP64 bound 1e-12 of the result's norm
(a few K eps), FP32 2e-5."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [("float64", 1e-12), ("float32", 2e-5)])
@pytest.mark.parametrize("chiL,wl,wm,wr,d,chiR", [
    (1, 1, 5, 5, 2, 3), (15, 5, 5, 1, 2, 17), (16, 5, 5, 5, 2, 16), (33, 3, 4, 6, 2, 9),
    (40, 14, 14, 14, 2, 31), (199, 5, 5, 5, 3, 20), (200, 2, 2, 2, 3, 21), (217, 6, 7, 8, 2, 40),
    (300, 5, 5, 5, 2, 2200), (20, 1, 2, 1100, 1, 3), (6, 14, 3, 20, 2, 250)])
def test_heff_shapes(chiL, wl, wm, wr, d, chiR, dtype, tol):
    from itg import ops
    rng = np.random.default_rng(chiL + chiR)
    L = rng.standard_normal((chiL, wl, chiL)).astype(dtype)
    R = rng.standard_normal((chiR, wr, chiR)).astype(dtype)
    W1 = rng.standard_normal((wl, wm, d, d)).astype(dtype)
    W2 = rng.standard_normal((wm, wr, d, d)).astype(dtype)
    psi = rng.standard_normal((chiL, d, d, chiR)).astype(dtype)
    up = lambda x: ops.to_device(np.ravel(x, order="F"), dtype)
    y = ops.heff2_apply(up(L), up(W1), up(W2), up(R), up(psi), chiL, wl, wm, wr, d, chiR)
    got = np.reshape(ops.to_host(y), psi.shape, order="F").astype(np.float64)
    L, R, W1, W2, psi = [x.astype(np.float64) for x in (L, R, W1, W2, psi)]
    T = np.tensordot(L, psi, (2, 0))                       # a' l s t b
    T = np.tensordot(T, W1, ([1, 2], [0, 3]))              # a' t b m s'
    T = np.tensordot(T, W2, ([1, 3], [3, 0]))              # a' b s' r t'
    ref = np.tensordot(T, R, ([1, 3], [2, 1]))             # a' s' t' b'
    assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref)
