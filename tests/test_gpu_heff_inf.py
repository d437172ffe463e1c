"""The Heff apply on a psi that holds an infinity, all other entries of all
operands positive: every output sums it and nothing cancels it, so all are
+inf, whatever the number of the operator's channels (the W pass pads them to
whole products of four)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("chiL,w,d,chiR", [(20, 5, 2, 18), (20, 5, 3, 18), (33, 3, 1, 9), (210, 7, 1, 5),
                                           (16, 6, 3, 16)])
def test_infinity_passes(chiL, w, d, chiR, dtype):
    from itg import ops
    rng = np.random.default_rng(chiL)
    pos = lambda *s: rng.uniform(0.5, 1.0, s).astype(dtype)
    psi = pos(chiL, d, d, chiR)
    psi[3, d - 1, d - 1, 2] = np.inf
    up = lambda x: ops.to_device(np.ravel(x, order="F"), dtype)
    y = ops.heff2_apply(up(pos(chiL, w, chiL)), up(pos(w, w, d, d)), up(pos(w, w, d, d)),
                        up(pos(chiR, w, chiR)), up(psi), chiL, w, w, w, d, chiR)
    assert (ops.to_host(y) == np.inf).all()
