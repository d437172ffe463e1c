"""Bias gradients where the rows cancel: every row occurs twice, at random
places, with opposite output errors, so each bias gradient is a sum of pairs
d, -d and is zero but for the roundings of the FP64 sums, rows 2^-53 sum |d|
(partial sums rounded to FP32 would leave 2^-24 of each)."""
import numpy as np
import pytest

from oracle import mlp as omlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,i,h,o", [(200, 12, 64, 4), (4096, 12, 256, 4), (6000, 27, 300, 9)])
def test_cancelling_rows(rows, i, h, o):
    from itg import ops
    rng = np.random.default_rng(rows)
    p = (rng.standard_normal(omlp.param_count(i, h, o)) / np.sqrt(h)).astype(np.float32)
    half = rng.standard_normal((rows // 2, i)).astype(np.float32)
    err = rng.standard_normal((rows // 2, o)).astype(np.float32)
    order = rng.permutation(rows)
    X = np.concatenate([half, half])[order]
    Y = np.concatenate([err, -err])[order]
    P, Xd, Yd = (ops.to_device(a.ravel(), "float32") for a in (p, X, Y))
    T = ops.to_device(np.zeros(rows * o, np.float32), "float32")
    _, acts = ops.mlp_forward(P, Xd, rows, i, h, o)
    G, _ = ops.mlp_backward(P, Xd, T, acts, Yd, rows, i, h, o)
    g = ops.to_host(G).astype(np.float64)
    W1, b1, W2, b2, W3, b3 = omlp.unpack(p, i, h, o)
    Z1, A1, Z2, A2 = ops.to_host(acts).reshape(4, rows, h).astype(np.float64)
    dZ2 = 2.0 / (rows * o) * Y.astype(np.float64) @ W3 * omlp.gelu_grad(Z2)
    dZ1 = dZ2 @ W2 * omlp.gelu_grad(Z1)
    at = np.cumsum([0, h * i, h, h * h, h])
    # sum |d| from FP32 weights and activations: good to far better than 2
    for got, d in ((g[at[1]:at[2]], dZ1), (g[at[3]:at[4]], dZ2)):
        assert (abs(got) <= 2 * rows * 2.0 ** -53 * abs(d).sum(0)).all()
