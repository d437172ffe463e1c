"""The MLP's training passes at the edges of the fused outer layers: inputs and
outputs at and one past the register tiles, hidden widths around a block,
rows around the LDS tile and one block's share, and the shapes past the limit
that run as matrix products. Each stage is held to the a-priori bound of its
sums in FP32 (u = 2^-24), from the values the device itself gave to the stage
before; GELU and its derivative are taken within 8 u of their argument's scale.
"""
import numpy as np
import pytest

from oracle import mlp as omlp

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def _within(got, want, bound):
    assert got.shape == want.shape
    assert (np.abs(got - want) <= bound + 1e-37).all(), (np.abs(got - want) / (bound + 1e-37)).max()


@pytest.mark.parametrize("rows,i,h,o", [
    (1, 1, 1, 1), (15, 16, 255, 4), (16, 17, 256, 5), (17, 32, 257, 16), (513, 33, 64, 9),
    (700, 12, 300, 17), (2049, 12, 256, 4), (4100, 27, 100, 9), (9000, 31, 513, 15)])
def test_stages(rows, i, h, o):
    from itg import ops
    rng = np.random.default_rng(rows + i)
    p = (rng.standard_normal(omlp.param_count(i, h, o)) / np.sqrt(h)).astype(np.float32)
    X = rng.standard_normal((rows, i)).astype(np.float32)
    T = rng.standard_normal((rows, o)).astype(np.float32)
    P, Xd, Td = (ops.to_device(a.ravel(), "float32") for a in (p, X, T))
    Y, acts = ops.mlp_forward(P, Xd, rows, i, h, o)
    G, loss = ops.mlp_backward(P, Xd, Td, acts, Y, rows, i, h, o)
    W1, b1, W2, b2, W3, b3 = omlp.unpack(p, i, h, o)
    X, T = X.astype(np.float64), T.astype(np.float64)
    Y = ops.to_host(Y).reshape(rows, o).astype(np.float64)
    Z1, A1, Z2, A2 = ops.to_host(acts).reshape(4, rows, h).astype(np.float64)

    def affine(x, W, b):
        return x @ W.T + b, (x.shape[1] + 4) * U * (abs(x) @ abs(W).T + abs(b))

    _within(Z1, *affine(X, W1, b1))
    _within(A1, omlp.gelu(Z1), 8 * U * abs(Z1))
    _within(Z2, *affine(A1, W2, b2))
    _within(A2, omlp.gelu(Z2), 8 * U * abs(Z2))
    _within(Y, *affine(A2, W3, b3))

    sizes = np.cumsum([0, h * i, h, h * h, h, o * h, o])
    g = ops.to_host(G).astype(np.float64)
    gW1, gb1, gW2, gb2, gW3, gb3 = (g[a:b] for a, b in zip(sizes[:-1], sizes[1:]))
    n = rows * o
    assert abs(loss - ((Y - T) ** 2).mean()) <= 8 * U * ((Y - T) ** 2).mean()
    dY = 2 * (Y - T) / n
    k = rows + o + 8
    _within(gb3, dY.sum(0), k * U * abs(dY).sum(0))
    _within(gW3.reshape(o, h), dY.T @ A2, k * U * (abs(dY).T @ abs(A2)))
    M2 = 1.13 * (abs(dY) @ abs(W3))                    # |gelu'| <= 1.13
    dZ2 = (dY @ W3) * omlp.gelu_grad(Z2)
    k += 16
    _within(gb2, dZ2.sum(0), k * U * M2.sum(0))
    _within(gW2.reshape(h, h), dZ2.T @ A1, k * U * (M2.T @ abs(A1)))
    M1 = 1.13 * (M2 @ abs(W2))
    dZ1 = (dZ2 @ W2) * omlp.gelu_grad(Z1)
    k += h + 16
    _within(gb1, dZ1.sum(0), k * U * M1.sum(0))
    _within(gW1.reshape(h, i), dZ1.T @ X, k * U * (M1.T @ abs(X)))
