"""The device Davidson's vector passes at their edges: vectors of fewer
elements than a block, one block and many, basis sizes on both sides of the
2, 4, 8 and 17 vector kernels, a basis that exhausts the space, a start vector
that is an eigenvector. Against the same iteration in numpy, energies and
vectors to 1e-11 (a few hundred eps, both orthogonalised twice)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _operator(chiL, w, d, chiR, seed):
    rng = np.random.default_rng(seed)
    sym = lambda x, p: x + np.transpose(x, p)
    L = sym(rng.standard_normal((chiL, w, chiL)), (2, 1, 0)) / np.sqrt(chiL)
    R = sym(rng.standard_normal((chiR, w, chiR)), (2, 1, 0)) / np.sqrt(chiR)
    W1 = sym(rng.standard_normal((w, w, d, d)), (0, 1, 3, 2)) / w
    W2 = sym(rng.standard_normal((w, w, d, d)), (0, 1, 3, 2)) / w
    return L, W1, W2, R, rng.standard_normal((chiL, d, d, chiR))


def _apply(L, W1, W2, R, x):
    T = np.tensordot(L, x, (2, 0))
    T = np.tensordot(T, W1, ([1, 2], [0, 3]))
    T = np.tensordot(T, W2, ([1, 3], [3, 0]))
    return np.tensordot(T, R, ([1, 3], [2, 1]))


def _reference(op, x, maxiter):
    V = [x / np.linalg.norm(x)]
    AV = [op(V[0])]
    lam = np.vdot(V[0], AV[0])
    phi, q = V[0], AV[0] - lam * V[0]
    for _ in range(maxiter):
        if np.linalg.norm(q) < 1e-12:
            break
        t = q
        for _ in range(2):
            t = t - sum(np.vdot(v, t) * v for v in V)
        V.append(t / np.linalg.norm(t))
        AV.append(op(V[-1]))
        M = np.array([[np.vdot(a, b) for b in AV] for a in V])
        ev, U = np.linalg.eigh(0.5 * (M + M.T))
        u = U[:, 0] * (1.0 if U[0, 0] >= 0 else -1.0)
        lam = ev[0]
        phi = sum(c * v for c, v in zip(u, V))
        q = sum(c * v for c, v in zip(u, AV)) - lam * phi
    return lam, phi / np.linalg.norm(phi), len(V)


def _device(L, W1, W2, R, x, maxiter, **kw):
    from itg import ops
    up = lambda a: ops.to_device(np.ravel(a, order="F"))
    dims = (L.shape[0], W1.shape[0], W1.shape[1], W2.shape[1], x.shape[1], R.shape[0])
    Ld, Rd, psi = up(L), up(R), up(x)
    prep = ops.heff2_prepare(Ld, up(W1), up(W2), Rd, *dims)
    e, n = ops.davidson2(Ld, Rd, prep, psi, *dims, maxiter=maxiter, **kw)
    return e, np.reshape(ops.to_host(psi), x.shape, order="F"), n


@pytest.mark.parametrize("dims", [(1, 3, 2, 1), (3, 2, 2, 5), (16, 5, 2, 16), (33, 3, 2, 20),
                                  (150, 3, 2, 171)])
@pytest.mark.parametrize("maxiter", [1, 2, 3, 4, 7, 8, 16])
def test_davidson_passes(dims, maxiter):
    chiL, w, d, chiR = dims
    L, W1, W2, R, x = _operator(chiL, w, d, chiR, sum(dims))
    maxiter = min(maxiter, x.size - 1)
    e, phi, n = _device(L, W1, W2, R, x, maxiter)
    er, pr, nr = _reference(lambda v: _apply(L, W1, W2, R, v), x, maxiter)
    assert abs(e - er) <= 1e-11 * max(1.0, abs(er))
    assert n == nr
    assert np.linalg.norm(phi - pr) <= 1e-11


def test_davidson_start_is_eigenvector():
    L, W1, W2, R, x = _operator(4, 3, 2, 3, 7)
    n = x.size
    H = np.array([_apply(L, W1, W2, R, v.reshape(x.shape)).ravel() for v in np.eye(n)])
    w, U = np.linalg.eigh(0.5 * (H + H.T))
    v = U[:, 0].reshape(x.shape)
    e, phi, _ = _device(L, W1, W2, R, 3.0 * v, 4)
    assert abs(e - w[0]) <= 1e-11 * abs(w[0])
    assert min(np.linalg.norm(phi - v), np.linalg.norm(phi + v)) <= 1e-9


def test_davidson_zero_start_refused():
    from itg import _lib
    L, W1, W2, R, x = _operator(4, 3, 2, 3, 7)
    with pytest.raises(_lib.ArgumentError):
        _device(L, W1, W2, R, 0.0 * x, 2)
