"""Edges of the native contraction kernel's tiles, stages and K split: rows,
columns and K one off the tile and stage sizes, K tables (contracted modes
that do not merge), operands read along either index, accumulation into C.
The bound is the a-priori one of a K-term sum in the accumulator's
precision: |C - AB| <= (K + 4) u (|A| |B| + |C0|) element by element.
"""
import numpy as np
import pytest

from oracle import tensor_ops as ot

pytestmark = pytest.mark.gpu


def _run(dtype, ea, eb, ec, dims, beta, seed):
    from itg import ops
    rng = np.random.default_rng(seed)
    A = rng.standard_normal([dims[x] for x in ea]).astype(dtype)
    B = rng.standard_normal([dims[x] for x in eb]).astype(dtype)
    C0 = rng.standard_normal([dims[x] for x in ec]).astype(dtype)
    lab = {x: i + 1 for i, x in enumerate(dims)}
    up = lambda x: ops.to_device(ot.to_flat(x), dtype)
    out = up(C0)
    ops.contract(up(A), A.shape, [lab[x] for x in ea], up(B), B.shape, [lab[x] for x in eb],
                 [lab[x] for x in ec], beta=beta, out=out)
    got = ot.from_flat(ops.to_host(out), C0.shape).astype(np.float64)
    e = "%s,%s->%s" % (ea, eb, ec)
    A, B, C0 = A.astype(np.float64), B.astype(np.float64), C0.astype(np.float64)
    ref = np.einsum(e, A, B, optimize=True) + beta * C0
    K = int(np.prod([dims[x] for x in ea if x in eb]))
    u = 2.0 ** (-53 if dtype == "float64" else -24)
    bound = (K + 4) * u * (np.einsum(e, abs(A), abs(B), optimize=True) + abs(beta * C0))
    assert (abs(got - ref) <= bound).all(), (abs(got - ref) / bound).max()


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("m,n,k", [(1, 17, 1), (31, 33, 15), (32, 32, 16), (33, 31, 17),
                                   (63, 65, 31), (64, 64, 32), (65, 63, 33), (127, 129, 48),
                                   (129, 127, 49), (20, 700, 7), (700, 20, 500), (40, 24, 3001),
                                   (1500, 1100, 30)])
@pytest.mark.parametrize("ea,eb", [("mk", "kn"), ("km", "kn"), ("mk", "nk"), ("km", "nk")])
def test_tiles(dtype, m, n, k, ea, eb):
    _run(dtype, ea, eb, "mn", dict(m=m, n=n, k=k), 0.0, m + n + k)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("s", [(3, 5, 7, 2, 5, 3), (9, 8, 7, 11, 6, 5), (13, 10, 17, 9, 16, 2),
                               (2, 40, 3, 30, 19, 23)])
@pytest.mark.parametrize("ea,eb,ec", [
    ("akbl", "lckd", "abcd"), ("kalb", "dkcl", "abcd"), ("klab", "cdlk", "cadb"),
    ("abkl", "cldk", "dbca"), ("lakb", "kcld", "bdac")])
@pytest.mark.parametrize("beta", [0.0, -0.5])
def test_tables(dtype, s, ea, eb, ec, beta):
    _run(dtype, ea, eb, ec, dict(zip("abcdkl", s)), beta, sum(s))
