"""Contractions with one small operand (one thread per fibre of the large one,
the outputs split over the grid) and sums over many K partials: fibres one off
a block of 256 and around the change from one output part to several, every
output group size with remainders, K around the eight loads in flight; partial
counts around the eight at which four waves share an output.
The bound is the a-priori one of a K-term sum in the accumulator's precision:
|C - AB| <= (K + 4) u (|A| |B| + |C0|) element by element.
"""
import pytest

from test_gpu_contract_tiles import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("f,k,g", [(4096, 1, 1), (4097, 7, 3), (4351, 8, 4), (5000, 9, 5),
                                   (4608, 64, 32), (65537, 15, 17), (66000, 28, 28),
                                   (263000, 16, 9), (140000, 13, 31)])
@pytest.mark.parametrize("ea,eb,ec", [("fk", "kg", "fg"), ("kf", "gk", "gf"), ("gk", "kf", "fg")])
@pytest.mark.parametrize("beta", [0.0, -0.5])
def test_small_operand(dtype, f, k, g, ea, eb, ec, beta):
    _run(dtype, ea, eb, ec, dict(f=f, k=k, g=g), beta, f + k + g)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_small_operand_modes(dtype):
    """the fibres are two modes on either side of the contracted ones"""
    _run(dtype, "akblc", "lpkq", "cpbqa", dict(a=37, b=5, c=41, k=3, l=4, p=3, q=3), -0.5, 7)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("m,n", [(20, 20), (33, 63), (96, 130), (256, 256)])
@pytest.mark.parametrize("k", [400, 900, 1800, 4097, 20000])
def test_long_sums(dtype, m, n, k):
    _run(dtype, "km", "nk", "mn", dict(m=m, n=n, k=k), -0.5, m + n + k)
