"""Products of few output tiles (et_amd/csrc/gemm.hip gemm_few_tiles) against numpy."""
import numpy as np
import pytest

from et_amd import ccsd

pytestmark = pytest.mark.gpu

# edges of the 16 and 32 tiles and of the 16-deep chunks, one wave's chunk only, k splits with a
# short last one (deep and shallow reductions), GEMV shapes, the ends of the range by operations
SHAPES = [(1, 1, 1), (16, 16, 16), (17, 15, 17), (33, 31, 63), (32, 64, 64), (95, 95, 279), (19, 5, 5301),
          (5, 300, 129), (361, 1, 1000), (1, 361, 65), (700, 900, 601), (20, 20, 40007), (3, 2, 100003)]


@pytest.mark.parametrize('ta', ['N', 'T'])
@pytest.mark.parametrize('tb', ['N', 'T'])
@pytest.mark.parametrize('m,n,k', SHAPES)
def test_few_tiles(ta, tb, m, n, k):
    """Each output a sum of k products, every partial sum rounded: |error| <= (k + 3) u sum |a b|,
    with u = 2^-53 (and FP32 operands and sums: (k + 5) 2^-24)."""
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    A, B, C = rng.normal(size=(m, k)), rng.normal(size=(k, n)), rng.normal(size=(m, n))
    ref = 0.7 * A @ B - 0.3 * C
    mag = 0.7 * np.abs(A) @ np.abs(B) + 0.3 * np.abs(C)
    a, b = (A.T if ta == 'T' else A), (B.T if tb == 'T' else B)
    out = ccsd.device_gemm(ta, tb, 0.7, a, b, -0.3, C)
    assert (np.abs(out - ref) <= 2 * (k + 3) * 2.0 ** -53 * mag).all()
    assert np.abs(out - ref).max() < 1e-14 * np.sqrt(k) * 8
    out32 = ccsd.device_gemm(ta, tb, 0.7, a, b, -0.3, C, precision=ccsd.FP32)
    assert (np.abs(out32 - ref) <= 2 * (k + 5) * 2.0 ** -24 * mag).all()
    assert np.abs(out32 - ref).max() < 2.0 ** -24 * np.sqrt(k) * 40
