"""Small products: the route taken in FP32 is no slower than the one in FP64."""
import pytest

from et_amd import ccsd

pytestmark = pytest.mark.gpu

SHAPES = [
    # few tiles, operands that lanes read along the rows
    (510, 254, 5347, 'N', 'T'),
    (107, 640, 3408, 'N', 'T'),
]


@pytest.mark.parametrize('m,n,k,ta,tb', SHAPES)
def test_fp32_is_not_slower_than_fp64(m, n, k, ta, tb):
    def seconds(precision):
        return min(ccsd.bench_gemm(m, n, k, precision, reps=20, ta=ta, tb=tb) for _ in range(5))
    t32, t64 = seconds(ccsd.FP32), seconds(ccsd.FP64)
    assert t32 < 1.25 * t64, (t32, t64)
