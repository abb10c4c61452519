"""Small products: the route taken in FP32 is no slower than the one in FP64, and right on both sides of the rule."""
import numpy as np
import pytest

from et_amd import ccsd

pytestmark = pytest.mark.gpu

SHAPES = [
    # few tiles (the first two with operands that lanes read along the rows), then tiled
    (510, 254, 5347, 'N', 'T'),
    (107, 640, 3408, 'N', 'T'),
    (1526, 1201, 141, 'T', 'T'),
    (3137, 589, 145, 'T', 'N'),
]


@pytest.mark.parametrize('m,n,k,ta,tb', SHAPES[:2])
def test_fp32_is_not_slower_than_fp64(m, n, k, ta, tb):
    def seconds(precision):
        return min(ccsd.bench_gemm(m, n, k, precision, reps=20, ta=ta, tb=tb) for _ in range(5))
    t32, t64 = seconds(ccsd.FP32), seconds(ccsd.FP64)
    assert t32 < 1.25 * t64, (t32, t64)


def test_short_k_over_many_outputs_is_tiled():
    """Three times the k (past the rule's range) takes 2.2 times as long as the tiled kernel, 1.4 times as
    long as the products of few tiles."""
    def seconds(k):
        return min(ccsd.bench_gemm(1526, 1201, k, ccsd.FP64, reps=20, ta='T', tb='T') for _ in range(5))
    t, t3 = seconds(141), seconds(423)
    assert t < 0.57 * t3, (t, t3)


@pytest.mark.parametrize('m,n,k,ta,tb', SHAPES)
@pytest.mark.parametrize('precision', [ccsd.FP64, ccsd.FP32])
def test_product(precision, m, n, k, ta, tb):
    rng = np.random.default_rng(k)
    A, B, C = rng.normal(size=(m, k)), rng.normal(size=(k, n)), rng.normal(size=(m, n))
    out = ccsd.device_gemm(ta, tb, 0.7, A.T if ta == 'T' else A, B.T if tb == 'T' else B, -0.3, C, precision)
    eps = 2.0 ** -53 if precision == ccsd.FP64 else 2.0 ** -24
    # every operation's rounding, all in one direction, is k eps; here a random walk of at most sqrt(k)
    # steps, five times its deviation, and the operands' rounding
    tol = (5 * np.sqrt(k) + 10) * eps * (np.abs(A) @ np.abs(B) + np.abs(C))
    assert (np.abs(out - (0.7 * (A @ B) - 0.3 * C)) <= tol).all()
