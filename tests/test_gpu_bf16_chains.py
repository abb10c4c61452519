"""The FP32 chains of split-bf16 products do not grow with the number of tiles."""
import numpy as np
import pytest

from et_amd import ccsd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('m,n,k', [(4352, 4096, 6144), (2100, 8000, 6000)])
def test_error_of_whole_tiles(m, n, k):
    """Operands of one sign, where a chain's rounding grows in proportion to its length.  More tiles
    than CUs against the first row of tiles alone, whose k is cut into twice as many chains (12 and 6,
    8 and 4): the error may be twice as large (and a quarter for chance)."""
    print(f'split-bf16 chains m={m} n={n} k={k}', flush=True)
    rng = np.random.default_rng(m + k)
    A, B = rng.random((m, k)), rng.random((k, n))
    ref = A[:256] @ B

    def rms(rows):
        got = ccsd.device_gemm('N', 'N', 1.0, A[:rows], B, 0.0, np.zeros((rows, n)), ccsd.BF16X3)
        return np.sqrt(np.mean(((got[:256] - ref) / ref) ** 2))
    assert rms(m) < 2.5 * rms(256)


@pytest.mark.parametrize('m,n,k,beta', [
    (4352, 4090, 1100, 1.5),      # 272 tiles in two chains, the last ones split
    (4352, 4351, 1555, -0.5),     # 289 tiles, odd edges
    (8191, 8161, 1024, 0.0),      # 1024 tiles: whole rounds only
    (65787, 250, 1090, 1.0),      # one tile more than a round
])
def test_products_of_several_chains(m, n, k, beta):
    """The elementwise bound of test_gpu_bf16_rounds."""
    print(f'split-bf16 m={m} n={n} k={k} beta={beta}', flush=True)
    rng = np.random.default_rng(m + n + k)
    A, B, C = rng.standard_normal((m, k)), rng.standard_normal((k, n)), rng.standard_normal((m, n))
    got = ccsd.device_gemm('N', 'N', 1.25, A, B, beta, C, ccsd.BF16X3)
    bound = 1.25 * (3 * 2.0 ** -18 + (3 * k / 32 + 32) * 2.0 ** -24) * (np.abs(A) @ np.abs(B)) + 1e-15
    assert np.all(np.abs(got - (1.25 * (A @ B) + beta * C)) <= bound)
