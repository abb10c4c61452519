"""Split-bf16 products whose tiles do not fill whole rounds of the chip (the last
round's tiles split their k), and the ladder's triangle of G on them.

Elementwise bound of a product: the split leaves 3 x 2^-18 of |A| |B| (the two
operands' remainders and the dropped lo lo term), and each of the 3 k / 32 matrix
instructions and the 32 terms inside one rounds the FP32 sum, 2^-24 each."""
import numpy as np
import pytest

from et_amd import ccsd
from et_amd import synthetic as syn

pytestmark = pytest.mark.gpu


# one tile after 256, tiles for one round and a sixteenth, fewer than a round, odd edges, one tile
@pytest.mark.parametrize('m,n,k,beta', [(65787, 250, 1024, 0.0), (4352, 4090, 1100, 1.5), (1500, 1403, 2048, 0.0),
                                        (303, 301, 5000, -0.5), (130, 256, 1055, 1.0), (4096, 4096, 640, 0.0)])
def test_last_round(m, n, k, beta):
    print(f'split-bf16 m={m} n={n} k={k} beta={beta}', flush=True)
    rng = np.random.default_rng(m + n + k)
    A = rng.standard_normal((m, k))
    B = rng.standard_normal((k, n))
    C = rng.standard_normal((m, n))
    got = ccsd.device_gemm('N', 'N', 1.25, A, B, beta, C, ccsd.BF16X3)
    bound = 1.25 * (3 * 2.0 ** -18 + (3 * k / 32 + 32) * 2.0 ** -24) * (np.abs(A) @ np.abs(B)) + 1e-15
    assert np.all(np.abs(got - (1.25 * (A @ B) + beta * C)) <= bound)


@pytest.mark.parametrize('o,v,J,batches', [(3, 130, 300, (65, 44)), (2, 37, 70, (20, 9))])
def test_ladder_triangle(o, v, J, batches):
    """Against the FP64 residual, to the 2e-4 that split-bf16 residuals are tested to."""
    print(f'split-bf16 ladder o={o} v={v} J={J}', flush=True)
    s = syn.system(8, o, v, J, t2_sigma=1e-3, t1_sigma=1e-2, L_scale=0.02)
    with ccsd.CCSD(o, v, J) as wf:
        wf.set_cholesky(s['L'])
        wf.set_oei(s['h'])
        wf.set_amplitudes(np.concatenate([s['t1'].ravel(order='F'), s['t2']]))
        wf.construct_t1_cholesky()
        ref = wf.construct_omega(ccsd.FP64)
        for nb in (v,) + batches:
            wf.set_ladder_batch(nb)
            err = np.abs(wf.construct_omega(ccsd.BF16X3) - ref).max() / np.abs(ref).max()
            assert err < 2e-4
