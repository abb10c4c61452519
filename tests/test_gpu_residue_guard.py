"""FP64 products on the int8 matrix cores: blocks whose outputs need more digits than the rows' scaled
integers hold, and rows that are not finite, go to the FP64 kernel.

Error bound, relative to sum |a_k b_k| of each output: 0.82 u rms (u = 2^-53) from the operands' rounding
where an output stays on the int8 path, and about 0.5 u for an FP64 sum of terms of random sign
(u / sqrt(6) of each partial sum); 2 u rms is asked for over the samples."""
import time

import numpy as np
import pytest

from et_amd import ccsd
from et_amd import synthetic as syn

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


def _relative_errors(rng, A, B, out, count=1500, rows=None, cols=None):
    m, n = out.shape
    i = rng.choice(rows if rows is not None else m, count)
    j = rng.choice(cols if cols is not None else n, count)
    a, b = A[i], B[:, j].T
    exact = np.einsum('sk,sk->s', a.astype(np.longdouble), b.astype(np.longdouble))
    return np.asarray((out[i, j] - exact) / np.einsum('sk,sk->s', np.abs(a), np.abs(b)), dtype=float)


@pytest.mark.parametrize('decades', [0, 2, 3, 4, 6, 8, 12])
@pytest.mark.parametrize('m,n,k,ta,tb', [(2100, 2000, 2048, 'N', 'N'), (1793, 2051, 4097, 'T', 'N'),
                                         (2560, 2432, 1600, 'N', 'T'), (1800, 1790, 4000, 'T', 'T')])
def test_opposite_grading(m, n, k, ta, tb, decades):
    """Large elements of every row meet small ones of every column."""
    rng = np.random.default_rng(decades + k)
    g = 10.0 ** (-decades * np.arange(k) / k)
    A, B = rng.normal(size=(m, k)) * g, rng.normal(size=(k, n)) * g[::-1, None]
    out = ccsd.device_gemm(ta, tb, 1.0, A.T if ta == 'T' else A, B.T if tb == 'T' else B, 0.0, np.zeros((m, n)))
    e = _relative_errors(rng, A, B, out)
    print('grading %d: rms %.2f u, largest %.1f u' % (decades, np.sqrt(np.mean(e ** 2)) / U, np.abs(e).max() / U), flush=True)
    assert np.sqrt(np.mean(e ** 2)) < 2 * U


@pytest.mark.parametrize('m,n,k', [(2561, 2433, 2561), (1793, 2051, 4097)])
def test_some_blocks(m, n, k):
    """Rows of one block graded against the columns of another: those rows and columns meet in one
    block, the others in blocks that keep the int8 product's very bits."""
    rng = np.random.default_rng(m)
    A, B = rng.normal(size=(m, k)), rng.normal(size=(k, n))
    plain = ccsd.device_gemm('N', 'N', 1.5, A, B, 0.0, np.zeros((m, n)))
    g = 10.0 ** (-9 * np.arange(k) / k)
    rows, cols = slice(640, 700), slice(1290, 1400)
    A2, B2 = A.copy(), B.copy()
    A2[rows] *= g
    B2[:, cols] *= g[::-1, None]
    C = rng.normal(size=(m, n))
    out = ccsd.device_gemm('N', 'N', 1.5, A2, B2, 0.0, C)
    same = np.ones((m, n), bool)
    same[rows] = False
    same[:, cols] = False
    same[640:768, 1280:1408] = False
    assert np.array_equal(out[same], plain[same])
    e = _relative_errors(rng, 1.5 * A2, B2, out, rows=np.arange(640, 700), cols=np.arange(1290, 1400))
    assert np.sqrt(np.mean(e ** 2)) < 2 * U


def test_rows_of_zeros_and_of_nans():
    rng = np.random.default_rng(3)
    m, n, k = 2100, 2000, 2048
    A, B = rng.normal(size=(m, k)), rng.normal(size=(k, n))
    plain = ccsd.device_gemm('N', 'N', 1.0, A, B, 0.0, np.zeros((m, n)))
    A[5], A[1500:1520], B[:, 77] = 0.0, 0.0, 0.0
    A[300, 9] = np.nan
    out = ccsd.device_gemm('N', 'N', 1.0, A, B, 0.0, np.zeros((m, n)))
    live = np.setdiff1d(np.arange(m), np.r_[5, 300, 1500:1520])
    cols = np.setdiff1d(np.arange(n), [77])
    assert (out[5] == 0).all() and (out[1500:1520] == 0).all() and (out[live, 77] == 0).all() and np.isnan(out[300]).all()
    away = live[(live < 256) | (live >= 384)]                 # zeros leave the other rows of their block alone
    assert np.array_equal(out[np.ix_(away, cols)], plain[np.ix_(away, cols)])
    near = live[(live >= 256) & (live < 384)]
    e = _relative_errors(rng, A, B, out, rows=near, cols=cols)
    assert np.sqrt(np.mean(e ** 2)) < 2 * U


def test_a_residual_that_is_not_finite_takes_no_longer():
    """All rows of the products are NaN (a diverged iteration): the FP64 kernels' time, within four of
    the finite residual's."""
    o, v, J = 20, 76, 900
    s = syn.system(3, o, v, J, t2_sigma=1e-3, t1_sigma=1e-2, L_scale=0.02)
    t = np.concatenate([s['t1'].ravel(order='F'), s['t2']])
    with ccsd.CCSD(o, v, J) as wf:
        wf.set_cholesky(s['L'])
        wf.set_oei(s['h'])

        def seconds(t):
            wf.set_amplitudes(t)
            wf.construct_t1_cholesky()
            wf.construct_omega(copy_out=False)
            best = np.inf
            for _ in range(5):
                t0 = time.perf_counter()
                wf.construct_omega(copy_out=False)
                best = min(best, time.perf_counter() - t0)
            return best
        finite, nan = seconds(t), seconds(np.full_like(t, np.nan))
        assert np.isnan(wf.get_omega()).any()
    print('finite %.2f ms, not finite %.2f ms' % (1e3 * finite, 1e3 * nan), flush=True)
    assert nan < 4 * finite
