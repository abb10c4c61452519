"""FP64 products that run as exact int8 products (et_amd/csrc/gemm_residue.hip) against long double."""
import numpy as np
import pytest

from et_amd import ccsd
from et_amd import synthetic as syn

pytestmark = pytest.mark.gpu


def _operands(rng, m, n, k, kind):
    A, B = rng.normal(size=(m, k)), rng.normal(size=(k, n))
    if kind == 'positive':
        A, B = np.abs(A), np.abs(B)
    if kind == 'wide':      # rows of very different size, elements over eight decades
        A *= 10.0 ** rng.uniform(-150, 150, size=(m, 1)) * 10.0 ** rng.uniform(-8, 0, size=(m, k))
    return A, B


def _check(rng, A, B, C, alpha, beta, out, extra=()):
    """Sampled outputs (the corners and `extra` among them) within the rounding of the operands to
    integers (2^-58 (|a|_2 |b|_1 + |b|_2 |a|_1)) and of the final operations."""
    m, n = out.shape
    ii = np.concatenate([[0, m - 1, 0, m - 1], rng.integers(0, m, 2000), [e[0] for e in extra]]).astype(int)
    jj = np.concatenate([[0, 0, n - 1, n - 1], rng.integers(0, n, 2000), [e[1] for e in extra]]).astype(int)
    for lo in range(0, len(ii), 256):
        i, j = ii[lo:lo + 256], jj[lo:lo + 256]
        a, b = A[i], B[:, j].T
        exact = np.einsum('sk,sk->s', a.astype(np.longdouble), b.astype(np.longdouble))
        a2, b2 = np.linalg.norm(a, axis=1), np.linalg.norm(b, axis=1)
        a1, b1 = np.abs(a).sum(1), np.abs(b).sum(1)
        ref = alpha * exact + beta * C[i, j]
        tol = abs(alpha) * (2.0 ** -58 * (a2 * b1 + b2 * a1) + 2.0 ** -50 * np.abs(exact)) \
            + 2.0 ** -50 * np.abs(beta * C[i, j])
        assert (np.abs(out[i, j] - ref) <= tol).all()


@pytest.mark.parametrize('m,n,k,kind', [
    (2561, 2433, 2561, 'normal'),       # one row, column and k beyond whole tiles and steps (256 x 128 tiles)
    (2560, 2432, 2560, 'positive'),     # whole tiles
    (1793, 2051, 4097, 'wide'),         # 256 x 256 tiles
    (820, 4003, 4000, 'normal'),        # few rows
    (4100, 4099, 1270, 'wide'),         # short k
])
@pytest.mark.parametrize('ta', ['N', 'T'])
@pytest.mark.parametrize('tb', ['N', 'T'])
def test_product(ta, tb, m, n, k, kind):
    rng = np.random.default_rng(m + k)
    A, B = _operands(rng, m, n, k, kind)
    C = rng.normal(size=(m, n))
    out = ccsd.device_gemm(ta, tb, 0.7, A.T if ta == 'T' else A, B.T if tb == 'T' else B, -0.3, C)
    _check(rng, A, B, C, 0.7, -0.3, out)


@pytest.mark.parametrize('m,n', [(9000, 5000), (5000, 9000)])
def test_product_in_panels(m, n):
    """Packs and outputs beyond the workspace: two panels of the longer operand."""
    rng = np.random.default_rng(m)
    k = 5000
    A, B = rng.normal(size=(m, k)), rng.normal(size=(k, n))
    C = np.zeros((m, n))
    out = ccsd.device_gemm('N', 'N', 1.0, A, B, 0.0, C)
    edge = [(i, j) for i in (4607, 4608, 4500) for j in (4607, 4608, 4500)]
    _check(rng, A, B, C, 1.0, 0.0, out, [(min(i, m - 1), min(j, n - 1)) for i, j in edge])


def test_infinities_and_nans():
    """An infinity or NaN reaches the outputs of its row or column, as in the sum itself, and no others."""
    rng = np.random.default_rng(4)
    m, n, k = 2100, 2000, 2048
    A, B = rng.normal(size=(m, k)), rng.normal(size=(k, n))
    A[5, 7], A[300, 0], A[300, 1], A[2099, k - 1] = np.inf, np.inf, -np.inf, np.nan
    B[9, 11], B[7, 1500] = -np.inf, 0.0
    C = np.ones((m, n))
    out = ccsd.device_gemm('N', 'N', 1.0, A, B, 0.5, C)
    with np.errstate(invalid='ignore'):
        ref = A @ B + 0.5
    assert np.array_equal(np.isnan(out), np.isnan(ref))
    assert np.array_equal(np.isposinf(out), np.isposinf(ref)) and np.array_equal(np.isneginf(out), np.isneginf(ref))
    ok = np.isfinite(ref)
    assert np.abs(out[ok] - ref[ok]).max() < 1e-14 * np.sqrt(k) * 8


def test_transformations_of_a_group():
    """Shared and batched operands: FP64 transformations of one group equal single ones, replayed
    graphs equal the first pass, and left and right are adjoint; the products run as int8 ones."""
    o, v, J = 20, 76, 900
    s = syn.system(3, o, v, J, t2_sigma=1e-3, t1_sigma=1e-2, L_scale=0.02)
    rng = np.random.default_rng(0)
    with ccsd.CCSD(o, v, J) as wf:
        wf.set_cholesky(s['L'])
        wf.set_oei(s['h'])
        wf.set_orbital_energies(s['eps'])
        wf.set_amplitudes(np.concatenate([s['t1'].ravel(order='F'), s['t2']]))
        wf.construct_t1_cholesky()
        wf.set_kernel_ledger(True)
        wf.prepare_for_jacobian()
        assert any('gemm_residue' in r[0] for r in wf.kernel_ledger())
        wf.set_kernel_ledger(False)
        X = np.asfortranarray(rng.normal(size=(wf.n_gs_amplitudes, 3)))
        Y = np.asfortranarray(rng.normal(size=(wf.n_gs_amplitudes, 3)))
        AX, AtY = wf.jacobian_transformations(X, 'right'), wf.jacobian_transformations(Y, 'left')
        for side, V, R in (('right', X, AX), ('left', Y, AtY)):
            assert np.array_equal(wf.jacobian_transformations(V, side), R)
            one = wf.jacobian_transformations(V[:, 1:2], side)
            assert np.abs(one[:, 0] - R[:, 1]).max() < 1e-13 * np.abs(R[:, 1]).max()
        left, right = Y.T @ AX, AtY.T @ X
        assert np.abs(left - right).max() < 1e-12 * np.linalg.norm(Y[:, 0]) * np.linalg.norm(AX[:, 0])


@pytest.mark.parametrize('o,v,J', [(12, 61, 700), (10, 76, 1270)])
def test_ladder_blocks(o, v, J):
    """The residual with the G of the ladder as one triangle, as triangles and off-diagonal blocks,
    and as blocks too small for the int8 path; oddly aligned columns of a block row too."""
    s = syn.system(5, o, v, J, t2_sigma=1e-3, t1_sigma=1e-2, L_scale=0.02)
    with ccsd.CCSD(o, v, J) as wf:
        wf.set_cholesky(s['L'])
        wf.set_oei(s['h'])
        wf.set_amplitudes(np.concatenate([s['t1'].ravel(order='F'), s['t2']]))
        wf.construct_t1_cholesky()
        ref = wf.construct_omega()
        wf.set_kernel_ledger(True)
        wf.construct_omega(copy_out=False)
        assert any('gemm_residue' in r[0] for r in wf.kernel_ledger())
        wf.set_kernel_ledger(False)
        for nb in (v // 2 + 1, 33, 5):
            wf.set_ladder_batch(nb)
            assert np.abs(wf.construct_omega() - ref).max() < 1e-13 * np.abs(ref).max()
