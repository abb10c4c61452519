"""int8 products that do not fit their workspace at once: groups of a batch, panels of a triangle; and
long results copied to the host from each entry point that stages them."""
import numpy as np
import pytest

from et_amd import ccsd
from et_amd import synthetic as syn

pytestmark = pytest.mark.gpu


def _load(o, v, J):
    s = syn.system(3, o, v, J, t2_sigma=1e-3, t1_sigma=1e-2, L_scale=0.02)
    wf = ccsd.CCSD(o, v, J)
    wf.set_cholesky(s['L'])
    wf.set_oei(s['h'])
    wf.set_orbital_energies(s['eps'])
    wf.set_amplitudes(np.concatenate([s['t1'].ravel(order='F'), s['t2']]))
    wf.construct_t1_cholesky()
    return wf


def test_batches_in_groups():
    """Eleven vectors at n_t1 = 1520: the 0.4 GB workspace takes them in several groups, the last one
    ragged.  Against single transformations, and left against right."""
    with _load(20, 76, 900) as wf:
        wf.prepare_for_jacobian()
        rng = np.random.default_rng(0)
        X = np.asfortranarray(rng.normal(size=(wf.n_gs_amplitudes, 11)))
        Y = np.asfortranarray(rng.normal(size=(wf.n_gs_amplitudes, 11)))
        out = {}
        for side, V in (('right', X), ('left', Y)):
            print('eleven vectors, %s' % side, flush=True)
            R = out[side] = wf.jacobian_transformations(V, side)
            assert np.array_equal(wf.jacobian_transformations(V, side), R)
            for k in (0, 5, 6, 10):
                one = wf.jacobian_transformations(V[:, k:k + 1], side)
                assert np.abs(one[:, 0] - R[:, k]).max() < 1e-13 * np.abs(R[:, k]).max()
        left, right = Y.T @ out['right'], out['left'].T @ X
        assert np.abs(left - right).max() < 1e-12 * np.linalg.norm(Y[:, 0]) * np.linalg.norm(out['right'][:, 0])


def test_triangle_in_panels():
    """G of 22500 x 22500 for 2000 Cholesky vectors: rows and columns of its triangle in panels; against
    ladder blocks that fit at once."""
    with _load(4, 150, 2000) as wf:
        whole = wf.construct_omega()
        wf.set_kernel_ledger(True)
        wf.construct_omega(copy_out=False)
        assert any('gemm_residue' in r[0] for r in wf.kernel_ledger())
        wf.set_kernel_ledger(False)
        for nb in (50, 37):
            wf.set_ladder_batch(nb)
            assert np.abs(wf.construct_omega() - whole).max() < 1e-13 * np.abs(whole).max()


def test_staged_copies_of_every_entry_point():
    """More than 16 MB from the residual, the transformations and the multipliers."""
    with _load(24, 100, 60) as wf:                        # 23 MB
        om = wf.construct_omega()
        assert np.array_equal(wf.get_omega(), om)
        wf.prepare_for_jacobian()
        n = wf.n_gs_amplitudes
        X = np.asfortranarray(np.random.default_rng(1).normal(size=(n, 2)))
        R = wf.jacobian_transformations(X, 'right')
        for k in range(2):
            assert np.array_equal(wf.jacobian_transformation(X[:, k]), wf.jacobian_transformations(X[:, k:k + 1], 'right')[:, 0])
        assert np.array_equal(wf.jacobian_transformations(X, 'right'), R)
        wf.set_multipliers(X[:, 0])
        assert np.array_equal(wf.get_multipliers(), X[:, 0])
