"""A transformation leaves nothing behind for the next one: derivatives that start with an
operation of their own do not depend on what the memory held before."""
import numpy as np
import pytest

from et_amd import ccsd
from et_amd import synthetic as syn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('side', ['right', 'left'])
@pytest.mark.parametrize('value', [np.nan, np.inf])
@pytest.mark.parametrize('n_vec', [1, 3])
def test_transformation_after_one_that_is_not_finite(side, value, n_vec):
    o, v, J = 4, 9, 20
    s = syn.system(3, o, v, J, t2_sigma=1e-2, t1_sigma=1e-2, L_scale=0.3)
    with ccsd.CCSD(o, v, J) as wf:
        wf.set_cholesky(s['L'])
        wf.set_oei(s['h'])
        wf.set_orbital_energies(s['eps'])
        wf.set_amplitudes(np.concatenate([s['t1'].ravel(order='F'), s['t2']]))
        wf.construct_t1_cholesky()
        wf.prepare_for_jacobian()
        X = np.asfortranarray(np.random.default_rng(0).normal(size=(wf.n_gs_amplitudes, n_vec)))
        R = wf.jacobian_transformations(X, side)
        bad = wf.jacobian_transformations(np.full_like(X, value), side)
        assert np.isnan(bad).any()
        assert np.array_equal(wf.jacobian_transformations(X, side), R)
