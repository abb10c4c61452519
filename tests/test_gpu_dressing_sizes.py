"""T1 dressing, Fock matrix and residual where the products that start from another array
(the MO vectors, blocks of the Fock matrix) run on the tiled kernels (a copy and a product)
and where they read it themselves, mixed; the ladder's G whole and in strips.  Against the
oracle, to the tolerances of the other sizes."""
import numpy as np
import pytest

from et_amd import ccsd
from et_amd import synthetic as syn
from oracle import ccsd as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('o,v,J', [(20, 30, 1500), (30, 9, 700), (2, 24, 460), (2, 26, 460)])
def test_residual(o, v, J):
    print(f'dressing o={o} v={v} J={J}', flush=True)
    s = syn.system(o * v, o, v, J, t2_sigma=0.02, t1_sigma=0.03, J_decay=8.0, L_scale=0.1)
    Lt = O.t1_cholesky(s['L'], s['t1'], o)
    F = O.fock_t1(s['h'], Lt, s['t1'], o)
    ref = O.omega(s['L'], Lt, F, s['t1'], s['t2'], o)
    with ccsd.CCSD(o, v, J) as wf:
        wf.set_cholesky(s['L'])
        wf.set_oei(s['h'])
        wf.set_orbital_energies(s['eps'])
        wf.set_amplitudes(np.concatenate([s['t1'].ravel(order='F'), s['t2']]))
        wf.construct_t1_cholesky()
        np.testing.assert_allclose(wf.construct_fock(), F, rtol=0, atol=1e-12 * np.abs(F).max())
        assert np.abs(wf.construct_omega() - ref).max() < 1e-12 * np.abs(ref).max()
