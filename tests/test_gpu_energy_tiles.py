"""The energy's 32 x 32 tiles of (b, j) at their edges: occupied and virtual counts below,
at and above one and two tiles.  Against the oracle, to the tolerance that the energies of
the other sizes are tested to."""
import numpy as np
import pytest

from et_amd import ccsd
from et_amd import synthetic as syn
from oracle import ccsd as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('o,v', [(1, 1), (1, 33), (5, 31), (31, 4), (32, 32), (33, 3), (40, 37), (65, 2)])
def test_energy(o, v):
    print(f'energy o={o} v={v}', flush=True)
    s = syn.system(o + v, o, v, 6, t2_sigma=0.05, t1_sigma=0.1, L_scale=0.3)
    with ccsd.CCSD(o, v, 6) as wf:
        wf.set_cholesky(s['L'])
        wf.set_oei(s['h'])
        wf.set_amplitudes(np.concatenate([s['t1'].ravel(order='F'), s['t2']]))
        wf.construct_t1_cholesky()
        e = wf.calculate_energy()
    e_ref = O.correlation_energy(O.t1_cholesky(s['L'], s['t1'], o), s['t1'], s['t2'], o)
    assert abs(e - e_ref) < 1e-12 * max(1.0, abs(e_ref))
