"""Tangent products whose two operand pairs run as one k range (remainders of the 16-deep
chunks and of the tiles, one vector and several, k splits), through the duality of the two
transformations: the left one forms its products one by one.  1e-12 of the norms, as for
the groups of larger systems."""
import numpy as np
import pytest

from et_amd import ccsd
from et_amd import synthetic as syn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('o,v,J,nb', [(1, 2, 3, 1), (2, 5, 16, 3), (4, 16, 32, 2), (3, 17, 33, 5), (5, 31, 290, 1),
                                      (12, 15, 70, 2)])
def test_right_against_left(o, v, J, nb):
    print(f'operand pairs o={o} v={v} J={J} vectors={nb}', flush=True)
    s = syn.system(o + v, o, v, J, t2_sigma=0.02, t1_sigma=0.03, J_decay=8.0, L_scale=0.2)
    N = o * v
    n = N + N * (N + 1) // 2
    rng = np.random.default_rng(n)
    X, Y = (np.asfortranarray(rng.standard_normal((n, nb))) for _ in range(2))
    with ccsd.CCSD(o, v, J) as wf:
        wf.set_cholesky(s['L'])
        wf.set_oei(s['h'])
        wf.set_orbital_energies(s['eps'])
        wf.set_amplitudes(np.concatenate([s['t1'].ravel(order='F'), s['t2']]))
        wf.construct_t1_cholesky()
        wf.prepare_for_jacobian()
        for _ in range(3):                               # eager, captured, replayed
            AX = wf.jacobian_transformations(X, 'right')
            AtY = wf.jacobian_transformations(Y, 'left')
            scale = np.linalg.norm(Y, axis=0)[:, None] * np.linalg.norm(AX, axis=0)[None, :]
            assert np.all(np.abs(Y.T @ AX - AtY.T @ X) <= 1e-12 * scale)
