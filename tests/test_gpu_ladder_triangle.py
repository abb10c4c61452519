"""The triangle of G that the ladder takes as one int8 product, by column pieces whose
tiles above the diagonal are left out: many groups of row tiles, blocks that do not
divide a tile, and the same residual from triangles and off-diagonal blocks of other
sizes.  The residues are exact, so only the order of the ladder's k panels differs:
1e-13 of the largest element, as for the other block sizes' tests."""
import numpy as np
import pytest

from et_amd import ccsd
from et_amd import synthetic as syn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('o,v,J,batches', [(3, 130, 300, (65, 44)), (4, 97, 500, (50,)), (2, 64, 1100, (33,))])
def test_triangle_pieces(o, v, J, batches):
    print(f'ladder triangle o={o} v={v} J={J}', flush=True)
    s = syn.system(7, o, v, J, t2_sigma=1e-3, t1_sigma=1e-2, L_scale=0.02)
    with ccsd.CCSD(o, v, J) as wf:
        wf.set_cholesky(s['L'])
        wf.set_oei(s['h'])
        wf.set_amplitudes(np.concatenate([s['t1'].ravel(order='F'), s['t2']]))
        wf.construct_t1_cholesky()
        ref = wf.construct_omega()
        for nb in batches:
            wf.set_ladder_batch(nb)
            assert np.abs(wf.construct_omega() - ref).max() < 1e-13 * np.abs(ref).max()
