"""Allocations that fail."""
import numpy as np
import pytest
import torch

from et_amd import ccsd
from et_amd import synthetic as syn

pytestmark = pytest.mark.gpu


def _system(o, v, J):
    s = syn.system(5, o, v, J, t2_sigma=1e-3, t1_sigma=1e-2, L_scale=0.02)
    wf = ccsd.CCSD(o, v, J)
    wf.set_cholesky(s['L'])
    wf.set_oei(s['h'])
    wf.set_orbital_energies(s['eps'])
    wf.set_amplitudes(np.concatenate([s['t1'].ravel(order='F'), s['t2']]))
    wf.construct_t1_cholesky()
    return wf


def _fail_an_allocation(wf, v):
    """A ladder block of v x v pairs: beyond the card's memory, refused by the runtime."""
    assert 8 * v ** 4 > 1.5 * torch.cuda.get_device_properties(0).total_memory
    with pytest.raises(ccsd.ETGError, match='out of memory'):
        wf.set_ladder_batch(v)


def test_a_failed_allocation_is_reported_once():
    """It is an error of its own call; the next launch does not report it again."""
    v = 520
    with _system(1, v, 3) as wf:
        wf.set_ladder_batch(40)
        ref = wf.construct_omega()
        _fail_an_allocation(wf, v)
        wf.set_ladder_batch(40)
        assert np.array_equal(wf.construct_omega(), ref)
