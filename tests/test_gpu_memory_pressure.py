"""Allocations that fail: the workspace of the int8 products is given back first: what fits
without it runs without it, on the FP64 kernels."""
import numpy as np
import pytest

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
    """A ladder block of v x v pairs: beyond the card's 288 GB, refused by the runtime."""
    assert 8 * v ** 4 > 500e9
    with pytest.raises(ccsd.ETGError, match='out of memory'):
        wf.set_ladder_batch(v)


def _runs_int8(wf, call):
    wf.set_kernel_ledger(True)
    call()
    used = any('gemm_residue' in r[0] for r in wf.kernel_ledger())
    wf.set_kernel_ledger(False)
    return used


def test_workspace_is_given_back():
    v = 520
    with _system(1, v, 600) as wf:
        wf.set_ladder_batch(40)
        ref = wf.construct_omega()
        assert _runs_int8(wf, lambda: wf.construct_omega(copy_out=False))
        _fail_an_allocation(wf, v)
        wf.set_ladder_batch(40)
        om = wf.construct_omega()
        assert not _runs_int8(wf, lambda: wf.construct_omega(copy_out=False))
        assert np.abs(om - ref).max() < 1e-12 * np.abs(ref).max()


def test_captured_passes_after_it():
    """Transformations whose captured launches hold the workspace's address run again without it."""
    v = 520
    with _system(2, v, 600) as wf:
        wf.set_ladder_batch(40)
        wf.prepare_for_jacobian()
        assert _runs_int8(wf, lambda: wf.jacobian_transformation(np.ones(wf.n_gs_amplitudes)))
        x = np.random.default_rng(0).normal(size=wf.n_gs_amplitudes)
        r = [wf.jacobian_transformation(x) for _ in range(2)]
        assert np.array_equal(r[0], r[1])
        _fail_an_allocation(wf, v)
        wf.set_ladder_batch(40)
        wf.prepare_for_jacobian()
        q = [wf.jacobian_transformation(x) for _ in range(3)]
        assert np.array_equal(q[0], q[1]) and np.array_equal(q[0], q[2])
        assert np.abs(q[0] - r[0]).max() < 1e-12 * np.abs(r[0]).max()


def test_a_failed_allocation_is_reported_once():
    """It is an error of its own call; the next launch does not report it again."""
    v = 520
    with _system(1, v, 3) as wf:
        wf.set_ladder_batch(40)
        ref = wf.construct_omega()
        _fail_an_allocation(wf, v)
        wf.set_ladder_batch(40)
        assert np.array_equal(wf.construct_omega(), ref)
