"""A long copy to the host behind queued work: one thread waits for the work."""
import time

import numpy as np
import pytest

from et_amd import ccsd
from et_amd import synthetic as syn

pytestmark = pytest.mark.gpu


def test_host_threads_while_the_device_works():
    o, v, J = 24, 130, 600
    s = syn.system(3, o, v, J, t2_sigma=1e-3, t1_sigma=1e-2, L_scale=0.02)
    with ccsd.CCSD(o, v, J) as wf:
        wf.set_cholesky(s['L'])
        wf.set_oei(s['h'])
        wf.set_amplitudes(np.concatenate([s['t1'].ravel(order='F'), s['t2']]))
        wf.construct_t1_cholesky()
        ref = wf.construct_omega()
        wf.get_omega()                                    # the ring is there
        t0 = time.perf_counter()
        wf.get_omega()
        copy = time.perf_counter() - t0
        for _ in range(30):                               # queued, not waited for
            assert wf._lib.etg_construct_omega_resident(wf._h, ccsd.FP64) == 0
        w0, c0 = time.perf_counter(), time.process_time()
        om = wf.get_omega()
        wall, cpu = time.perf_counter() - w0, time.process_time() - c0
        assert np.array_equal(om, ref)
    print('wait %.1f ms (copy alone %.1f ms), processor time %.1f ms' % (1e3 * wall, 1e3 * copy, 1e3 * cpu), flush=True)
    assert wall > 5 * copy                                # there was something to wait for
    # the waiting thread, at most one of the runtime's own, and the copy by nine threads
    assert cpu < 2 * (wall - copy) + 9 * copy
