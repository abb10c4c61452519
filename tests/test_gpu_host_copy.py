"""Long vectors read back into pageable memory (et_amd/csrc/host_copy.hpp): lengths around the
staged copy's pieces and ring, fresh and reused destinations, two wavefunctions from two threads."""
import threading

import numpy as np
import pytest

from et_amd import ccsd

pytestmark = pytest.mark.gpu


def _round_trip(o, v, seed, out=None):
    rng = np.random.default_rng(seed)
    with ccsd.CCSD(o, v, 3) as wf:
        for _ in range(2):
            t = rng.normal(size=wf.n_gs_amplitudes)
            wf.set_amplitudes(t)
            ok = np.array_equal(wf.get_amplitudes(), t)
            assert ok
            if out is not None:
                out.append(ok)


# 16 MB and below (runtime's copy), just above, several pieces, more than the ring holds
@pytest.mark.parametrize('o,v', [(7, 70), (32, 63), (32, 64), (23, 101), (30, 152), (31, 200)])
def test_lengths(o, v):
    _round_trip(o, v, o * v)


def test_two_threads():
    out = []
    ts = [threading.Thread(target=_round_trip, args=(30 + k, 90, k, out)) for k in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert out == [True] * 4
