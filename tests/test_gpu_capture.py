"""Steps that a caller captures into a HIP graph of its own keep working
whatever the context runs between the replays."""
import ctypes as C
import re

import numpy as np
import pytest

import uppasd_amd as U
from uppasd_amd import configs as CF

pytestmark = pytest.mark.gpu


def _hip():
    """The HIP runtime that the library has loaded."""
    maps = open("/proc/self/maps").read()
    return C.CDLL(re.search(r"\S*libamdhip64\.so\S*", maps).group(0))


class _Captured:
    """What fn() enqueues on a context's stream, as a graph."""

    def __init__(self, eng, fn):
        self.hip, self.stream = _hip(), C.c_void_p(eng.stream())
        g, self.exec = C.c_void_p(), C.c_void_p()
        self._ok(self.hip.hipStreamBeginCapture(self.stream, 1))    # thread local
        fn()
        self._ok(self.hip.hipStreamEndCapture(self.stream, C.byref(g)))
        self._ok(self.hip.hipGraphInstantiate(C.byref(self.exec), g, None, None, 0))

    def _ok(self, r):
        assert r == 0, r

    def replay(self):
        self._ok(self.hip.hipGraphLaunch(self.exec, self.stream))


def _engine(precision):
    s = CF.bcc_shells((5, 5, 5), [1.34, 0.77], moment=2.2)      # 250 sites: resident launches
    N = s["lattice"].natom
    eng = U.Engine(N, 2, precision)
    eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
    e = CF.random_unit(N, np.random.default_rng(4), 2)
    mm = np.broadcast_to(s["mmom"], (2, N))
    eng.set_moments(e, mm)
    eng.set_llg(0.1, 300.0, 1e-16)
    eng.set_noise(U.UASD_NOISE_PHILOX, 7)
    return eng, mm


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_captured_steps_between_longer_calls(precision):
    """Three steps captured after a short call, replayed between longer eager
    ones: their deviates' memory is still theirs.  The reference run takes the
    same steps eagerly, setting the counter back by way of another seed."""
    a, mm = _engine(precision)
    b, _ = _engine(precision)
    a.sd_steps(5, 1)
    g = _Captured(a, lambda: a.sd_steps(5, 3))        # steps 1 to 3, not run yet
    b.sd_steps(5, 1)
    e = b.get_moments()[0]
    b.sd_steps(5, 3)
    b.set_moments(e, mm)
    for n in (100, 5, 70):
        a.sd_steps(5, n)
        b.sd_steps(5, n)
        at = 4 + n if n == 100 else at + n            # b's counter
        g.replay()
        e = b.get_moments()[0]
        b.set_noise(U.UASD_NOISE_PHILOX, 8)
        b.set_noise(U.UASD_NOISE_PHILOX, 7)
        b.sd_steps(5, 1)
        b.set_moments(e, mm)
        b.sd_steps(5, 3)
        e = b.get_moments()[0]
        assert np.array_equal(a.get_moments()[0], e), n
        b.sd_steps(5, at - 4)                         # the counter where a's is
        b.set_moments(e, mm)
