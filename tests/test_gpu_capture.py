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


def _chain_engine(n, stream=None):
    """A ring of n sites: too many for resident launches, few enough for replays."""
    i = np.arange(n)
    nl = np.stack([(i + 1) % n + 1, (i - 1) % n + 1], axis=1).astype(np.int32)
    eng = U.Engine(n, 1)
    if stream is not None:
        eng.set_stream(stream)
    eng.set_exchange(nl, np.full(n, 2, np.int32), np.full((n, 2), 3.0))
    eng.set_moments(CF.random_unit(n, np.random.default_rng(3), 1), np.ones((1, n)))
    eng.set_llg(0.1, 300.0, 1e-16)
    eng.set_noise(U.UASD_NOISE_PHILOX, 7)
    return eng


RUNS = {"llg": (1000, lambda e, k: e.sd_steps(5, 64 * k), 32, "llg_list"),
        "mc": (12000, lambda e, k: e.mc_sweeps("M", 400.0, 16 * k, 5), 32, "mc_colour")}


def _stream(kind):
    """A caller's stream: its own, or the legacy stream, which cannot be captured."""
    if kind == "legacy":
        return 1
    s = C.c_void_p()
    assert _hip().hipStreamCreate(C.byref(s)) == 0
    return s.value


@pytest.mark.parametrize("what", list(RUNS))
@pytest.mark.parametrize("kind", ["own", "blocking", "legacy"])
def test_repeats_on_any_stream(kind, what):
    """Steps and sweeps that repeat go on where they would be replayed, on every
    stream a caller may give, with the same results; the context's own stream
    and ordinary ones are replayed."""
    n, run, before, single = RUNS[what]
    ref = _chain_engine(n)
    ref.set_kernel_timing(True)                        # single launches throughout
    eng = _chain_engine(n, None if kind == "own" else _stream(kind))
    for k in (before, 3, 2):
        run(ref, k)
        run(eng, k)
        assert np.array_equal(eng.get_moments()[0], ref.get_moments()[0]), k
    replays = eng.launch_counts()[what + "_graph"]
    assert ref.launch_counts()[what + "_graph"] == 0
    assert replays == 5 or (kind == "legacy" and replays == 0)
    print(kind, what, eng.launch_counts())


def test_another_stream_captured_meanwhile():
    """The calling thread captures the context's own stream for itself while the
    context runs on another: the steps go on, replayed or launched, with the
    same results."""
    what = "llg"
    n, run, before, single = RUNS[what]
    ref = _chain_engine(n)
    ref.set_kernel_timing(True)
    eng = _chain_engine(n)
    hip, own = _hip(), C.c_void_p(eng.stream())
    eng.set_stream(_stream("blocking"))
    for e in (ref, eng):
        run(e, before)
    eng.get_moments()
    assert hip.hipStreamBeginCapture(own, 1) == 0
    run(eng, 1)
    g = C.c_void_p()
    assert hip.hipStreamEndCapture(own, C.byref(g)) == 0
    run(eng, 1)
    for _ in range(2):
        run(ref, 1)
    assert np.array_equal(eng.get_moments()[0], ref.get_moments()[0])
    replays = eng.launch_counts()[what + "_graph"]
    eng.set_stream(_stream("blocking"))
    run(eng, 1)
    run(ref, 1)
    assert eng.launch_counts()[what + "_graph"] == replays + 1
    assert np.array_equal(eng.get_moments()[0], ref.get_moments()[0])


@pytest.mark.parametrize("asked", [0, 64])
def test_settings_changed_while_replays_run(asked):
    """A new temperature right after an asynchronous call ends the graphs that
    call is still replaying; asked for or not, the moments are those of single
    launches."""
    out = []
    for replayed in (True, False):
        eng = _chain_engine(30000)
        if replayed:
            eng.set_graph_steps(asked)
        else:
            eng.set_kernel_timing(True)
        for k in range(4):
            eng.set_llg(0.1, 100.0 * (k + 1), 1e-16)
            eng.sd_steps(5, 2048)
            eng.sd_steps(5, 640)
        n = eng.launch_counts()["llg_graph"]
        assert n == ((4 * 2688 // 64 if asked else 4 * 10) if replayed else 0)
        out.append(eng.get_moments()[0])
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["tile", "resident"])
def test_graphs_of_kernels_with_much_lds(kind, precision):
    """Graph nodes of kernels that ask for more than 64 KB of LDS: the tile
    kernel and resident sweeps, replays against launches."""
    L, shells = ((16, 16, 16), CF.bcc5_couplings()) if kind == "tile" else ((12, 12, 12), [1.34, 0.77])
    s = CF.bcc_shells(L, shells, moment=2.2)
    N, out = s["lattice"].natom, []
    for graph in (0, 4):
        eng = U.Engine(N, 1, precision, site_order=2)
        eng.set_lattice_dims(2, *L)
        eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
        eng.set_moments(CF.random_unit(N, np.random.default_rng(3), 1), s["mmom"][None])
        eng.set_llg(0.1, 300.0, 1e-16)
        eng.set_noise(U.UASD_NOISE_PHILOX, 7)
        eng.set_graph_steps(graph)
        if kind == "tile":
            eng.set_tuning(eng.TUNE_LLG, 4, 256 | (4 << 18) | 0x400000)
            assert eng.llg_tile() == 4
        for k in (4, 9, 3):
            eng.sd_steps(1, k) if kind == "tile" else eng.mc_sweeps("M", 400.0, k, 5)
            eng.measure()
        c = eng.launch_counts()
        assert c["llg_graph"] + c["mc_graph"] == (3 if graph else 0)
        assert (c["llg_tile"] > 0) == (kind == "tile") and (c["mc_resident"] > 0) != (kind == "tile")
        out.append(eng.get_moments()[0])
    assert np.array_equal(out[0], out[1])
