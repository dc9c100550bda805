"""Contexts on several threads: different contexts may be used at the same
time, whatever launch limits their kernels share.

The dynamic LDS limit of a kernel belongs to the process, so a context whose
systems need little LDS must not take it from one whose systems need much."""
import ctypes as C
import re
import threading

import numpy as np
import pytest

import uppasd_amd as U
from uppasd_amd import configs as CF

pytestmark = pytest.mark.gpu


def _in_threads(jobs):
    """Runs every job in a thread of its own, all at once; results in order."""
    out, errs = [None] * len(jobs), []
    start = threading.Barrier(len(jobs))

    def go(k):
        try:
            start.wait()
            out[k] = jobs[k]()
        except Exception as ex:   # reported by the test's own thread
            errs.append(ex)
    ts = [threading.Thread(target=go, args=(k,)) for k in range(len(jobs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errs, errs
    return out


def _engine(L, shells):
    s = CF.bcc_shells(L, shells, moment=2.2)
    N = s["lattice"].natom
    eng = U.Engine(N, 1)
    eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
    eng.set_moments(CF.random_unit(N, np.random.default_rng(N), 1), s["mmom"][None])
    eng.set_llg(0.1, 300.0, 1e-16)
    eng.set_noise(U.UASD_NOISE_PHILOX, 5)
    return eng


def _sweeps(L):
    eng = _engine(L, [1.34, 0.77])
    for _ in range(150):
        eng.mc_sweeps("M", 400.0, 1, 3)
    return eng.get_moments()[0]


def _steps(L):
    eng = _engine(L, CF.bcc5_couplings())
    for _ in range(150):
        eng.sd_steps(1, 2)
    return eng.get_moments()[0]


@pytest.mark.parametrize("run,sizes", [
    (_sweeps, ((10, 10, 10), (3, 3, 3), (6, 5, 4), (12, 9, 10))),   # 2 to 133 KB of LDS
    (_steps, ((6, 6, 6), (3, 3, 3), (5, 5, 5), (4, 4, 4))),         # 11 to 91 KB
])
def test_contexts_of_different_lds_needs_in_threads(run, sizes):
    want = [run(L) for L in sizes]
    got = _in_threads([lambda L=L: run(L) for L in sizes])
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


def test_tile_shapes_in_threads():
    """Two lattices of one tile kernel with different halos and threads (their
    workgroups per CU differ), resident workgroups looping over units."""
    def run(L, shape):
        s = CF.bcc_shells(L, CF.bcc5_couplings(), moment=2.2)
        N = s["lattice"].natom
        eng = U.Engine(N, 1, site_order=2)
        eng.set_lattice_dims(2, *L)
        eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
        eng.set_moments(CF.random_unit(N, np.random.default_rng(N), 1), s["mmom"][None])
        eng.set_llg(0.1, 300.0, 1e-16)
        eng.set_noise(U.UASD_NOISE_PHILOX, 5)
        eng.set_tuning(eng.TUNE_LLG, 4, 256 | (shape << 18) | 0x400000)
        assert eng.llg_tile() == shape
        for _ in range(60):
            eng.sd_steps(1, 1)
        return eng.get_moments()[0]
    sizes = [((16, 16, 16), 8), ((18, 17, 16), 9), ((16, 16, 16), 9), ((18, 17, 16), 8)]
    want = [run(*a) for a in sizes]
    got = _in_threads([lambda a=a: run(*a) for a in sizes])
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


def _hip_calls():
    """Ordinary calls of a program's other threads, which HIP refuses while any
    stream of the process is being captured."""
    hip = C.CDLL(re.search(r"\S*libamdhip64\.so\S*", open("/proc/self/maps").read()).group(0))
    buf, host = C.c_void_p(), (C.c_char * 4096)()
    assert hip.hipMalloc(C.byref(buf), C.c_size_t(4096)) == 0

    def malloc():
        p = C.c_void_p()
        return hip.hipMalloc(C.byref(p), C.c_size_t(1 << 16)) or hip.hipFree(p)
    return {"device": hip.hipDeviceSynchronize, "malloc": malloc,
            "copy": lambda: hip.hipMemcpy(buf, host, C.c_size_t(4096), 1),
            "legacy": lambda: hip.hipStreamSynchronize(None)}


@pytest.mark.parametrize("asked", [0, 64])
@pytest.mark.parametrize("call", ["device", "malloc", "copy", "legacy"])
def test_other_threads_calls_while_graphs_are_built(call, asked):
    """Steps that are replayed, asked for or not, neither fail nor make another
    thread's calls fail while their graphs are built."""
    def run(graph):
        n = 1000
        i = np.arange(n)
        nl = np.stack([(i + 1) % n, (i - 1) % n], axis=1).astype(np.int32) + 1
        eng = U.Engine(n, 1)
        eng.set_exchange(nl, np.full(n, 2, np.int32), np.full((n, 2), 3.0))
        eng.set_moments(CF.random_unit(n, np.random.default_rng(3), 1), np.ones((1, n)))
        eng.set_noise(U.UASD_NOISE_PHILOX, 7)
        if graph:
            eng.set_graph_steps(asked)
        else:
            eng.set_kernel_timing(True)
        for k in range(12):
            eng.set_llg(0.1, 100.0 + k, 1e-16)       # the graph of the last turn is stale
            eng.sd_steps(5, 2048 if not asked else 64)
            eng.sd_steps(5, 128)
        assert (eng.launch_counts()["llg_graph"] > 0) == graph
        return eng.get_moments()[0]

    want = run(False)
    hip_call, stop, codes = _hip_calls()[call], threading.Event(), set()

    def other():
        while not stop.is_set():
            codes.add(hip_call())
    t = threading.Thread(target=other)
    t.start()
    try:
        got = run(True)
    finally:
        stop.set()
        t.join()
    assert np.array_equal(got, want)
    assert codes == {0}


def test_replays_in_threads():
    """Contexts on four threads whose steps and sweeps are replayed, their graphs
    built and dropped side by side."""
    def run(n, alg):
        i = np.arange(n)
        nl = np.stack([(i + 1) % n, (i - 1) % n], axis=1).astype(np.int32) + 1
        eng = U.Engine(n, 1)
        eng.set_exchange(nl, np.full(n, 2, np.int32), np.full((n, 2), 3.0))
        eng.set_moments(CF.random_unit(n, np.random.default_rng(n), 1), np.ones((1, n)))
        eng.set_noise(U.UASD_NOISE_PHILOX, 7)
        eng.set_graph_steps(16)
        for k in range(20):
            eng.set_llg(0.1, 100.0 + k, 1e-16)
            eng.sd_steps(alg, 40)
            eng.mc_sweeps("M", 400.0, 20, k)
        return eng.get_moments()[0]
    jobs = [(1000, 5), (777, 1), (20000, 4), (12000, 5)]
    want = [run(*a) for a in jobs]
    got = _in_threads([lambda a=a: run(*a) for a in jobs])
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
