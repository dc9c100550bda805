"""Host arrays in and out of the device quads: site orders, ensembles, both
precisions, the most pairs that pass through pinned memory (16,384) and one
more, and more (site, ensemble) pairs than one transfer takes at a time
(2^22).  Directions and moments come back bit for bit: FP64 values unchanged,
FP32 values rounded once."""
import numpy as np
import pytest

import uppasd_amd as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("N,M,na", [(2, 1, 1), (6, 5, 3), (255, 2, 5), (16384, 1, 1),
                                    (16385, 1, 5), (65536, 65, 2), (4194305, 1, 1)])
def test_moments_round_trip(N, M, na, precision):
    rng = np.random.default_rng(N + M)
    e = rng.normal(size=(M, N, 3))
    mm = rng.uniform(0.5, 2.5, size=(M, N))
    eng = U.Engine(N, M, precision, site_order=na)
    eng.set_moments(e, mm)
    if precision == "fp32":
        e, mm = (a.astype(np.float32).astype(np.float64) for a in (e, mm))
    got, gotM = eng.get_moments()
    assert np.array_equal(got, e)
    assert np.array_equal(gotM, e * mm[..., None])


@pytest.mark.parametrize("N,M,na", [(6, 5, 3), (65536, 65, 2)])
def test_field_of_host_moments(N, M, na):
    rng = np.random.default_rng(N)
    nl = (np.arange(N)[:, None] + 1) % N + 1           # one bond per site, J = 2
    eng = U.Engine(N, M, site_order=na)
    eng.set_exchange(nl.astype(np.int32), np.ones(N, np.int32), np.full((N, 1), 2.0))
    ext = rng.normal(size=(M, N, 3))
    eng.set_external_field(ext)
    eng.set_moments(rng.normal(size=(M, N, 3)), np.ones((M, N)))
    eM = rng.normal(size=(M, N, 3))
    beff, _, b1, b2 = eng.effective_field(eM, parts=True)
    assert np.array_equal(b1, 2.0 * np.roll(eM, -1, axis=1))
    assert np.array_equal(b2, ext)
    assert np.array_equal(beff, b1 + b2)


@pytest.mark.parametrize("precision,per_pair", [("fp64", 96), ("fp32", 48)])
def test_context_holds_three_quads_a_pair(precision, per_pair):
    """A new context's device memory is its three quad arrays: the staging of
    the moments on their way in has no room of its own."""
    import ctypes as C
    import re
    N = 1 << 24
    small = U.Engine(1, 1)                       # the library and its device are up
    hip = C.CDLL(re.search(r"\S*libamdhip64\.so\S*", open("/proc/self/maps").read()).group(0))

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value
    before = free()
    eng = U.Engine(N, 1, precision)
    assert before - free() <= per_pair * N + (16 << 20)
    e = np.random.default_rng(1).normal(size=(1, N, 3)).astype(np.float32).astype(np.float64)
    eng.set_moments(e, np.ones((1, N)))
    assert np.array_equal(eng.get_moments()[0], e)
    small.close()


def test_moments_come_back_from_a_full_device():
    """With too little device memory left for the largest piece of a transfer,
    smaller pieces take it."""
    import ctypes as C
    import re
    N = (1 << 22) + 5
    e = np.random.default_rng(1).normal(size=(1, N, 3))
    warm = U.Engine(N, 1)                              # what the runtime itself allocates
    warm.set_moments(e, np.ones((1, N)))
    warm.get_moments()
    warm.close()
    eng = U.Engine(N, 1)
    eng.set_moments(e, np.ones((1, N)))
    hip = C.CDLL(re.search(r"\S*libamdhip64\.so\S*", open("/proc/self/maps").read()).group(0))
    held = []
    try:
        size = 1 << 35
        while size >= 1 << 24:                         # leaves 16 to 32 MB of it
            p = C.c_void_p()
            if hip.hipMalloc(C.byref(p), C.c_size_t(size)) == 0:
                held.append(p)
            else:
                hip.hipGetLastError()
                size //= 2
        hip.hipFree(held.pop())
        got = eng.get_moments()
    finally:
        for p in held:
            hip.hipFree(p)
    assert np.array_equal(got[0], e) and np.array_equal(got[1], e)
