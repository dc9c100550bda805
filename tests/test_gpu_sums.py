"""FP64 sums per (segment, ensemble) at the edges of their chunks of sites.

Segments of 1 to 16,385 sites (a partial chunk, whole ones, many chunks and
few per segment), ensemble counts that divide the workgroup and ones that do
not.  The tolerance is the bound of any summation order: n sums of terms of
at most |x| carry at most n eps sum|x|.
"""
import numpy as np
import pytest

import uppasd_amd as U

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.mark.parametrize("M", [1, 3, 32, 256])
@pytest.mark.parametrize("sizes", [(1, 255, 256, 257, 1023), (16385, 1), (5,) * 300])
def test_segment_sums_at_chunk_edges(sizes, M):
    N = int(np.sum(sizes))
    rng = np.random.default_rng(N + M)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    e = rng.normal(size=(M, N, 3))
    mm = rng.uniform(0.5, 2.5, size=(M, N))
    eng = U.Engine(N, M)
    # bonds i -> i (mod N) + 1: an exchange energy every site takes part in
    nl = (np.arange(N)[:, None] + 1) % N + 1
    J = rng.normal(size=N)
    eng.set_exchange(nl.astype(np.int32), np.ones(N, np.int32), J[:, None])
    eng.set_segments(off)
    eng.set_moments(e, mm)
    ms, en = eng.measure_segments(with_energy=True)
    mom = e * mm[..., None]
    site = -0.5 * J * np.einsum("kij,kij->ki", mom, np.roll(mom, -1, axis=1))
    site = site * (9.274009994e-24 / 2.179872325e-21)
    for s, (a, b) in enumerate(zip(off[:-1], off[1:])):
        tol = (b - a + 4) * EPS * (np.abs(mom[:, a:b]).sum(axis=1) + 1)
        assert np.all(np.abs(ms[s] - mom[:, a:b].sum(axis=1)) <= tol), (s, sizes)
        tol = (b - a + 8) * EPS * 3 * (np.abs(site[:, a:b]).sum(axis=1) + 1)
        assert np.all(np.abs(en[s] - site[:, a:b].sum(axis=1)) <= tol), (s, sizes)
    t = eng.energy_terms().reshape(len(sizes), M, 4)
    n = np.diff(off)[:, None]
    assert np.allclose(t[..., 0] * n, en, rtol=1e-11, atol=1e-13 * np.abs(en).max())
    assert np.array_equal(eng.energy_terms().reshape(t.shape), t)
    whole, ew = eng.measure(with_energy=True)
    tol = (N + 4) * EPS * (np.abs(mom).sum(axis=1) + 1)
    assert np.all(np.abs(whole - mom.sum(axis=1)) <= tol)
    assert np.all(np.abs(ew - site.sum(axis=1)) <= (N + 8) * EPS * 3 * (np.abs(site).sum(axis=1) + 1))
