"""Every variant of the resident kernels (state, trial moves and lists in LDS or
in global memory, every solver, both precisions) and the scalar-coupling form of
the colour pass, bit for bit against the launched kernels, which an asked-for
launch shape selects."""
import numpy as np
import pytest

import uppasd_amd as U
from uppasd_amd import batch as Bt
from uppasd_amd import configs as CF

pytestmark = pytest.mark.gpu
I32, PAIR = 0x20000, 0x1000000


def _crystal(L, shells):
    return CF.bcc_shells(L, shells, moment=2.2)


def _circulant(n, reach):
    """Every site bonded to its `reach` nearest on both sides of a ring."""
    d = np.concatenate([np.arange(1, reach + 1), -np.arange(1, reach + 1)])
    nl = ((np.arange(n)[:, None] + d) % n + 1).astype(np.int32)
    return dict(nlist=nl, nlistsize=np.full(n, 2 * reach, np.int32),
                ncoup=np.broadcast_to(1.0 / np.abs(d), (n, 2 * reach)).copy(),
                mmom=np.full(n, 1.7))


def _ragged():
    """A random graph, 1 to 6 bonds a site and a coupling of its own each."""
    N, rng = 301, np.random.default_rng(5)
    adj = [set() for _ in range(N)]
    for i in range(N):
        for j in rng.integers(0, N, 2):
            if j != i and len(adj[i]) < 6 and len(adj[j]) < 6:
                adj[i].add(int(j))
                adj[j].add(i)
    W = max(len(a) for a in adj)
    nl, nc = np.zeros((N, W), np.int32), np.zeros((N, W))
    for i, a in enumerate(adj):
        nl[i, :len(a)] = np.array(sorted(a)) + 1
        nc[i, :len(a)] = 5.0 * rng.normal(size=len(a))
    return dict(nlist=nl, nlistsize=np.array([len(a) for a in adj], np.int32), ncoup=nc,
                mmom=rng.uniform(0.5, 2.5, N))


def _film():
    s = CF.triangular_dmi((13, 11, 1))
    N, rng = s["lattice"].natom, np.random.default_rng(3)
    s["taniso"] = rng.choice([0, 1, 2, 7], size=N).astype(np.int32)
    s["eaniso"], s["kaniso"] = CF.random_unit(N, rng)[0], rng.normal(size=(N, 2))
    s["sb"] = rng.normal(size=N)
    return s


def _engine(s, M, precision, order=1):
    N = s["nlistsize"].shape[0]
    eng = U.Engine(N, M, precision, site_order=order)
    eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
    if "dmlist" in s:
        eng.set_dm(s["dmlist"], s["dmlistsize"], s["dm_vect"])
    if "taniso" in s:
        eng.set_anisotropy(s["taniso"], s["eaniso"], s["kaniso"], s["sb"])
    mm = s["mmom"] if "mmom" in s else np.full(N, 2.2)
    eng.set_moments(CF.random_unit(N, np.random.default_rng(N), M), np.broadcast_to(mm, (M, N)))
    return eng, N


# LDS of 160 KB: 2000 sites hold spins and trial moves but not their lists, 2574
# spins and lists but not the moves, 4394 (FP64) the spins alone; with 58
# neighbours the lists of 1024 sites do not fit beside FP64 spins and moves
MC = {
    "sites2000": lambda: _crystal((10, 10, 10), [1.34, 0.77]),
    "sites2574": lambda: _crystal((9, 11, 13), [1.34, 0.77]),
    "sites4394": lambda: _crystal((13, 13, 13), [1.34, 0.77]),
    "shells5_1024": lambda: _crystal((8, 8, 8), CF.bcc5_couplings()),
    "shells5_432": lambda: _crystal((6, 6, 6), CF.bcc5_couplings()),
}


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("mode", ["M", "H"])
@pytest.mark.parametrize("name", list(MC))
def test_resident_sweeps(name, mode, precision, order):
    s, M, out = MC[name](), 3, []
    for shape in (None, (4, 64), (8, 128 | I32)):
        eng, N = _engine(s, M, precision, order)
        eng.set_external_field(np.array([4.0, -3.0, 9.0]))
        if shape:
            eng.set_tuning(eng.TUNE_MC, *shape)
        eng.mc_sweeps(mode, np.array([150.0, 600.0, 1500.0]), 4, 9)
        c = eng.launch_counts()
        assert (c["mc_resident"], c["mc_colour"]) == ((0, 4 * eng.coloring()[0]) if shape
                                                      else (1, 0))
        out.append(eng.get_moments()[0])
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


# 512 FP64 (FP32) sites leave room for lists of 112 (136) neighbours
LLG = {
    "circulant140": lambda: _circulant(512, 70),
    "circulant110": lambda: _circulant(512, 55),
    "ragged": _ragged,
    "film": _film,
    "shells5": lambda: _crystal((5, 6, 7), CF.bcc5_couplings()),
}


@pytest.mark.parametrize("alg", [1, 4, 5, 6, 7])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("name", list(LLG))
def test_resident_steps(name, precision, alg):
    """Also with a damping, a temperature and a g factor of each site's own, and
    (the crystal) in both device site orders."""
    s, M, out = LLG[name](), 2, []
    rng = np.random.default_rng(11)
    n = s["nlistsize"].shape[0]
    lam, temp, g = rng.uniform(0.05, 0.3, n), rng.uniform(0.0, 400.0, n), rng.uniform(0.9, 1.2, n)
    ext = rng.normal(size=(M, n, 3)) * 20.0
    orders = (1, 2) if name == "shells5" else (1,)
    for order in orders:
        for shape in (None, (4, 64)):
            eng, N = _engine(s, M, precision, order)
            if shape:
                eng.set_tuning(eng.TUNE_LLG, *shape)
            eng.set_external_field(ext)
            eng.set_noise(U.UASD_NOISE_PHILOX, 7)
            eng.set_llg(0.1, 300.0, 1e-16)
            eng.sd_steps(alg, 20)
            eng.set_llg(lam, temp, 1e-16, landeg=g)
            eng.sd_steps(alg, 7)
            c = eng.launch_counts()
            assert (c["llg_resident"], c["llg_list"]) == ((0, 54) if shape else (2, 0))
            out.append(eng.get_moments()[0])
    for e in out[1:]:
        assert np.array_equal(e, out[0])


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("mode", ["M", "H"])
def test_colour_pass_with_scalar_couplings(mode, precision):
    """One site class and more than 131,072 (site, ensemble) pairs: the colour
    pass reads its couplings through the scalar cache, one and two ensembles a
    thread, against the same crystal beside a chain of another class."""
    s = dict(_crystal((33, 32, 32), [1.34, 0.77]))
    n, M, out = s["nlistsize"].shape[0], 4, []
    i = np.arange(4)
    chain = dict(nlist=np.stack([(i + 1) % 4, (i - 1) % 4], axis=1).astype(np.int32) + 1,
                 nlistsize=np.full(4, 2, np.int32), ncoup=np.full((4, 2), 3.0), mmom=np.ones(4))
    for systems, shape in (([s, chain], (4, 256)), ([s], (4, 256)), ([s], (8, 64 | PAIR)),
                           ([s], (2, 128 | PAIR | I32))):
        j = Bt.join(systems)
        eng = Bt.engine_for(j, M, precision)
        e = CF.random_unit(j.natom, np.random.default_rng(1), M)
        e[:, :n] = CF.random_unit(n, np.random.default_rng(2), M)
        eng.set_moments(e, np.broadcast_to(j.mmom, (M, j.natom)))
        eng.set_tuning(eng.TUNE_MC, *shape)
        eng.mc_sweeps(mode, np.linspace(200.0, 900.0, M), 2, 5)
        out.append(eng.get_moments()[0][:, :n])
    for e in out[1:]:
        assert np.array_equal(e, out[0])


def test_no_room_for_resident_tables():
    """On a device filled after a context's set-up, systems whose resident tables
    find no room are launched, with the same results."""
    import ctypes as C
    import re
    s = Bt.join([_circulant(512, 70) for _ in range(32)])       # lists of 4.6 MB
    out = []
    for full in (False, True):
        eng = Bt.engine_for(s, 1, "fp64")
        eng.set_moments(CF.random_unit(s.natom, np.random.default_rng(3), 1), s.mmom[None])
        eng.set_llg(0.1, 0.0, 1e-16)
        eng.field(with_energy=True)
        hip = C.CDLL(re.search(r"\S*libamdhip64\.so\S*", open("/proc/self/maps").read()).group(0))
        held, size = [], 1 << 35 if full else 0
        try:
            while size >= 1 << 21:
                p = C.c_void_p()
                if hip.hipMalloc(C.byref(p), C.c_size_t(size)) == 0:
                    held.append(p)
                else:
                    hip.hipGetLastError()
                    size //= 2
            eng.sd_steps(5, 12)
            c = eng.launch_counts()
            out.append(eng.get_moments()[0])
        finally:
            for p in held:
                hip.hipFree(p)
        assert (c["llg_resident"], c["llg_list"]) == ((0, 24) if full else (1, 0))
    assert np.array_equal(out[0], out[1])
