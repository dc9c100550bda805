"""Small systems swept by one workgroup each (resident launches) against the
same systems swept colour by colour in launches of the whole lattice.

The resident path is taken by size, so the reference run joins the system to a
second one that is too large for it: sites of one system share no bond with the
other's, the random numbers are keyed by the site's index and the greedy
colouring starts with the first system, so the first system's chain is the
same, bit for bit (every update is the same arithmetic)."""
import numpy as np
import pytest

import uppasd_amd as U
from uppasd_amd import batch as Bt
from uppasd_amd import configs as CF

pytestmark = pytest.mark.gpu


def _big():
    """One system of 20,000 sites in a chain: more than LDS holds."""
    N = 20000
    i = np.arange(N)
    nl = np.stack([(i + 1) % N + 1, (i - 1) % N + 1], axis=1).astype(np.int32)
    return dict(nlist=nl, nlistsize=np.full(N, 2, np.int32), ncoup=np.full((N, 2), 3.0),
                mmom=np.ones(N))


def _crystal(n, shells):
    s = CF.bcc_shells(n, shells, moment=2.2)
    return dict(s, mmom=s["mmom"])


def _film(L):
    s = CF.triangular_dmi(L)
    N = s["lattice"].natom
    rng = np.random.default_rng(3)
    s["taniso"] = rng.choice([0, 1, 2, 7], size=N).astype(np.int32)   # every anisotropy on the path
    s["eaniso"] = CF.random_unit(N, rng)[0]
    s["kaniso"] = rng.normal(size=(N, 2))
    s["sb"] = rng.normal(size=N)
    return s


def _ragged():
    """Rows of uneven length: a random graph, 1 to 6 bonds a site."""
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


SYSTEMS = {
    "sites63": lambda: _crystal((3, 3, 3), [1.34]),            # 54 sites: under a wavefront
    "sites500": lambda: _crystal((5, 5, 10), [1.34, 0.77]),    # one round of the workgroup
    "sites2574": lambda: _crystal((9, 11, 13), [1.34, 0.77]),  # FP64 trials beyond LDS
    "shells5": lambda: _crystal((5, 6, 7), CF.bcc5_couplings()),
    "film": lambda: _film((13, 11, 1)),                        # DM, anisotropies
    "ragged": _ragged,
}


@pytest.mark.parametrize("name", list(SYSTEMS))
@pytest.mark.parametrize("mode", ["M", "H"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_resident_sweeps_equal_launched_ones(name, mode, precision):
    small, M = SYSTEMS[name](), 3
    big = _big()
    n = small["nlistsize"].shape[0]
    rng = np.random.default_rng(17)
    temps = np.array([150.0, 600.0, 1500.0])
    ext = rng.normal(size=(M, 1, 3)) * 20.0
    out = []
    for systems in ([small], [small, big], [small, small]):
        if "dmlist" in small:
            for s in systems:
                k = s["nlistsize"].shape[0]
                s.setdefault("dmlist", np.ones((k, 1), np.int32))
                s.setdefault("dmlistsize", np.zeros(k, np.int32))
                s.setdefault("dm_vect", np.zeros((k, 1, 3)))
                s.setdefault("taniso", np.zeros(k, np.int32))
                s.setdefault("eaniso", np.tile([0.0, 0.0, 1.0], (k, 1)))
                s.setdefault("kaniso", np.zeros((k, 2)))
                s.setdefault("sb", np.zeros(k))
        j = Bt.join(systems)
        eng = Bt.engine_for(j, M, precision)
        N = j.natom
        e = CF.random_unit(N, np.random.default_rng(1), M)
        e[:, :n] = CF.random_unit(n, np.random.default_rng(2), M)
        eng.set_moments(e, np.broadcast_to(j.mmom, (M, N)))
        eng.set_external_field(np.broadcast_to(ext, (M, N, 3)))
        eng.set_kernel_timing(True)
        eng.mc_sweeps(mode, temps, 3, 9)
        launches = eng.kernel_timing(3)[0]
        eng.set_kernel_timing(False)
        if len(systems) == 2 and systems[1] is big:
            assert launches == 3 * eng.coloring()[0], name     # a launch per colour and sweep
        else:
            assert launches == 1, name                         # one resident launch
        eng.set_graph_steps(2)
        eng.mc_sweeps(mode, temps, 5, 9)                       # two replays and one sweep
        out.append(eng.get_moments()[0][:, :n])
    assert np.array_equal(out[0], out[1]), name
    assert np.array_equal(out[2], out[1]), name


@pytest.mark.parametrize("mode", ["M", "H"])
def test_resident_fp32_trials_beyond_lds(mode):
    """8192 FP32 sites of 16 colours: the spins alone fill the LDS, the trial
    moves and the lists stay in global memory."""
    SYSTEMS["sites8192"] = lambda: _crystal((16, 16, 16), CF.bcc5_couplings())
    try:
        test_resident_sweeps_equal_launched_ones("sites8192", mode, "fp32")
    finally:
        del SYSTEMS["sites8192"]
