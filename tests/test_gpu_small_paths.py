"""Paths that a run takes by size or by repetition give the same bits as the
general ones: deviates drawn ahead, replayed steps and sweeps, a class that
comes with the launch, couplings through the scalar cache, resident steps.

Where the path is chosen by size, the reference run joins the system to another
one that moves the whole lattice to the general path (more sites, or a second
class of sites): no bond connects the two and random numbers are keyed by the
site's index, so the first system's trajectory does not change.  Every
comparison is exact: the arithmetic of a site is the same on both paths."""
import numpy as np
import pytest

import uppasd_amd as U
from uppasd_amd import batch as Bt
from uppasd_amd import configs as CF

pytestmark = pytest.mark.gpu


def _chain(n, J=3.0, mom=1.5):
    i = np.arange(n)
    nl = np.stack([(i + 1) % n + 1, (i - 1) % n + 1], axis=1).astype(np.int32)
    return dict(nlist=nl, nlistsize=np.full(n, 2, np.int32), ncoup=np.full((n, 2), J),
                mmom=np.full(n, mom))


def _run(systems, M, precision, steps, alg, temp=300.0):
    j = Bt.join(systems)
    n, N = systems[0]["nlistsize"].shape[0], j.natom
    eng = Bt.engine_for(j, M, precision)
    e = CF.random_unit(N, np.random.default_rng(1), M)
    e[:, :n] = CF.random_unit(n, np.random.default_rng(2), M)
    eng.set_moments(e, np.broadcast_to(j.mmom, (M, N)))
    eng.set_llg(0.1, temp, 1e-16)
    eng.set_noise(U.UASD_NOISE_PHILOX, 7)
    for k in steps:
        eng.sd_steps(alg, k)
    return eng.get_moments()[0][:, :n]


@pytest.mark.parametrize("alg", [1, 4, 5, 6, 7])
@pytest.mark.parametrize("n,M", [(3, 1), (1001, 3), (32768, 1)])
def test_deviates_drawn_ahead(n, M, alg):
    """Up to 32,768 FP64 items: 16 steps' deviates in one launch; calls of 1,
    16, 17 and 5 steps.  The joined run has 33,000 sites more."""
    steps = (1, 16, 17, 5)
    a = _run([_chain(n)], M, "fp64", steps, alg)
    b = _run([_chain(n), _chain(33000)], M, "fp64", steps, alg)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_repeated_steps_replayed(precision):
    """After 2048 steps under unchanged settings the rest of a small run is
    replayed; changed settings start the count again.  Kernel timing keeps the
    reference run on single launches."""
    out = []
    for timed in (False, True):
        s = CF.bcc_shells((7, 7, 7), [1.34, 0.77], moment=2.2)    # 686: not resident
        N = s["lattice"].natom
        eng = U.Engine(N, 2, precision)
        eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
        eng.set_moments(CF.random_unit(N, np.random.default_rng(3), 2), s["mmom"])
        eng.set_llg(0.1, 300.0, 1e-16)
        eng.set_noise(U.UASD_NOISE_PHILOX, 5)
        got = []
        for block in range(26):
            if timed:
                eng.set_kernel_timing(True)
            eng.sd_steps(5, 100)
            if block == 23:
                eng.set_llg(0.1, 150.0, 1e-16)
            got.append(eng.measure(with_energy=True))
            if block >= 20:
                got.append((eng.get_moments()[0],))
        out.append(got)
    for a, b in zip(*out):
        assert all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("mode", ["M", "H"])
def test_repeated_sweeps_replayed(mode):
    """The same for sweeps, after 512 of them; 12,000 FP64 sites are more than
    a resident launch takes."""
    out, n = [], 12000
    for timed in (False, True):
        eng = U.Engine(n, 1)
        s = _chain(n)
        eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
        eng.set_moments(CF.random_unit(n, np.random.default_rng(3), 1), s["mmom"])
        got = []
        for block in range(24):
            if timed:
                eng.set_kernel_timing(True)
            eng.mc_sweeps(mode, 400.0, 25, 11)
            got.append(eng.measure(with_energy=True))
        got.append((eng.get_moments()[0],))
        out.append(got)
    for a, b in zip(*out):
        assert all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("system,alg", [("bcc", 1), ("film", 5)])
@pytest.mark.parametrize("size", ["small", "large"])
def test_one_site_class(system, alg, size, precision):
    """A crystal of one class, below and above 131,072 sites (from there on its
    couplings come through the scalar cache), against the same crystal beside a
    four-site chain of another class."""
    if system == "bcc":
        s = CF.bcc_shells((41, 40, 43) if size == "large" else (5, 4, 7), [1.34, 0.77], moment=2.2)
        other = _chain(4)
    else:
        s = CF.triangular_dmi((381, 357, 1) if size == "large" else (9, 7, 1))
        other = dict(_chain(4), dmlist=np.ones((4, 1), np.int32),
                     dmlistsize=np.zeros(4, np.int32), dm_vect=np.zeros((4, 1, 3)),
                     taniso=np.zeros(4, np.int32), eaniso=np.tile([0.0, 0.0, 1.0], (4, 1)),
                     kaniso=np.zeros((4, 2)), sb=np.zeros(4))
        other["nlist"] = other["nlist"][:, :2]
    s = dict(s, mmom=np.full(s["lattice"].natom, 1.5))
    a = _run([s], 1, precision, (3,), alg)
    b = _run([s, other], 1, precision, (3,), alg)
    assert np.array_equal(a, b)


def _film(L):
    s = CF.triangular_dmi(L)
    N, rng = s["lattice"].natom, np.random.default_rng(3)
    s["taniso"] = rng.choice([0, 1, 2, 7], size=N).astype(np.int32)   # every anisotropy on the path
    s["eaniso"], s["kaniso"] = CF.random_unit(N, rng)[0], rng.normal(size=(N, 2))
    s["sb"] = rng.normal(size=N)
    return s


RESIDENT = {
    "sites1": lambda: _chain(1, J=0.0),
    "sites511": lambda: _chain(511),
    "sites512": lambda: _chain(512),
    "shells5": lambda: CF.bcc_shells((5, 6, 7), CF.bcc5_couplings(), moment=2.2),
    "film": lambda: _film((13, 11, 1)),
}


@pytest.mark.parametrize("noise", ["philox", "injected", "none"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("name", list(RESIDENT))
def test_resident_steps_equal_launched_ones(name, precision, noise):
    """Systems of up to 512 sites, stepped by one workgroup each, alone, twice
    over and beside a chain of 66,000 sites (more than the resident path takes, so
    that run launches every half step), with a per-site external
    field and calls of 1, 70 and 3 steps."""
    small, M = RESIDENT[name](), 2
    n = small["nlistsize"].shape[0]
    rng = np.random.default_rng(23)
    e0, ext0, nrm0 = CF.random_unit(n, rng, M), rng.normal(size=(M, n, 3)) * 30.0, rng.normal(size=(M, n, 3))
    out = []
    for systems in ([small], [small, small], [small, _chain(66000)]):
        systems = [dict(s) for s in systems]
        for s in systems if "dmlist" in small else ():
            k = s["nlistsize"].shape[0]
            for key, v in (("dmlist", np.ones((k, 1), np.int32)), ("dmlistsize", np.zeros(k, np.int32)),
                           ("dm_vect", np.zeros((k, 1, 3))), ("taniso", np.zeros(k, np.int32)),
                           ("eaniso", np.tile([0.0, 0.0, 1.0], (k, 1))), ("kaniso", np.zeros((k, 2))),
                           ("sb", np.zeros(k))):
                s.setdefault(key, v)
        j = Bt.join(systems)
        N = j.natom
        eng = Bt.engine_for(j, M, precision)

        def pad(a, fill):
            full = np.broadcast_to(np.asarray(fill, dtype=np.float64), (M, N, 3)).copy()
            full[:, :n] = a
            return full
        eng.set_moments(pad(e0, [0.0, 0.0, 1.0]), np.broadcast_to(j.mmom, (M, N)))
        eng.set_external_field(pad(ext0, [0.0, 0.0, 5.0]))
        eng.set_llg(0.1, 200.0, 1e-16)
        if noise == "injected":
            eng.set_noise(U.UASD_NOISE_INJECTED, 0, pad(nrm0, 0.0))
        else:
            eng.set_noise(U.UASD_NOISE_PHILOX if noise == "philox" else U.UASD_NOISE_NONE, 9)
        got = []
        for alg in (1, 5, 4):
            for k in (1, 70, 3):
                eng.sd_steps(alg, k)
            got.append(eng.get_moments()[0][:, :n])
        out.append(got)
    for k in range(3):
        assert np.array_equal(out[0][k], out[2][k]), (name, k)
        assert np.array_equal(out[1][k], out[2][k]), (name, k)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", ["list", "tile", "colour"])
def test_asked_for_shapes_are_launched(shape, precision):
    """A launch shape that was set is the one that runs, also on systems small
    enough for resident launches, which run where none was set; with the same
    results."""
    s = CF.triangular_dmi(20)                                # 400 sites, DM + K + B
    N, M, alg, steps = s["lattice"].natom, 2, 5, 6
    temps = [300.0, 900.0]
    out = []
    for asked in (False, True):
        eng = U.Engine(N, M, precision)
        eng.set_lattice_dims(1, *s["lattice"].n)
        eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
        eng.set_dm(s["dmlist"], s["dmlistsize"], s["dm_vect"])
        eng.set_anisotropy(s["taniso"], s["eaniso"], s["kaniso"], s["sb"])
        eng.set_external_field(s["ext"])
        eng.set_moments(CF.random_unit(N, np.random.default_rng(6), M),
                        np.broadcast_to(s["mmom"], (M, N)))
        eng.set_llg(0.1, 200.0, 1e-16)
        eng.set_noise(U.UASD_NOISE_PHILOX, 3)
        if asked and shape == "colour":
            eng.set_tuning(eng.TUNE_MC, 8, 128 | 0x1000000)
        elif asked:
            eng.set_tuning(eng.TUNE_LLG, 4, 256 | ((5 << 18) if shape == "tile" else 0))
        if shape == "colour":
            eng.mc_sweeps("M", temps, steps, 9)
            want = {"mc_colour": steps * eng.coloring()[0]} if asked else {"mc_resident": 1}
        else:
            eng.sd_steps(alg, steps)
            want = {"llg_" + shape: 2 * steps} if asked else {"llg_resident": 1}
        n = {k: v for k, v in eng.launch_counts().items() if v and k != "draw"}
        assert n == want
        if asked and shape != "colour":
            assert eng.llg_tile() == (5 if shape == "tile" else 0)
        out.append(eng.get_moments()[0])
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("kind", ["llg", "mc"])
def test_autotuner_times_what_runs(kind, tmp_path):
    """On small systems the autotuner times the shapes with the kernels they
    belong to and the resident launch beside them; what it keeps is what the
    next call runs, in this context and in one that takes the kept result."""
    s = CF.bcc_shells((6, 6, 6), CF.bcc5_couplings(), moment=2.2)
    N, path = s["lattice"].natom, tmp_path / "tune.txt"

    def make():
        eng = U.Engine(N, 1)
        eng.set_lattice_dims(2, 6, 6, 6)
        eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
        eng.set_moments(CF.random_unit(N, np.random.default_rng(8), 1), s["mmom"][None])
        eng.set_llg(0.1, 300.0, 1e-16)
        eng.set_noise(U.UASD_NOISE_PHILOX, 3)
        return eng

    def tune(eng):
        return eng.autotune_llg(1, steps=4) if kind == "llg" else eng.autotune_mc("M", 400.0, 2)

    def run(eng):
        before = eng.launch_counts()
        eng.sd_steps(1, 4) if kind == "llg" else eng.mc_sweeps("M", 400.0, 2, 9)
        after = eng.launch_counts()
        return {k for k in after if after[k] > before[k] and k != "draw"}, eng.get_moments()[0]

    ref = run(make())
    try:
        U.set_tune_cache(True, str(path))
        a = make()
        ms = tune(a)
        n = a.launch_counts()
        launched = n["llg_list"] + n["llg_tile"] if kind == "llg" else n["mc_colour"]
        assert launched > 0 and n[kind + "_resident"] > 0 and ms > 0.0    # both were timed
        line, = path.read_text().splitlines()
        won = line.split()[0].endswith("/res1")
        assert won or line.split()[0].endswith("/res0")
        b = make()
        assert tune(b) == ms and sum(b.launch_counts().values()) == 0     # taken over, not timed
        for eng in (a, b):
            path_of, e = run(eng)
            assert (path_of == {kind + "_resident"}) == won
            assert won or path_of <= {"llg_list", "llg_tile", "mc_colour"}
            assert np.array_equal(e, ref[1])
            assert kind == "mc" or not (won and eng.llg_tile())
    finally:
        U.set_tune_cache(False)


@pytest.mark.parametrize("L,shells,want", [
    ((7, 7, 7), [1.34, 0.77], (4, 64)),              # small, 14 neighbours
    ((7, 7, 7), CF.bcc5_couplings(), (8, 64)),       # small, 58
    ((64, 64, 32), [1.34, 0.77], (4, 64)),           # 2^18 items: the last small size
    ((64, 64, 33), [1.34, 0.77], (4, 256)),
])
def test_tuning_reports_what_is_launched(L, shells, want):
    s = CF.bcc_shells(L, shells, moment=2.2)
    eng = U.Engine(s["lattice"].natom, 1)
    eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
    assert eng.tuning(eng.TUNE_LLG) == eng.tuning(eng.TUNE_FIELD) == want
    eng.set_tuning(eng.TUNE_LLG, *eng.tuning(eng.TUNE_LLG))
    assert eng.tuning(eng.TUNE_LLG) == want
    eng.set_tuning(eng.TUNE_FIELD, 16, 128)
    assert eng.tuning(eng.TUNE_FIELD) == (16, 128)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [250, 2000])
def test_short_calls_draw_in_the_predictor(n, precision):
    """Calls of one Philox step, or of too few for a launch of their deviates to
    be repaid, and such a rest of a longer call, are half steps that draw for
    themselves; the moments are those of one long call."""
    s = _chain(n)
    out = []
    for calls in ((1, 5, 1, 1, 70, 6), (84,)):
        eng = U.Engine(n, 1, precision)
        eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
        eng.set_moments(CF.random_unit(n, np.random.default_rng(3), 1), s["mmom"][None])
        eng.set_llg(0.1, 300.0, 1e-16)
        eng.set_noise(U.UASD_NOISE_PHILOX, 5)
        for k in calls:
            before = eng.launch_counts()
            eng.sd_steps(5, k)
            c = {key: v - before[key] for key, v in eng.launch_counts().items()}
            if n == 250:        # resident from two steps on, in launches of up to 64
                assert c["llg_list"] == (2 if k == 1 else 0)
                assert c["draw"] == c["llg_resident"] == (0 if k == 1 else (k + 63) // 64)
            else:               # groups of 16 steps, a rest of 6 or more
                assert c["llg_list"] == 2 * k
                assert c["draw"] == (k // 16 + (k % 16 >= 6) if precision == "fp64" else 0)
        out.append(eng.get_moments()[0])
    assert np.array_equal(out[0], out[1])


def _rings(n, R):
    """R rings of n sites (single sites for n = 1)."""
    i = np.arange(n * R)
    b, k = i // n * n, i % n
    nl = np.stack([b + (k + 1) % n, b + (k - 1) % n], axis=1).astype(np.int32) + 1
    return dict(nlist=nl, nlistsize=np.full(n * R, 2 if n > 1 else 0, np.int32),
                ncoup=np.full((n * R, 2), 3.0))


@pytest.mark.parametrize("kind,precision,n,R,M,resident", [
    ("llg", "fp64", 1, 2069, 1, True), ("llg", "fp64", 1, 2070, 1, False),
    ("llg", "fp32", 4, 529, 8, True), ("llg", "fp32", 4, 530, 8, False),
    ("llg", "fp64", 64, 256, 8, True), ("llg", "fp64", 65, 252, 8, False),
    ("llg", "fp64", 32, 510, 8, False),
    ("H", "fp64", 2, 3059, 1, True), ("H", "fp32", 2, 3060, 1, False),
    ("M", "fp64", 4, 1560, 2, True), ("M", "fp64", 4, 1561, 2, False),
    ("M", "fp32", 4, 2341, 4, True), ("M", "fp32", 4, 2342, 4, False),
    ("H", "fp64", 256, 512, 4, True), ("H", "fp64", 64, 2048, 4, False)])
def test_batches_of_many_tiny_systems_are_launched(kind, precision, n, R, M, resident):
    """A system takes a workgroup of at least one wavefront: batches of more
    wavefronts than the rule allows go half step by half step, colour by colour."""
    s = _rings(n, R)
    eng = U.Engine(n * R, M, precision)
    eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
    eng.set_moments(CF.random_unit(n * R, np.random.default_rng(2), M), np.ones((M, n * R)))
    if kind == "llg":
        eng.set_llg(0.1, 300.0, 1e-16)
        eng.set_noise(U.UASD_NOISE_PHILOX, 7)
        eng.sd_steps(5, 8)
    else:
        eng.mc_sweeps(kind, np.full(M, 300.0), 3, 9)
    c = eng.launch_counts()
    ran = c["llg_resident"] if kind == "llg" else c["mc_resident"]
    launched = c["llg_list"] if kind == "llg" else c["mc_colour"]
    assert (ran > 0, launched == 0) == (resident, resident), c


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind,L,M", [("M", (8, 8, 8), 257), ("H", (8, 8, 8), 257),
                                      ("llg", (6, 7, 6), 257)])
def test_more_systems_than_lists_in_lds_allow(kind, L, M, precision):
    """257 systems whose lists would leave one workgroup a CU (256 CUs): the
    lists stay in global memory, the moments are those of the launched kernels."""
    s = CF.bcc_shells(L, CF.bcc5_couplings(), moment=2.2)
    N, out = s["lattice"].natom, []
    for asked in (False, True):
        eng = U.Engine(N, M, precision)
        eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
        eng.set_moments(CF.random_unit(N, np.random.default_rng(2), M),
                        np.broadcast_to(s["mmom"], (M, N)))
        eng.set_llg(0.1, 300.0, 1e-16)
        eng.set_noise(U.UASD_NOISE_PHILOX, 7)
        if asked:
            eng.set_tuning(eng.TUNE_LLG, 8, 64)
            eng.set_tuning(eng.TUNE_MC, 8, 64)
        if kind == "llg":
            eng.sd_steps(1, 5)
        else:
            eng.mc_sweeps(kind, np.linspace(100.0, 1500.0, M), 3, 9)
        c = eng.launch_counts()
        assert (c["llg_resident"] + c["mc_resident"] > 0) != asked
        out.append(eng.get_moments()[0])
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("kind,n,resident", [("M", 1024, True), ("H", 1026, False),
                                             ("llg", 512, True), ("llg", 513, False)])
def test_largest_resident_systems(kind, n, resident):
    """Rings, whose closing bond spans the whole system, at the most sites that
    resident launches take (512 a colour, 512 a half step) and beyond."""
    s = _rings(n, 1)
    eng = U.Engine(n, 1)
    eng.set_exchange(s["nlist"], s["nlistsize"], s["ncoup"])
    eng.set_moments(CF.random_unit(n, np.random.default_rng(2), 1), np.ones((1, n)))
    eng.set_llg(0.1, 300.0, 1e-16)
    eng.set_noise(U.UASD_NOISE_PHILOX, 7)
    eng.sd_steps(5, 8) if kind == "llg" else eng.mc_sweeps(kind, 300.0, 2, 9)
    c = eng.launch_counts()
    assert (c["llg_resident" if kind == "llg" else "mc_resident"] == 1) == resident


@pytest.mark.parametrize("kind", ["llg", "mc"])
def test_tuned_batches_stay_resident(kind):
    """A search over calls of one sweep or three steps, whose resident launches
    are mostly the loading of their systems, does not cost a batch of small
    systems the resident launches of its longer calls."""
    rng = np.random.default_rng(7)
    reps = [CF.bcc_alloy(L, rng.integers(0, 2, 2 * L ** 3)) for L in (5, 6, 7, 5, 6, 7, 5, 6)] \
        if kind == "mc" else [CF.bcc_shells(L, [1.34, 0.77], moment=2.2) for L in (4, 5, 6, 4, 5, 6)]
    j = Bt.join(reps)
    M = 32 if kind == "mc" else 1
    eng = Bt.engine_for(j, M, "fp32")
    eng.set_moments(CF.random_unit(j.natom, rng, M), np.broadcast_to(j.mmom, (M, j.natom)))
    eng.set_llg(0.1, 300.0, 1e-16)
    eng.set_noise(U.UASD_NOISE_PHILOX, 3)
    if kind == "mc":
        eng.autotune_mc("M", np.linspace(200.0, 1600.0, M))
    else:
        eng.autotune_llg(5)
    before = eng.launch_counts()
    eng.mc_sweeps("M", np.linspace(200.0, 1600.0, M), 20, 5) if kind == "mc" else eng.sd_steps(5, 20)
    after = eng.launch_counts()
    assert {k for k in after if after[k] > before[k]} - {"draw"} == {kind + "_resident"}
