"""Performance cases of the spin-update engine: what a program that uses it has it do.

Every case is a run of one of four kinds, through the package's public calls:

  sd       spin dynamics kept on the device: blocks of `steps` LLG steps, the
           averages (moment sum and energy) read after each block, the moments
           at the end
  mc       Monte Carlo sweeps on the device: blocks of `sweeps`, one cumulant
           sample (with energy) per block, the accumulators and the moments at
           the end
  dropin   the host-array halves as a reference driver calls them, every array
           in and out on every call
  observe  the measurement calls on a state that is on the device: field,
           energy and its terms, moment sums

The lattices are the ones of the tests and the benchmark (bcc with two or five
shells, triangular with DM, anisotropy and Zeeman field, kagome batches, random
bcc alloys) with the neighbour lists written out here.  `exact` restates the
arithmetic in FP64 torch, on the same counter-based random numbers.
"""
from __future__ import annotations

import functools
import itertools
import math

import numpy as np
import torch

import uppasd_amd as U

GAMA, KB, MUB, MRY = 1.760859644e11, 1.38064852e-23, 9.274009994e-24, 2.179872325e-21
TESLA = MRY / MUB                       # Tesla per mRy/muB


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest jobs: a unit-test sized crystal, where launches and latency count
        dict(name="sd_bcc6_depondt", kind="sd", lattice="bcc2", n1=6, n2=6, n3=6, M=1,
             precision="fp64", alg=5, temp=300.0, tuned=False, graph=0, blocks=4, steps=50),
        # a few thousand spins, an ensemble average: the everyday relaxation run
        dict(name="sd_bcc12_heun_m3", kind="sd", lattice="bcc5", n1=12, n2=11, n3=13, M=3,
             precision="fp64", alg=4, temp=100.0, tuned=False, graph=0, blocks=4, steps=50),
        # the benchmark's small configuration: bcc 20^3 x 2, two shells, Depondt, 300 K
        dict(name="sd_bcc20_depondt", kind="sd", lattice="bcc2", n1=20, n2=20, n3=20, M=1,
             precision="fp64", alg=5, temp=300.0, tuned=True, graph=0, blocks=5, steps=100),
        # the benchmark's headline: bcc 64^3 x 2, 58 neighbours, midpoint, 300 K
        dict(name="sd_bcc64_midpoint", kind="sd", lattice="bcc5", n1=64, n2=64, n3=64, M=1,
             precision="fp64", alg=1, temp=300.0, tuned=True, graph=0, blocks=8, steps=100),
        # skyrmion-type film: triangular 512^2, J + DM + K + B, T = 0
        dict(name="sd_tri512_depondt", kind="sd", lattice="tri", n1=512, n2=512, n3=1, M=1,
             precision="fp64", alg=5, temp=0.0, tuned=True, graph=0, blocks=5, steps=200),
        # the same film, ragged, in single precision at a finite temperature
        dict(name="sd_tri_ragged_fp32", kind="sd", lattice="tri", n1=691, n2=517, n3=1, M=1,
             precision="fp32", alg=5, temp=10.0, tuned=True, graph=0, blocks=5, steps=200),
        # many kagome systems of uneven size and temperature in one launch, graph replays
        dict(name="sd_kagome_batch_fp32", kind="sd", lattice="kagome", systems=96, lo=24, hi=96,
             M=1, precision="fp32", alg=5, temp=100.0, tuned=True, graph=50, blocks=8, steps=100),
        # bccFe-sized Metropolis run of one ensemble
        dict(name="mc_bcc10_metropolis", kind="mc", lattice="bcc2", n1=10, n2=10, n3=10, M=1,
             precision="fp64", mode="M", tlo=500.0, thi=500.0, tuned=False, graph=0, blocks=10,
             sweeps=20),
        # a temperature scan with heat bath, FP64
        dict(name="mc_bcc20_heatbath_m16", kind="mc", lattice="bcc2", n1=20, n2=18, n3=22, M=16,
             precision="fp64", mode="H", tlo=200.0, thi=1600.0, tuned=True, graph=0, blocks=10,
             sweeps=20),
        # alloy replicas x temperatures in single precision, graph replays
        dict(name="mc_alloy_batch_fp32", kind="mc", lattice="alloy", systems=12, lo=8, hi=24, M=32,
             precision="fp32", mode="M", tlo=200.0, thi=1600.0, tuned=True, graph=10, blocks=80,
             sweeps=20),
        # the drop-in halves under a reference driver
        dict(name="dropin_bcc32_midpoint", kind="dropin", lattice="bcc5", n1=32, n2=32, n3=32, M=1,
             precision="fp64", alg=1, temp=300.0, tuned=False, graph=0, blocks=1, steps=4),
        # measurement of a large state: field, energy, energy terms, moment sums
        dict(name="observe_bcc48", kind="observe", lattice="bcc5", n1=48, n2=48, n3=48, M=1,
             precision="fp64", tuned=False, graph=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same kinds, lattices and ranges; sizes by their logarithm."""
    kind = rng.choice(["sd", "sd", "sd", "sd", "mc", "mc", "dropin", "observe"])
    c = dict(kind=kind, precision=rng.choice(["fp64", "fp64", "fp32"]))
    c["tuned"] = rng.random() < 0.5 and kind in ("sd", "mc")
    c["graph"] = 0
    if kind == "mc":
        c["lattice"] = rng.choice(["bcc2", "bcc5", "alloy"])
    elif kind == "sd":
        c["lattice"] = rng.choice(["bcc2", "bcc5", "bcc5", "tri", "kagome"])
    else:
        c["lattice"] = rng.choice(["bcc2", "bcc5", "tri"])
    c["M"] = rng.choice([1, 1, 1, 2, 3, 4, 8]) if c["lattice"] != "kagome" else 1
    cells = {"sd": 200_000, "mc": 30_000, "dropin": 50_000, "observe": 130_000}[kind]
    cells = _log(rng, 250, cells / c["M"] if c["lattice"] != "bcc5" or kind == "mc" else cells / 2)
    if c["lattice"] in ("alloy", "kagome"):
        c["systems"] = rng.randint(2, 10)
        side = (cells / c["systems"]) ** (1 / 3 if c["lattice"] == "alloy" else 1 / 2)
        c["lo"], c["hi"] = max(5, int(0.6 * side)), max(6, int(1.3 * side))
        c["graph"] = rng.choice([0, 10])
    elif c["lattice"] == "tri":
        c["n1"] = max(5, int(math.sqrt(cells) * rng.uniform(0.7, 1.4)))
        c["n2"], c["n3"] = max(5, cells // c["n1"]), 1
    else:
        c["n1"], c["n2"] = (max(5, int(cells ** (1 / 3) * rng.uniform(0.75, 1.3))) for _ in range(2))
        c["n3"] = max(5, cells // (c["n1"] * c["n2"]))
        if kind == "sd" and c["lattice"] == "bcc5":
            c["M"] = 1 if cells > 20_000 else c["M"]
    if kind == "mc":
        c["M"] = rng.choice([1, 4, 16, 32]) if cells < 4000 else c["M"]
        c.update(mode=rng.choice(["M", "H"]), tlo=200.0, thi=1600.0 if c["M"] > 1 else 200.0,
                 blocks=rng.randint(5, 12), sweeps=20)
    elif kind == "sd":
        c.update(alg=rng.choice([1, 1, 5, 5, 4]), temp=rng.choice([0.0, 100.0, 300.0]),
                 blocks=rng.randint(3, 6), steps=rng.choice([50, 60, 100]))
    elif kind == "dropin":
        c.update(alg=rng.choice([1, 5]), temp=rng.choice([0.0, 300.0]), blocks=1, steps=3)
    return c


# ---------------------------------------------------- lattices and their lists
def _bcc_bonds(shells):
    """(basis, basis', dx, dy, dz, J mRy) of the first shells of bcc."""
    vec = ((0.5, 0.5, 0.5), (1.0, 0.0, 0.0), (1.0, 1.0, 0.0), (1.5, 0.5, 0.5), (1.0, 1.0, 1.0))
    J = [1.34 * math.exp(-1.2 * k) for k in range(5)] if shells == 5 else [1.34, 0.77]
    sign = (1, 1, -1, 1, -1)
    out = []
    for b in (0, 1):
        for k in range(shells):
            for v in sorted({tuple(s * x for s, x in zip(ss, p)) for p in itertools.permutations(vec[k])
                             for ss in itertools.product((1, -1), repeat=3)}):
                r = [x + 0.5 * b for x in v]
                b2 = int(round(2 * r[0])) % 2
                d = [int(round(x - 0.5 * b2)) for x in r]
                out.append((b, b2, *d, J[k] * (sign[k] if shells == 5 else 1)))
    return out


def _list(bonds, na, n1, n2, n3):
    """(N, W) 1-based neighbours, site = b + na*(x + n1*(y + n2*z)), and (na, W) values."""
    W = len(bonds) // na
    x, y, z = (np.arange(n) for n in (n1, n2, n3))
    nl = np.zeros((n3, n2, n1, na, W), dtype=np.int32)
    val = np.zeros((na, W))
    for b in range(na):
        for j, (_, b2, dx, dy, dz, v) in enumerate([t for t in bonds if t[0] == b]):
            cell = (((x + dx) % n1)[None, None, :]
                    + n1 * (((y + dy) % n2)[None, :, None] + n2 * ((z + dz) % n3)[:, None, None]))
            nl[..., b, j] = b2 + na * cell + 1
            val[b, j] = v
    return nl.reshape(-1, W), val


TRI = ((1, 0), (-1, 0), (1, 1), (-1, -1), (0, 1), (0, -1))
KAGOME = ((0, 1, 0, 0), (0, 1, -1, 0), (0, 2, 0, 0), (0, 2, 0, -1), (1, 0, 0, 0), (1, 0, 1, 0),
          (1, 2, 0, 0), (1, 2, 1, -1), (2, 0, 0, 0), (2, 0, 0, 1), (2, 1, 0, 0), (2, 1, -1, 1))


@functools.lru_cache(maxsize=16)
def _model(key):
    """The Hamiltonian of a case: a crystal, or joined systems.  Rows of couplings per basis atom
    (aham) or, for alloys and batches, per site."""
    c = dict(key)
    lat = c["lattice"]
    if lat in ("bcc2", "bcc5"):
        na, dims = 2, (c["n1"], c["n2"], c["n3"])
        nl, J = _list(_bcc_bonds(int(lat[3])), na, *dims)
        m = 2.2
        h = dict(nlist=nl, ncoup=J * 2 * TESLA / m / m, mmom=np.full(nl.shape[0], m))
    elif lat == "tri":
        na, dims = 1, (c["n1"], c["n2"], 1)
        nl, J = _list([(0, 0, dx, dy, 0, 1.0) for dx, dy in TRI], 1, *dims)
        cell = np.array([[1.0, 0.0], [-0.5, math.sqrt(3) / 2]])
        r = np.array([np.array(t) @ cell for t in TRI])
        D = 0.2 * np.stack([-r[:, 1], r[:, 0], np.zeros(6)], axis=1)
        N = nl.shape[0]
        h = dict(nlist=nl, ncoup=J * 2 * TESLA, dm=D[None] * 2 * TESLA, mmom=np.ones(N),
                 kani=TESLA * 0.05, ext=np.array([0.0, 0.0, 0.3 * TESLA]))
    elif lat == "kagome":
        na, dims = 3, None
        sides = [int(round(c["lo"] + (c["hi"] - c["lo"]) * k / (c["systems"] - 1)))
                 for k in range(c["systems"])]
        bonds = [(b, b2, dx, dy, 0, -1.0) for b, b2, dx, dy in KAGOME]
        sign = np.array([[1.0 if (b2 - b) % 3 == 1 else -1.0 for b1, b2, _, _ in KAGOME if b1 == b]
                         for b in range(3)])
        parts, offs, segs = [], [0], [0]
        for s in sides:             # sites of each system sublattice by sublattice: its segments
            nl, J = _list(bonds, 3, s, s, 1)
            cells = s * s
            new = (np.arange(3 * cells) % 3) * cells + np.arange(3 * cells) // 3
            old = np.empty_like(new)
            old[new] = np.arange(3 * cells)
            parts.append(new[nl[old] - 1] + offs[-1] + 1)
            segs += [offs[-1] + (k + 1) * cells for k in range(3)]
            offs.append(offs[-1] + 3 * cells)
        nl = np.concatenate(parts).astype(np.int32)
        aham = np.concatenate([np.repeat(np.arange(3), s * s) for s in sides]).astype(np.int32) + 1
        D = np.zeros((3, 4, 3))
        D[..., 2] = 0.08 * sign
        T = np.logspace(0.0, math.log10(max(c["temp"], 1.001)), c["systems"])
        h = dict(nlist=nl, ncoup=J * 2 * TESLA, dm=D * 2 * TESLA, mmom=np.ones(nl.shape[0]),
                 aham=aham, segments=np.array(segs, dtype=np.int32),
                 temp=np.repeat(T, [3 * s * s for s in sides]))
    else:
        na, dims = 1, None
        rng = np.random.default_rng(4000 + c["systems"])
        Jp = np.array([[1.2, 2.0], [2.0, 0.4]])
        mom = np.array([2.6, 1.7])
        nls, ncs, mms, offs = [], [], [], [0]
        for k in range(c["systems"]):
            s = int(round(c["lo"] + (c["hi"] - c["lo"]) * k / (c["systems"] - 1)))
            nl, _ = _list([t for t in _bcc_bonds(2) if t[5] == 1.34], 2, s, s, s)
            occ = rng.integers(0, 2, nl.shape[0])
            mm = mom[occ]
            ncs.append(Jp[occ[:, None], occ[nl - 1]] * 2 * TESLA / mm[:, None] / mm[nl - 1])
            nls.append(nl + offs[-1])
            mms.append(mm)
            offs.append(offs[-1] + nl.shape[0])
        N = offs[-1]
        h = dict(nlist=np.concatenate(nls).astype(np.int32), ncoup=np.concatenate(ncs),
                 mmom=np.concatenate(mms), aham=np.arange(1, N + 1, dtype=np.int32),
                 segments=np.array(offs, dtype=np.int32))
    N = h["nlist"].shape[0]
    if "aham" not in h:
        h["aham"] = (np.arange(N) % na + 1).astype(np.int32)
    h.update(N=N, na=na, dims=dims, size=np.full(h["ncoup"].shape[0], h["nlist"].shape[1], np.int32))
    return h


def _key(case):
    return tuple(sorted((k, case[k]) for k in ("lattice", "n1", "n2", "n3", "systems", "lo", "hi",
                                               "temp") if k in case
                        and (k != "temp" or case["lattice"] == "kagome")))


def _start(case, N, seed):
    """Starting directions: a thermal tilt about z for Monte Carlo (its equilibrium side), random
    for spin dynamics from a quench."""
    rng = np.random.default_rng(seed)
    v = rng.normal(size=(case["M"], N, 3))
    if case["kind"] == "mc":
        v = 0.5 * v + np.array([0.0, 0.0, 1.0])
    return v / np.linalg.norm(v, axis=2, keepdims=True)


def _temps(case):
    return np.linspace(case["tlo"], case["thi"], case["M"])


LAMBDA, DT = 0.1, 1e-16


# ------------------------------------------------------------- prepare and run
def prepare(case, seed):
    h = _model(_key(case))
    N, M = h["N"], case["M"]
    crystal = case["tuned"] and h["dims"] is not None
    eng = U.Engine(N, M, case["precision"], site_order=h["na"] if crystal else 1)
    if crystal:                         # the two calls that declare a periodic crystal
        eng.set_lattice_dims(h["na"], *h["dims"])
    eng.set_exchange(h["nlist"], h["size"], h["ncoup"], h["aham"])
    if "dm" in h:
        eng.set_dm(h["nlist"], h["size"], h["dm"], h["aham"])
    if "kani" in h:
        eng.set_anisotropy(np.ones(N, np.int32), np.tile([0.0, 0.0, 1.0], (N, 1)),
                           np.tile([h["kani"], 0.0], (N, 1)), np.zeros(N))
        eng.set_external_field(h["ext"])
    if "segments" in h:
        eng.set_segments(h["segments"])
    e = _start(case, N, seed)
    eng.set_moments(e, h["mmom"])
    s = dict(case=case, eng=eng, seed=int(seed))
    if case["kind"] in ("sd", "dropin"):
        temp = h.get("temp", case["temp"])
        eng.set_llg(LAMBDA, temp, DT)
        eng.set_noise(U.UASD_NOISE_PHILOX if np.max(temp) > 0 else U.UASD_NOISE_NONE, seed)
    if case["tuned"]:
        U.set_tune_cache(True)          # winners kept for the process, as a long-lived program does
        if case["kind"] == "sd":
            eng.autotune_llg(case["alg"])
        else:
            eng.autotune_mc(case["mode"], _temps(case))
    if case["graph"]:
        eng.set_graph_steps(case["graph"])
    if case["kind"] == "dropin":
        s["mmom"] = np.ascontiguousarray(np.broadcast_to(h["mmom"], (M, N)))
        s["emom"], s["emom2"] = e, e.copy()
        s["emomM"] = e * s["mmom"][..., None]
        s["b2eff"] = np.zeros_like(e)
    return s


def _own(case, *arrays):
    """The FP32 engine's results in its own precision."""
    return [a.astype(np.float32) if case["precision"] == "fp32" else a for a in arrays]


def run(s):
    case, eng = s["case"], s["eng"]
    kind = case["kind"]
    if kind == "sd":
        av = []
        for _ in range(case["blocks"]):
            eng.sd_steps(case["alg"], case["steps"])
            if case["lattice"] == "kagome":
                av.append(eng.measure_segments(with_energy=True))
            else:
                av.append(eng.measure(with_energy=True))
        out = _own(case, eng.get_moments()[0], np.array([a[0] for a in av]),
                   np.array([a[1] for a in av]))
        return dict(zip(("emom", "msum", "energy"), out))
    if kind == "mc":
        eng.reset_accumulators()
        t = _temps(case)
        for _ in range(case["blocks"]):
            eng.mc_sweeps(case["mode"], t, case["sweeps"], s["seed"])
            eng.accumulate(with_energy=True)
        acc = eng.accumulators()
        out = _own(case, eng.get_moments()[0], *(acc[k] for k in ("m", "m2", "m4", "e", "e2")))
        return dict(zip(("emom", "m", "m2", "m4", "e", "e2"), out))
    if kind == "dropin":
        e, e2, eM, b2, mm = (s[k] for k in ("emom", "emom2", "emomM", "b2eff", "mmom"))
        en = []
        for _ in range(case["steps"]):
            beff, energy = eng.effective_field(eM)
            en.append(energy)
            eng.evolve_first(case["alg"], beff, e, e2, eM, b2)
            beff, _ = eng.effective_field(eM)
            eng.evolve_second(case["alg"], beff, b2, e, e2)
            U.moment_update(mm, e, e2, eM)
        out = _own(case, e, eM, beff, np.array(en))
        return dict(zip(("emom", "emomM", "beff", "energy"), out))
    beff, energy = eng.field()
    terms = eng.energy_terms()
    msum, en = eng.measure(with_energy=True)
    out = _own(case, beff, np.array(energy), terms, msum, en)
    return dict(zip(("beff", "energy", "terms", "msum", "energies"), out))


# ----------------------------------------------------------------------- work
def work(case):
    """Per LLG step every spin is read and written once and its field summed twice over its W
    neighbours; per sweep every spin is read and written and its field summed once."""
    h = _model(_key(case))
    N, W = h["N"] * case["M"], h["nlist"].shape[1]
    s = 8 if case["precision"] == "fp64" else 4
    term = 6 if "dm" not in h else 18
    if case["kind"] == "sd":
        n = case["blocks"] * case["steps"]
        return dict(bytes=float(n * N * 6 * s), flops=float(n * N * 2 * (term * W + 100)))
    if case["kind"] == "mc":
        n = case["blocks"] * case["sweeps"]
        return dict(bytes=float(n * N * 6 * s), flops=float(n * N * (term * W + 100)))
    if case["kind"] == "dropin":        # 14 vectors of every step cross between host and device
        n = case["steps"]
        return dict(bytes=float(n * N * 3 * 8 * 14), flops=float(n * N * 2 * (term * W + 100)))
    return dict(bytes=float(N * 3 * (8 + s)), flops=float(N * (term * W + 30)))


# ---------------------------------------------------------------------- exact
def _philox(site, ens, step, tag, seed, dev):
    """Philox4x32-10 words of counter (site, ens, step, tag), key seed, as int64 tensors (M, N)."""
    mask = 0xFFFFFFFF
    c = [site[None, :].expand(len(ens), -1), ens[:, None].expand(-1, len(site)),
         torch.full((1, 1), step & mask, dtype=torch.int64, device=dev),
         torch.full((1, 1), (tag & 0xFF) | ((step >> 32) << 8), dtype=torch.int64, device=dev)]
    k0, k1 = seed & mask, (seed >> 32) & mask
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [((p1 >> 32) & mask) ^ c[1] ^ k0, p1 & mask, ((p0 >> 32) & mask) ^ c[3] ^ k1, p0 & mask]
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    return c


class _Exact:
    """The Hamiltonian in FP64 torch."""

    def __init__(self, case, seed):
        h = _model(_key(case))
        self.case, self.h, self.seed = case, h, int(seed)
        self.dev = dev = "cuda" if torch.cuda.is_available() else "cpu"
        t = functools.partial(torch.as_tensor, dtype=torch.float64, device=dev)
        self.N, self.M, self.W = h["N"], case["M"], h["nlist"].shape[1]
        self.nb = torch.as_tensor(np.ascontiguousarray(h["nlist"].T) - 1, dtype=torch.int64, device=dev)
        row = torch.as_tensor(h["aham"] - 1, dtype=torch.int64, device=dev)
        self.J = t(h["ncoup"])[row].T.contiguous()                        # (W, N)
        self.D = t(h["dm"])[row].transpose(0, 1).contiguous() if "dm" in h else None
        self.m = t(h["mmom"])
        self.ext = t(h["ext"]) if "ext" in h else None
        # the FP32 engine is given these numbers rounded
        r32 = (lambda x: x.float().double()) if case["precision"] == "fp32" else (lambda x: x)
        self.e = r32(t(_start(case, self.N, seed)))
        self.site = torch.arange(self.N, device=dev)
        self.ens = torch.arange(self.M, device=dev)
        self.numpy = lambda x: x.cpu().numpy()

    def terms(self, e):
        """(exchange, DM, uniaxial, external) fields, each (M, N, 3)."""
        mom = e * self.m[:, None]
        ex, dm = torch.zeros_like(e), torch.zeros_like(e)
        for j in range(self.W):
            g = mom[:, self.nb[j]]
            ex += self.J[j][:, None] * g
            if self.D is not None:
                dm += torch.linalg.cross(g, self.D[j].expand_as(g))
        an = torch.zeros_like(e)
        if "kani" in self.h:
            an[..., 2] = -2.0 * self.h["kani"] * mom[..., 2]
        x = torch.zeros_like(e) if self.ext is None else self.ext.expand_as(e)
        return ex, dm, an, x

    def field(self, e):
        return sum(self.terms(e))

    def energy(self, e):
        """Field-routine energy per ensemble and site, mRy."""
        ex, dm, an, x = self.terms(e)
        return -((e * self.m[:, None]) * (0.5 * (ex + dm + an) + x)).sum(-1) * (MUB / MRY)

    def normals(self, step):
        """Thermal deviates (M, N, 3) of one step: Box-Muller on 52-bit (FP64 engine) or 32- and
        23-bit uniforms (FP32 engine)."""
        w = _philox(self.site, self.ens, step, 0x11, self.seed, self.dev)
        if self.case["precision"] == "fp64":
            x = _philox(self.site, self.ens, step, 0x12, self.seed, self.dev)
            u = [(((a << 20) | (b >> 12)).double() + 0.5) * 2.0 ** -52
                 for a, b in ((w[0], w[1]), (w[2], w[3]), (x[0], x[1]), (x[2], x[3]))]
            r0, r1, v0, v1 = u[0], u[1], u[2], u[3]
        else:
            r0, r1 = ((w[k].double() + 0.5) * 2.0 ** -32 for k in (0, 2))
            v0, v1 = ((2 * (w[k] >> 9) + 1).double() * 2.0 ** -24 for k in (1, 3))
        r0, r1 = torch.sqrt(-2.0 * torch.log(r0)), torch.sqrt(-2.0 * torch.log(r1))
        v0, v1 = 2 * math.pi * v0, 2 * math.pi * v1
        return torch.stack([r0 * torch.cos(v0), r0 * torch.sin(v0), r1 * torch.cos(v1)], dim=-1)

    def llg_step(self, e, step):
        """(new directions, field of the start, predicted directions, field of those)."""
        c, m = self.case, self.m[:, None]
        T = torch.as_tensor(self.h.get("temp", c["temp"]), dtype=torch.float64, device=self.dev)
        T = T.expand(self.N)[:, None]
        n = self.normals(step) if float(T.max()) > 0 else torch.zeros_like(e)
        damp = 1.0 / (1.0 + LAMBDA ** 2)
        cross = lambda a, b: torch.linalg.cross(a, b.expand_as(a))  # noqa: E731
        b0 = self.field(e)
        if c["alg"] == 1:
            r = n * torch.sqrt(2.0 * LAMBDA * damp * KB / MUB / m * T)
            dtm = DT * GAMA * damp

            def half(p, b):
                a = 0.5 * dtm * (-b - LAMBDA * cross(p, b)) + 0.5 * math.sqrt(dtm) * (-r - LAMBDA * cross(p, r))
                rhs = e + cross(e, a)
                aa = (a * a).sum(-1, keepdim=True)
                return (rhs + a * (a * rhs).sum(-1, keepdim=True) + cross(rhs, a)) / (1.0 + aa)
            p = 0.5 * (e + half(e, b0))
            b1 = self.field(p)
            return half(p, b1), b0, p, b1
        if c["alg"] == 5:
            r = n * torch.sqrt(2.0 * LAMBDA * KB / (DT * GAMA * MUB) * T / m)

            def turn(bd):
                norm = torch.sqrt((bd * bd).sum(-1, keepdim=True)) + 1e-15
                k, v = bd / norm, norm * DT * GAMA * damp
                return (k * (k * e).sum(-1, keepdim=True) * (1 - torch.cos(v)) + torch.cos(v) * e
                        + torch.sin(v) * cross(k, e))
            d0 = b0 + r + LAMBDA * cross(e, b0 + r)
            p = turn(d0)
            b1 = self.field(p)
            return turn(0.5 * (b1 + r + LAMBDA * cross(p, b1 + r)) + 0.5 * d0), b0, p, b1
        w = n * torch.sqrt(DT * GAMA * 2.0 * LAMBDA * damp * KB / MUB / m * T)     # Heun
        dtg = DT * GAMA * damp

        def drift(v, b):
            return LAMBDA * b + cross(b, v) - v * (v * LAMBDA * b).sum(-1, keepdim=True)

        def noise(v, quirk):
            o = LAMBDA * w - LAMBDA * v * (v * w).sum(-1, keepdim=True) + cross(w, v)
            if quirk:                   # the corrector's zz element is -vz*vz
                o[..., 2] += (LAMBDA * v[..., 2] ** 2 - v[..., 2] ** 2 - LAMBDA) * w[..., 2]
            return o
        p = e + drift(e, b0) * dtg + noise(e, False)
        b1 = self.field(p)
        o = e + 0.5 * ((drift(p, b1) + drift(e, b0)) * dtg + noise(p, True) + noise(e, False))
        return o / torch.sqrt((o * o).sum(-1, keepdim=True)), b0, p, b1

    def sums(self, e):
        """Moment sums and energies per (segment, ensemble), or per ensemble."""
        mom, en = e * self.m[:, None], self.energy(e)
        if "segments" not in self.h:
            return self.numpy(mom.sum(1)), self.numpy(en.sum(1))
        off = self.h["segments"]
        ms = torch.stack([mom[:, a:b].sum(1) for a, b in zip(off[:-1], off[1:])])
        return self.numpy(ms), self.numpy(torch.stack([en[:, a:b].sum(1) for a, b in zip(off[:-1], off[1:])]))

    def colours(self):
        """Greedy colouring in site order of the (symmetric) bond graph."""
        col = [-1] * self.N
        for i, row in enumerate((self.h["nlist"] - 1).tolist()):
            used = {col[n] for n in row}
            k = 0
            while k in used:
                k += 1
            col[i] = k
        col = np.array(col)
        return [torch.as_tensor(np.nonzero(col == k)[0], device=self.dev) for k in range(col.max() + 1)]

    def sweep(self, e, sweep, colours, T):
        """One FP64 Metropolis sweep in place, colour by colour."""
        u01 = lambda tag, s: [(w.double() + 0.5) * 2.0 ** -32  # noqa: E731
                              for w in _philox(s, self.ens, sweep, tag, self.seed, self.dev)]
        T = T[:, None]
        for s in colours:
            f = torch.zeros(self.M, len(s), 3, dtype=torch.float64, device=self.dev)
            for j in range(self.W):
                n = self.nb[j][s]
                f += (self.J[j][s] * self.m[n])[:, None] * e[:, n]
            u, m, me = u01(0x21, s), self.m[s], e[:, s]
            g = u01(0x22, s)
            r0, r1 = torch.sqrt(-2 * torch.log(g[0])), torch.sqrt(-2 * torch.log(g[2]))
            step = torch.stack([r0 * torch.cos(2 * math.pi * g[1]), r0 * torch.sin(2 * math.pi * g[1]),
                                r1 * torch.cos(2 * math.pi * g[3])], dim=-1)
            delta = float(np.float32(2.0) / np.float32(25.0)) * (KB * T / MUB) ** 0.2
            gauss = me + step * delta[..., None]
            gauss = gauss / torch.sqrt((gauss * gauss).sum(-1, keepdim=True))
            zz, phi = 1 - 2 * u[2], 2 * math.pi * u[1]
            st = torch.sqrt(torch.clamp(1 - zz * zz, min=0.0))
            uni = torch.stack([st * torch.cos(phi), st * torch.sin(phi), zz], dim=-1)
            move = torch.floor(3 * u[0])[..., None]
            trial = torch.where(move == 0, uni, torch.where(move == 1, gauss, -me))
            de = -MUB * m * ((trial - me) * f).sum(-1)
            take = (de <= 0) | (u[3] < torch.exp(-de / KB / (T + 1e-15)))
            e[:, s] = torch.where(take[..., None], trial, me)


def exact(case, seed):
    kind = case["kind"]
    W = {"bcc5": 58, "bcc2": 14, "tri": 12, "kagome": 8, "alloy": 8}[case["lattice"]]
    # single-precision trial moves have no 64-bit counterpart; heat bath carries a rounding
    # difference from sweep to sweep until, within a hundred sweeps, the chains have parted
    if kind == "mc" and (case["precision"] == "fp32" or case["mode"] == "H"):
        return None
    if kind == "sd":
        h = _model(_key(case))
        n = case["blocks"] * case["steps"] * 2 * (W + 25)
        if n * (5e-6 * 6 + h["N"] * case["M"] * 3 * 8 * 4 / 1.5e12) > 20:
            return None
    x = _Exact(case, seed)
    e = x.e
    if kind == "sd":
        av, k = [], 0
        for _ in range(case["blocks"]):
            for _ in range(case["steps"]):
                e = x.llg_step(e, k)[0]
                k += 1
            av.append(x.sums(e))
        return dict(emom=x.numpy(e), msum=np.array([a[0] for a in av]), energy=np.array([a[1] for a in av]))
    if kind == "mc":
        T = torch.as_tensor(_temps(case), device=x.dev)
        colours = x.colours()
        seg = x.h.get("segments", np.array([0, x.N]))
        size, samples = np.diff(seg)[:, None], []
        for b in range(case["blocks"]):
            for k in range(case["sweeps"]):
                x.sweep(e, b * case["sweeps"] + k, colours, T)
            ms, en = x.sums(e)
            ms, en = (ms, en) if "segments" in x.h else (ms[None], en[None])
            m, en = np.linalg.norm(ms, axis=2) / size, en / size
            samples.append((m, m ** 2, m ** 4, en, en ** 2))
        w = np.arange(1, case["blocks"] + 1, dtype=np.float64)      # sample n counts n times
        mean = [np.tensordot(w, np.array(c), 1) / w.sum() for c in zip(*samples)]
        return dict(zip(("emom", "m", "m2", "m4", "e", "e2"), (x.numpy(e), *mean)))
    if kind == "dropin":
        en = []
        for k in range(case["steps"]):
            en.append(float(x.energy(e).sum()))
            e, b0, p, b1 = x.llg_step(e, k)
        return dict(emom=x.numpy(e), emomM=x.numpy(e * x.m[:, None]), beff=x.numpy(b1), energy=np.array(en))
    ex, dm, an, ext = x.terms(e)
    mom = e * x.m[:, None]
    t = [-f * (mom * b).sum((1, 2)) / x.N * (MUB / MRY) for b, f in ((ex, 0.5), (an, 0.5), (dm, 0.5), (ext, 1.0))]
    en = x.energy(e).sum(1)
    return dict(beff=x.numpy(ex + dm + an + ext), energy=np.array(float(en.sum())),
                terms=x.numpy(torch.stack(t, dim=1)), msum=x.numpy(mom.sum(1)), energies=x.numpy(en))
