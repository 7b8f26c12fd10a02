"""Workloads this engine is timed on: Monte-Carlo blocks of every potential
and layout users run, the heat-capacity analysis of finished runs, and the
potential functions called on configurations the caller holds.

A Monte-Carlo pass is a block of production cycles followed by the read-back
of the states (and, in FP64, of the counters and energy sums), as a program
that checkpoints or logs its ladders does.  Start configurations are fcc
fragments with thermal displacements, one per temperature, made from the seed
alone; no cycles run before the first pass, so that every pass starts from
states that do not depend on the code that is timed.
"""
import json
import math
import pathlib
import sys

import numpy as np
import torch

ROOT = pathlib.Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "paralleltemperingmontecarlo.jl_amd"))

import paralleltemperingmontecarlo as pt  # noqa: E402
from paralleltemperingmontecarlo import multihist, nnp_setup  # noqa: E402

GOLDEN = ROOT / "tests" / "golden"
A2B = 1.8897259886
P_ATM = 101325 / 2.9421015697e13  # 1 atm in Hartree / bohr^3
R_CU = 14 * A2B                   # container of the copper runs
D_CU, D_NE = 2.55 * A2B, 3.08 * A2B  # nearest-neighbour distances
LJ = (-4.0, 0.0, 0.0, 4.0)
# Sutton-Chen constants of the embedded-atom tests (n, m, eps, C, a)
EAM = (8.482, 4.692, 0.0367493 * 0.0370, 27.561, 0.25 * 18.8973)


def listed():
    return [
        # one extended-LJ neon ladder in FP64 with the engine's default layout:
        # the first run every user makes (latency of a single small ladder)
        dict(name="ne13_ladder_f64", kind="elj", atoms=13, temps=32, cycles=200),
        # 512 independent LJ ladders of 13-98 atoms, binary32, spread over the
        # chip: the throughput workload of the benchmark
        dict(name="lj_batch_f32", kind="lj", runs=512, lo=13, hi=98, cycles=100),
        # periodic bulk neon, one ladder: constant pressure, and the largest
        # constant-volume box, each configuration on a wave of its own
        dict(name="ne108_npt_f32", kind="bulk", atoms=108, temps=48, npt=True, cycles=20),
        dict(name="ne256_nvt_f32", kind="bulk", atoms=256, temps=48, npt=False, cycles=20),
        # copper with the Behler-Parrinello network: one ladder (a user's
        # study), many ladders (throughput), and clusters above 64 atoms
        dict(name="cu55_nnp_ladder", kind="nnp", atoms=55, temps=40, runs=1, cycles=2),
        dict(name="cu55_nnp_batch", kind="nnp", atoms=55, temps=40, runs=32, cycles=1),
        dict(name="cu78_nnp_ladder", kind="nnp", atoms=78, temps=20, runs=1, cycles=2),
        # two-species brass cluster with atom swaps (NNVT), FP64
        dict(name="brass55_nnvt_f64", kind="brass", n1=50, n2=5, temps=10, cycles=2),
        # copper with the embedded-atom potential, one FP64 ladder
        dict(name="cu55_eam_f64", kind="eam", atoms=55, temps=32, cycles=10),
        # heat capacities from the histograms of finished runs: the ladders of
        # a constant-volume batch, one constant-pressure ladder
        dict(name="heat_capacity_nvt", kind="cv", runs=16, temps=32, bins=100),
        dict(name="heat_capacity_npt", kind="cp", runs=1, temps=48, bins=100),
        # the network's energy_update! on a ladder that the caller's own
        # program holds (one trial per replica)
        dict(name="cu55_energy_update", kind="update", atoms=55, confs=40),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["elj", "lj", "bulk", "nnp", "nnp", "brass", "eam", "cv", "cp", "update"])
    if kind == "elj":
        return dict(kind=kind, atoms=rng.randint(7, 55), temps=rng.randint(8, 32), cycles=rng.randint(20, 100))
    if kind == "lj":
        return dict(kind=kind, runs=_log(rng, 16, 400), lo=rng.randint(7, 13), hi=rng.randint(38, 98),
                    cycles=rng.randint(20, 100))
    if kind == "bulk":
        return dict(kind=kind, atoms=rng.choice([32, 64, 108, 125, 216, 256]), temps=rng.randint(8, 48),
                    npt=rng.random() < 0.5, cycles=rng.randint(5, 20))
    if kind == "nnp":
        atoms = rng.randint(13, 100)
        return dict(kind=kind, atoms=atoms, temps=rng.randint(5, 40), runs=_log(rng, 1, 24 if atoms <= 64 else 6),
                    cycles=1)
    if kind == "brass":
        n2 = rng.randint(2, 12)
        return dict(kind=kind, n1=rng.randint(10, 55 - n2), n2=n2, temps=rng.randint(4, 40), cycles=1)
    if kind == "eam":
        return dict(kind=kind, atoms=rng.randint(13, 64), temps=rng.randint(8, 32), cycles=rng.randint(3, 10))
    if kind == "cv":
        return dict(kind=kind, runs=_log(rng, 1, 64), temps=rng.randint(8, 48), bins=rng.randint(40, 200))
    if kind == "cp":
        return dict(kind=kind, runs=_log(rng, 1, 4), temps=rng.randint(8, 48), bins=rng.randint(30, 100))
    return dict(kind=kind, atoms=rng.randint(13, 64), confs=_log(rng, 4, 64))


# ------------------------------------------------------------------ inputs


def _fcc_cluster(gen, n, d):
    """The n fcc sites nearest to a random point, neighbours d apart, centred."""
    a = d * math.sqrt(2.0)
    m = int(math.ceil((n / 4) ** (1.0 / 3.0))) + 2
    g = np.arange(-m, m + 1)
    cells = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 1, 3)
    base = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])
    sites = (cells + base).reshape(-1, 3) * a
    r2 = ((sites - gen.uniform(-0.25, 0.25, 3) * a) ** 2).sum(1)
    x = sites[np.argsort(r2, kind="stable")[:n]]
    return x - x.mean(0)


def _thermal(gen, x, d, temps):
    """One copy per temperature with displacements growing as sqrt(T), at most
    5 % of the neighbour distance a component."""
    s = 0.05 * d * np.sqrt(np.asarray(temps) / max(temps))
    return x[None] + gen.uniform(-1.0, 1.0, (len(temps),) + x.shape) * s[:, None, None]


def _bulk_start(n, d):
    """fcc for 4 k^3 atoms, simple cubic for k^3, at the same density."""
    length = (n * d**3 / math.sqrt(2.0)) ** (1.0 / 3.0)
    k = round((n / 4) ** (1.0 / 3.0))
    base = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])
    if 4 * k**3 != n:
        k, base = round(n ** (1.0 / 3.0)), np.zeros((1, 3))
    g = np.arange(k)
    cells = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 1, 3)
    x = (cells + base).reshape(-1, 3) * (length / k)
    return x - x.mean(0), length


def _ne_coeff():
    return json.loads((GOLDEN / "ne13_setup.json").read_text())["coeff"]


def _cu_potential(atoms):
    """The benchmark's 8 + 80 functions for clusters of one CU slot, the
    reference's Cu potential for larger ones."""
    d = GOLDEN / "nnp"
    if atoms > 64:
        return nnp_setup.reference_cu55_potential(d / "scaling.data", d / "weights.029.data")
    return nnp_setup.synthetic_cu55_potential(d / "scaling.data")


def _brass(n1, n2):
    d = GOLDEN / "nnp"
    setup = dict(json.loads((GOLDEN / "nnp2_brass.json").read_text()), n1=n1, n2=n2)
    return nnp_setup.reference_brass_potential(setup, d / "scaling.data", d / "weights.029.data",
                                               d / "weights.030.data")


def _ladders(case, seed):
    """Everything a Monte-Carlo case is made of: potential, ensemble, runs
    (atoms, beta, start configurations, container, lanes), engine options."""
    gen = np.random.default_rng(seed)
    kind = case["kind"]
    o = dict(precision="fp32", exchange="even_odd", seed=1000 + seed % 1000, recompute_every=1000)
    runs = []
    if kind == "elj":
        n, grid = case["atoms"], pt.TempGrid(4.0, 16.0, case["temps"])
        bc = pt.SphericalBC(radius=5.32 * A2B * (n / 13) ** (1.0 / 3.0) + 0.5 * D_NE * (n > 13))
        runs.append((n, grid.beta_grid, _thermal(gen, _fcc_cluster(gen, n, D_NE), D_NE, grid.t_grid), bc, 0))
        pot, ens, o = pt.ELJPotentialEven(_ne_coeff()), pt.NVT(n), dict(o, precision="fp64", max_displ=(0.4, 0.1))
    elif kind == "lj":
        # sizes of the batch by the case alone; lanes per configuration as the
        # autotuner chooses them by atom count
        sizes = np.random.default_rng(case["runs"])
        for _ in range(case["runs"]):
            n, r = int(sizes.integers(case["lo"], case["hi"] + 1)), int(sizes.integers(24, 65))
            t = 0.05 * 10.0 ** (np.arange(r) / (r - 1))
            x = _thermal(gen, _fcc_cluster(gen, n, 1.12), 1.12, t)
            lanes = 2 if n < 24 else 4 if n < 48 else 8 if n < 64 else 16 if n < 88 else 32
            runs.append((n, 1.0 / t, x, pt.SphericalBC(radius=1.2 * n ** (1.0 / 3.0) + 0.3), lanes))
        pot, ens = pt.ELJPotentialEven(LJ), pt.NVT(13)
        o = dict(o, workgroup_lanes=64, spread_streams=3, max_displ=(0.15, 0.1))
    elif kind == "bulk":
        n, grid = case["atoms"], pt.TempGrid(10.0, 40.0, case["temps"])
        x, length = _bulk_start(n, D_NE)
        runs.append((n, grid.beta_grid, _thermal(gen, x, D_NE, grid.t_grid), pt.CubicBC(length), 64))
        pot, ens = pt.ELJPotentialEven(_ne_coeff()), pt.NPT(n, P_ATM) if case["npt"] else pt.NVT(n)
        o = dict(o, workgroup_lanes=64, max_displ=(0.4, 0.02))
    elif kind in ("nnp", "eam"):
        n, grid = case["atoms"], pt.TempGrid(200.0, 1400.0, case["temps"])
        for _ in range(case.get("runs", 1)):
            x = _thermal(gen, _fcc_cluster(gen, n, D_CU), D_CU, grid.t_grid)
            runs.append((n, grid.beta_grid, x, pt.SphericalBC(radius=R_CU), 0))
        ens, o = pt.NVT(n), dict(o, max_displ=(0.25, 0.1))
        if kind == "eam":
            pot, o = pt.EmbeddedAtomPotential.from_constants(*EAM), dict(o, precision="fp64")
        else:
            pot = _cu_potential(n)
    else:
        n, grid = case["n1"] + case["n2"], pt.TempGrid(250.0, 900.0, case["temps"])
        x = gen.permutation(_fcc_cluster(gen, n, D_CU))
        runs.append((n, grid.beta_grid, _thermal(gen, x, D_CU, grid.t_grid), pt.SphericalBC(radius=R_CU), 0))
        pot, ens = _brass(case["n1"], case["n2"]), pt.NNVT.of([case["n1"], case["n2"]], natomswaps=2)
        o = dict(o, precision="fp64", exchange="reference", max_displ=(0.25, 0.1))
    return pot, ens, runs, o


def _histograms(case, gen):
    """Energy (and volume) histograms of 10^5 samples a temperature, drawn
    from the canonical distributions of a harmonic cluster, on the bins the
    sampling uses."""
    temps, nb, runs = case["temps"], case["bins"], case["runs"]
    grid = pt.TempGrid(5.0, 16.0, temps) if case["kind"] == "cv" else pt.TempGrid(10.0, 40.0, temps)
    kt = pt.kB * grid.t_grid
    shape = 18.0 if case["kind"] == "cv" else 45.0  # degrees of freedom / 2
    hist, lims = [], []
    for _ in range(runs):
        e0 = -5.6e-3 * gen.uniform(0.9, 1.1)
        lo, hi = e0 + kt[0] * shape * 0.4, e0 + kt[-1] * shape * 1.9
        e = lo + (np.arange(nb) + 0.5) * (hi - lo) / nb - e0
        logp = (shape - 1) * np.log(e)[None] - e[None] / kt[:, None]
        p = np.exp(logp - logp.max(1, keepdims=True))
        p /= p.sum(1, keepdims=True)
        if case["kind"] == "cv":
            h = np.zeros((temps, nb + 2))
            h[:, 1:-1] = [gen.multinomial(100_000, q) for q in p]
            lims.append((lo, hi, 0.0, 0.0))
        else:
            v0 = 16000.0 * gen.uniform(0.95, 1.05)
            v = 0.8 + (np.arange(nb) + 0.5) * 1.2 / nb
            w = np.exp(-0.5 * ((v[None] - 1.0 - 0.25 * grid.t_grid[:, None] / 40.0) / 0.04) ** 2)
            w /= w.sum(1, keepdims=True)
            h = np.zeros((temps, nb + 2, nb + 2))
            h[:, 1:-1, 1:-1] = [gen.multinomial(100_000, np.outer(a, b).ravel()).reshape(nb, nb)
                                for a, b in zip(p, w)]
            lims.append((lo, hi, 0.8 * v0, 2.0 * v0))
        hist.append(h)
    return grid, np.array(hist), np.array(lims)


def _trials(case, seed):
    gen = np.random.default_rng(seed)
    n, c = case["atoms"], case["confs"]
    x = _thermal(gen, _fcc_cluster(gen, n, D_CU), D_CU, np.geomspace(200.0, 1400.0, c))
    index = gen.integers(0, n, c)
    trial = x[np.arange(c), index] + gen.uniform(-0.15, 0.15, (c, 3))
    return x, index.astype(np.int32), trial


def prepare(case, seed):
    if case["kind"] in ("cv", "cp"):
        grid, hist, lims = _histograms(case, np.random.default_rng(seed))
        runs = case["runs"]
        return dict(case=case, t=[grid.t_grid] * runs, beta=np.tile(grid.beta_grid, (runs, 1)), hist=hist, lims=lims)
    if case["kind"] == "update":
        x, index, trial = _trials(case, seed)
        plug = pt.PotentialPlugin(_cu_potential(case["atoms"]), pt.NVT(case["atoms"]), pt.SphericalBC(radius=R_CU))
        en, ea, v = plug.initialise_energy(x)
        return dict(case=case, plug=plug, x=x, index=index, trial=trial, en=en, ea=ea, vars=v)
    pot, ens, runs, o = _ladders(case, seed)
    mc = pt.MCParams(1_000_000, len(runs[0][1]), runs[0][0], n_adjust=100, mc_sample=1, n_bin=100)
    eng = pt.PTEngine(pot, ens, runs[0][3], mc, pt.EngineOptions(**o))
    for k, (n, beta, x0, bc, lanes) in enumerate(runs):
        eng.add_run(n, beta, x0, bc, pressure=P_ATM if case.get("npt") else 0.0, lanes=lanes, run_key=k)
    eng.prepare()
    for k, (_, _, _, bc, _) in enumerate(runs):
        e = eng.energies(k)
        s = float(e.max() - e.min()) + 1e-3 * abs(float(e[0]))
        v = 0.0 if isinstance(bc, pt.SphericalBC) else pt.get_volume(bc)
        eng.set_histogram(k, float(e.min()) - s, float(e.max()) + s, 0.8 * v, 2.0 * v + (v == 0.0))
    eng.start_phase(True)
    return dict(case=case, eng=eng, runs=len(runs), cycles=case["cycles"], f64=o["precision"] == "fp64")


# -------------------------------------------------------------------- runs


def run(state):
    case = state["case"]
    if case["kind"] == "cv":
        cv, _, fe, it = multihist.multihistogram_nvt_batch(
            state["t"], state["beta"], state["hist"], state["lims"][:, 0], state["lims"][:, 1], case["bins"], 1e-9)
        return dict(cv=cv, free_energy=fe, iterations=it)
    if case["kind"] == "cp":
        l = state["lims"]
        cp, _, mom, fe, it = multihist.multihistogram_npt_batch(
            state["t"], state["beta"], state["hist"], l[:, 0], l[:, 1], l[:, 2], l[:, 3],
            [P_ATM] * case["runs"], case["bins"], 1e-9)
        return dict(cp=cp, moments=mom, free_energy=fe, iterations=it)
    if case["kind"] == "update":
        en, v, ea = state["plug"].energy_update(state["x"], state["index"], state["trial"], state["en"],
                                                state["vars"], en_atom=state["ea"])
        return dict(energy=en, features=v, atoms=ea)
    eng = state["eng"]
    eng.cycles(state["cycles"])
    eng.sync()
    got = [eng.state(k) for k in range(state["runs"])]
    out = dict(x=np.concatenate([g[0].ravel() for g in got]), energy=np.concatenate([g[1] for g in got]))
    if case.get("npt"):
        out["box"] = np.concatenate([np.ravel(g[2]) for g in got])
    if state["f64"]:
        ctr = [eng.counters(k) for k in range(state["runs"])]
        for key in ("max_displ", "ham", "count_atom", "count_vol", "count_exc"):
            out[key] = np.concatenate([c[key] for c in ctr])
    return out


def work(case):
    """Arithmetic of one pass; the bytes are the inputs and outputs of the call."""
    kind = case["kind"]
    if kind in ("cv", "cp"):
        bins = case["bins"] ** (2 if kind == "cp" else 1)
        hist = (case["bins"] + 2) ** (2 if kind == "cp" else 1)
        # per (temperature, bin): the histogram, the two sums of one iteration
        # of the fixed point (tens of iterations, of which 50 are counted),
        # and the ten output temperatures' moments
        return dict(bytes=8.0 * case["runs"] * case["temps"] * (hist + 30),
                    flops=case["runs"] * case["temps"] * bins * (50 * 4.0 + 10 * 8.0))
    if kind == "update":
        n, c = case["atoms"], case["confs"]
        tri, nf = (n - 1) * (n - 2) / 2, 31 if n > 64 else 88
        return dict(bytes=8.0 * c * n * (2 * 88 + 8), flops=c * (2 * tri * (40 + 6.0 * nf) + 2.0 * n * 2180))
    if kind == "lj":
        n, t = (case["lo"] + case["hi"]) / 2, 44.0 * case["runs"]
        move = 24.0 * (n - 1)
    else:
        n = case["n1"] + case["n2"] if kind == "brass" else case["atoms"]
        t = float(case["temps"] * case.get("runs", 1))
        tri = (n - 1) * (n - 2) / 2
        if kind == "elj":
            move = 38.0 * (n - 1)
        elif kind == "bulk":
            move = 38.0 * (n - 1) + (19.0 * (n - 1) / 2 if case["npt"] else 0.0)
        elif kind == "eam":
            # a distance, a logarithm and two exponentials (20 each) per new
            # pair, the four updates and a square root per partner
            move = 80.0 * (n - 1)
        else:
            # old and new term of every triangle of the moved atom at its three
            # corners, about a quarter of them inside the cut-off, and the
            # network of every atom
            nf = 80 if kind == "nnp" and n <= 64 else 26
            move = 0.25 * 2 * tri * (40 + 6.0 * nf) + 2.0 * n * 2180
    return dict(bytes=2 * 8.0 * t * (3 * n + 4), flops=case["cycles"] * t * n * move)


def tolerance(case):
    kind = case["kind"]
    if kind in ("elj", "eam", "brass"):
        # FP64 chains: against the 64-bit restatement below energies differ by
        # up to 3e-15 and no decision does; sums in another order add a few
        # 1e-15 per cycle
        return dict(rel=1e-11, max=1e-9, differ=0.0)
    if kind in ("cv", "cp"):
        # measured 3e-12 on the heat capacities: exponentials of arguments of
        # some hundreds (1e-13 each), amplified by <E^2> - <E>^2
        return dict(rel=2e-11, max=1e-9, differ=0.0)
    if kind == "update":
        # measured 1e-15; sums in another order and exponentials of products
        return dict(rel=1e-12, max=1e-10, differ=0.0)
    # binary32 chains: a rounding in another order now and then flips a
    # Metropolis decision, after which that configuration walks its own way
    # (start positions one unit in the last place apart: 1e-7 to 1e-2 on the
    # single ladders, with coordinates up to 0.15 root mean squares apart)
    return dict(rel=2e-2, max=0.9)


# --------------------------------------------------------- 64-bit references


def _philox(c0, c1, c2, c3, seed):
    """Philox4x32-10 of counter arrays, as four uint32 arrays."""
    c = [np.broadcast_to(np.asarray(v, np.uint64), np.broadcast(c0, c1, c2, c3).shape).copy() for v in (c0, c1, c2, c3)]
    k0, k1, m32 = seed & 0xFFFFFFFF, seed >> 32, np.uint64(0xFFFFFFFF)
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & m32, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & m32]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c


def _u53(hi, lo):
    return ((hi << np.uint64(21)) | (lo >> np.uint64(11))).astype(np.float64) * 2.0**-53


def _chain(energy, x, beta, radius, cycles, seed, delta, exchange, swaps=0, n1=0):
    """The Monte-Carlo cycles of one ladder in plain numpy: moves, Metropolis,
    replica exchange, energy sums (all temperatures at once, temperature order;
    step sizes stay, the passes are shorter than the adaptation interval or
    adapt below)."""
    x, en = x.copy(), energy(x)
    r, n = x.shape[:2]
    rows, steps = np.arange(r), n + swaps
    md = np.tile(np.asarray(delta, float), (r, 1))
    win, atom = np.zeros(r, np.int64), np.zeros((r, 2), np.int64)
    vol, exc, ham = np.zeros((r, 2), np.int64), np.zeros((r, 2), np.int64), np.zeros((r, 2))
    temp = np.arange(r, dtype=np.uint64)
    for cyc in range(cycles):
        for m in range(steps):
            def words(sub):
                return _philox(np.uint64(m), np.uint64(cyc), (np.uint64(sub) << np.uint64(20)) | temp, np.uint64(0), seed)

            a, b = words(0), words(1)
            w = (a[1] & np.uint64(0x7FF)) | ((a[3] & np.uint64(0x7FF)) << np.uint64(11)) | \
                ((b[1] & np.uint64(0x3FF)) << np.uint64(22))
            idx = ((w * np.uint64(steps)) >> np.uint64(32)).astype(np.int64)
            met, sw = _u53(b[2], b[3]), idx >= n
            i = np.where(sw, 0, idx)
            tx = x.copy()
            u = np.stack([_u53(a[0], a[1]), _u53(a[2], a[3]), _u53(b[0], b[1])], 1)
            t = x[rows, i] + (u - 0.5) * md[:, :1]
            for k in range(1, 49):
                out = ((t * t).sum(1) > radius * radius) & ~sw
                if not out.any():
                    break
                a, b = words(2 * k), words(2 * k + 1)
                u = np.stack([_u53(a[0], a[1]), _u53(a[2], a[3]), _u53(b[0], b[1])], 1)
                t = np.where(out[:, None], x[rows, i] + (u - 0.5) * md[:, :1], t)
            else:
                return None  # a recentred configuration: not restated here
            tx[rows, i] = np.where(sw[:, None], tx[rows, i], t)
            if sw.any():
                s = words(254)
                p = ((s[0] * np.uint64(n1)) >> np.uint64(32)).astype(np.int64)
                q = n1 + ((s[1] * np.uint64(n - n1)) >> np.uint64(32)).astype(np.int64)
                for k in np.nonzero(sw)[0]:
                    tx[k, [p[k], q[k]]] = x[k, [q[k], p[k]]]
            new = energy(tx)
            with np.errstate(over="ignore"):
                ok = (new <= en) | (np.exp(-(new - en) * beta) >= met)
            x[ok], en = tx[ok], np.where(ok, new, en)
            atom[:, 0] += ok & ~sw
            win += ok & ~sw
            vol[:, 0] += ok & sw
            vol[:, 1] += sw
        if exchange == "even_odd":
            pairs = range(cyc & 1, r - 1, 2)
        else:
            e = _philox(np.uint64(0), np.uint64(cyc), np.uint64(1 << 28), np.uint64(0), seed)
            pairs = [int((int(e[2]) * (r - 1)) >> 32)] if _u53(e[0], e[1]) < 0.1 else []
        for k in pairs:
            e = _philox(np.uint64(1 + k), np.uint64(cyc), np.uint64(1 << 28), np.uint64(0), seed)
            exc[[k, k + 1], 0] += 1
            if min(1.0, math.exp(min(0.0, (beta[k] - beta[k + 1]) * (en[k] - en[k + 1])))) > _u53(e[0], e[1]):
                exc[[k, k + 1], 1] += 1
                x[[k, k + 1]], en[[k, k + 1]] = x[[k + 1, k]], en[[k + 1, k]]
        if (cyc + 1) % 100 == 0:
            share = win / (100.0 * n)
            md[:, 0] *= np.where(share < 0.4, 0.9, np.where(share > 0.6, 1.1, 1.0))
            win[:] = 0
        ham[:, 0] += en
        ham[:, 1] += en * en
    atom[:, 1] = win
    return dict(x=x.ravel(), energy=en, max_displ=md, ham=ham, count_atom=atom, count_vol=vol, count_exc=exc)


def _d2(x):
    d = x[:, :, None] - x[:, None]
    return (d * d).sum(-1)


def _pair_energy(coeff):
    def energy(x):
        iu = np.triu_indices(x.shape[1], 1)
        u = 1.0 / _d2(x)[:, iu[0], iu[1]]
        return sum(c * u ** (k + 3) for k, c in enumerate(coeff)).sum(1)
    return energy


def _eam_energy(x):
    n, m, eps, c, a = EAM
    iu = np.triu_indices(x.shape[1], 1)
    h = 0.5 * np.log(_d2(x)[:, iu[0], iu[1]])
    out = []
    for p in (n, m):
        f = np.zeros(x.shape[:2] + (x.shape[1],))
        f[:, iu[0], iu[1]] = np.exp(-p * h)
        out.append((f + f.transpose(0, 2, 1)).sum(2))
    return (eps * a**n / 2 * out[0] - eps * c * a ** (m / 2) * np.sqrt(out[1])).sum(1)


class _Network:
    """Symmetry functions and networks in torch FP64: one species (tables of
    RuNNerPotential) or two (RuNNerPotential2Atom)."""

    def __init__(self, pot):
        self.two = isinstance(pot, pt.RuNNerPotential2Atom)
        self.rad, self.ang = pot.tables()
        self.rc, self.n1 = pot.r_cut, pot.n1 if self.two else None
        self.nets = [pot.nnp1, pot.nnp2] if self.two else [pot.nnp]
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")

    def features(self, x):
        x = torch.as_tensor(x, dtype=torch.float64, device=self.dev)
        n = x.shape[1]
        d = x[:, None] - x[:, :, None]  # [conf, centre, neighbour, xyz]
        r2 = (d * d).sum(-1)
        r = r2.sqrt()
        off = ~torch.eye(n, dtype=torch.bool, device=self.dev)
        f = torch.where((r < self.rc) & off, 0.5 * (torch.cos(math.pi * r / self.rc) + 1.0), torch.zeros_like(r))
        cos = torch.matmul(d, d.transpose(-1, -2).contiguous()) / (r[:, :, :, None] * r[:, :, None, :])
        w = f[:, :, :, None] * f[:, :, None, :] * f[:, None, :, :]
        w = torch.where(off[None, None], w, torch.zeros_like(w))
        keep = w != 0.0
        cos = torch.where(keep, cos, torch.zeros_like(cos))
        s3 = r2[:, :, :, None] + r2[:, :, None, :] + r2[:, None]
        sp = torch.zeros(n, dtype=torch.long, device=self.dev)
        if self.two:
            sp[self.n1:] = 1
        ns = 2 if self.two else 1
        cols = []
        for row in self.rad:
            g = f * torch.exp(-row[0] * r2)
            for b in range(ns):
                v = g[:, :, sp == b].sum(2)
                if self.two:
                    cols.append(v * self._at(row[1:5], sp, 2, b) + self._at(row[5:9], sp, 2, b))
                else:
                    cols.append(v * row[1] * row[3] + row[2] * row[3])
        last, ex = None, None
        for row in self.ang:
            if row[0] != last:
                last, ex = row[0], w * torch.exp(-row[0] * s3)
            g = ex * (1.0 + row[1] * cos) ** int(row[2])
            if not self.two:
                cols.append(0.5 * g.sum((2, 3)) * row[3] * row[5] + row[4] * row[5])
                continue
            for b, (p, q) in enumerate(((0, 0), (0, 1), (1, 1))):
                v = g[:, :, sp == p][:, :, :, sp == q].sum((2, 3)) * (1.0 if p != q else 0.5)
                cols.append(v * self._at(row[3:9], sp, 3, b) + self._at(row[9:15], sp, 3, b))
        return torch.stack(cols, 2), sp

    def _at(self, vals, sp, per, b):
        return torch.as_tensor(vals, device=self.dev)[per * sp + b]

    def atoms(self, g, sp):
        out = torch.zeros(g.shape[:2], dtype=torch.float64, device=self.dev)
        for s, net in enumerate(self.nets):
            h, o = g[:, sp == s], 0
            for k in range(1, len(net.num_nodes)):
                a, b = int(net.num_nodes[k - 1]), int(net.num_nodes[k])
                w = torch.as_tensor(net.parameters[o:o + a * b], device=self.dev).reshape(a, b)
                h = torch.matmul(h, w) + torch.as_tensor(net.parameters[o + a * b:o + a * b + b], device=self.dev)
                h = torch.tanh(h) if int(net.activation_functions[k]) == 2 else h
                o += a * b + b
            out[:, sp == s] = h[..., 0]
        return out

    def energy(self, x):
        return self.atoms(*self.features(x)).sum(1).cpu().numpy()


def _reweight(case, seed):
    """Multihistogram analysis of every run, vectorised over bins."""
    grid, hist, lims = _histograms(case, np.random.default_rng(seed))
    nb, r, npt = case["bins"], case["temps"], case["kind"] == "cp"
    k_b = pt.api.kB_multihist
    t = grid.t_grid[0] * (grid.t_grid[-1] / grid.t_grid[0]) ** (np.arange(10 * r) / (10 * r - 1))
    out, beta, mid = [], grid.beta_grid, np.arange(nb) + 0.5
    for h, (e0, e1, v0, v1) in zip(hist, lims):
        e = e0 + mid * ((e1 - e0) / nb)
        if npt:
            e, v = np.repeat(e, nb), np.tile(v0 + mid * ((v1 - v0) / nb), nb)
            ent, h = e + P_ATM * v, h[:, 1:-1, 1:-1].reshape(r, -1)
        else:
            v, ent, h = np.zeros(nb), e, h[:, 1:-1]
        cnt, tot, fe = h.sum(1), h.sum(0), np.zeros(r)

        def weights():
            z = -beta[:, None] * ent[None] - fe[:, None]
            off = np.maximum(-1e6, z.max(0)) + math.log(1000.0)
            return off, tot / (cnt[:, None] * np.exp(z - off)).sum(0)

        for it in range(1, 1001):
            off, ratio = weights()
            new = np.log((ratio * np.exp(-beta[:, None] * ent[None] - off)).sum(1))
            delta, fe = ((new - fe) ** 2).sum(), new
            if delta < 1e-9:
                break
        off, ratio = weights()
        q = ratio * np.exp(-(1.0 / (pt.kB * t))[:, None] * ent[None] - off)
        q /= q.sum(1, keepdims=True)
        m1 = q @ ent
        c = (q @ ent**2 - m1 * m1) / (k_b * t**2)
        out.append((c, np.stack([q @ e, q @ v, m1], 1), fe, it))
    c, mom, fe, it = (np.array(z) for z in zip(*out))
    if npt:
        return dict(cp=c, moments=mom, free_energy=fe, iterations=it.astype(np.int32))
    return dict(cv=c, free_energy=fe, iterations=it.astype(np.int32))


def exact(case, seed):
    """The same outputs in 64 bits without the engine; None for the binary32
    chains, whose decisions follow binary32 energies."""
    kind = case["kind"]
    if kind in ("cv", "cp"):
        return _reweight(case, seed)
    if kind == "update":
        x, index, trial = _trials(case, seed)
        x[np.arange(len(x)), index] = trial
        net = _Network(_cu_potential(case["atoms"]))
        g = [net.features(x[k:k + 4]) for k in range(0, len(x), 4)]
        v = torch.cat([a for a, _ in g])
        e = net.atoms(v, g[0][1])
        return dict(energy=e.sum(1).cpu().numpy(), features=v.cpu().numpy(), atoms=e.cpu().numpy())
    if kind not in ("elj", "eam", "brass"):
        return None
    pot, _, runs, o = _ladders(case, seed)
    _, beta, x0, bc, _ = runs[0]
    if kind == "brass":
        if case["temps"] > 16:
            return None
        fn, swaps, n1 = _Network(pot).energy, 2, case["n1"]
    else:
        fn, swaps, n1 = _pair_energy(pot.coeff) if kind == "elj" else _eam_energy, 0, 0
    return _chain(fn, x0, beta, bc.radius, case["cycles"], o["seed"], o["max_displ"], o["exchange"], swaps, n1)
