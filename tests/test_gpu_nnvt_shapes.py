"""NNVT moves of the two-species network potential at the sizes where the
kernel's work changes: groups of angular functions in one pass and in several
(more than eight eta), groups split at six functions, powers by squaring, by
pow and of non-integer zeta, layers of one and of several 16 x 16 tiles, no
radial or no angular functions, two atoms, a full slot of 64, weights that would
fill LDS to its last byte (the kernels declare some themselves); FP64 against the
oracle move by move, binary32 against the oracle's replay of its decisions."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no GPU visible", allow_module_level=True)

import paralleltemperingmontecarlo as pt  # noqa: E402
from paralleltemperingmontecarlo import api  # noqa: E402

KB = 3.166811429e-6
R_CUT = 11.338


def _potential(rng, n1, n2, etas, zetas, n_rad, hidden, act):
    rad = tuple(api.RadialType2a.from_scaling(e, R_CUT, 2, [[3.0, 0.0]] * 2, [[4.0, -0.5]] * 2)
                for e in np.geomspace(0.004, 0.3, max(n_rad, 1))[:n_rad])
    ang = tuple(api.AngularType3a.from_scaling(e, lam, z, R_CUT, 2, [[5.0, 0.0]] * 3, [[6.0, 0.2]] * 3)
                for e in etas for lam, z in zetas)
    nodes = [2 * n_rad + 3 * len(ang), *hidden, 1]
    n_par = sum(a * b + b for a, b in zip(nodes, nodes[1:]))
    nets = [pt.NeuralNetworkPotential(nodes, [1, *act, 1], rng.normal(0.0, 0.15, n_par)) for _ in range(2)]
    return pt.RuNNerPotential2Atom(*nets, rad, ang, n1, n2)


def _cluster(rng, n):
    g = np.arange(-3, 4) * 4.6
    pts = np.array(np.meshgrid(g, g, g, indexing="ij")).reshape(3, -1).T
    pts = pts[np.argsort((pts**2).sum(1), kind="stable")][:n]
    return pts + rng.uniform(-0.4, 0.4, pts.shape)


POW2 = ((1.0, 1.0), (-1.0, 2.0), (-1.0, 16.0))
MANY = tuple((lam, z) for lam in (1.0, -1.0) for z in (1.0, 2.0, 4.0, 8.0))  # eight of one eta: split at six
GENERAL = ((1.0, 3.0), (-1.0, 2.5), (0.5, 4.0), (-1.0, 5.0))


@pytest.mark.parametrize("n1,n2,etas,zetas,n_rad,hidden,act", [
    (6, 4, (0.01,), POW2, 2, (5, 3), (2, 2)),
    (4, 3, tuple(np.geomspace(0.002, 0.08, 11)), POW2[:2], 1, (17, 16), (2, 1)),
    (5, 3, (0.004, 0.03), MANY, 1, (16, 33), (1, 2)),
    (3, 5, (0.006, 0.05), GENERAL, 3, (20, 20), (2, 2)),
    (1, 1, (0.02,), POW2[:1], 2, (4, 4), (2, 2)),
    (7, 2, (), (), 4, (8, 8), (2, 2)),
    (50, 14, (0.008, 0.03), POW2, 2, (20, 20), (2, 2)),
    (14, 14, tuple(np.geomspace(0.002, 0.08, 8)), POW2, 2, (59, 8), (2, 2)),
])
def test_moves_match_oracle(oracle, n1, n2, etas, zetas, n_rad, hidden, act):
    rng = np.random.default_rng(100 * n1 + n2)
    pot = _potential(rng, n1, n2, etas, zetas, n_rad, hidden, act)
    n = n1 + n2
    x0 = _cluster(rng, n)
    beta = 1.0 / (KB * np.array([2e4, 6e4]))  # the random networks' energies are of the order of 0.1 Hartree
    ens = pt.NNVT.of([n1, n2], natomswaps=3)
    mc = pt.MCParams(100, 2, n, n_adjust=100)
    print(f"NNVT shapes n1={n1} n2={n2} angular={len(etas) * len(zetas)}", flush=True)
    cycles = 4 if n < 20 else 1
    eng = pt.PTEngine(pot, ens, pt.SphericalBC(25.0), mc,
                      pt.EngineOptions(precision="fp64", exchange="every", seed=9, recompute_every=2, max_displ=(0.6, 0.1)))
    eng.add_run(n, beta, x0[None], pt.SphericalBC(25.0))
    eng.prepare()
    run = oracle.OracleRun(n, beta, x0[None], pot=oracle.make_pot("nnp2", nnp2=oracle.NNP2(pot), n1=n1, n_swaps=3),
                           radius=25.0, exchange_mode=1, mode=oracle.engine_mode(), n_adjust=100, seed=9,
                           max_displ=(0.6, 0.1))
    np.testing.assert_allclose(eng.energies(0), run.en_tot, rtol=1e-12)
    eng.set_trace(cycles)
    eng.cycles(cycles)
    eng.sync()
    de, acc, idx = eng.trace(0, cycles)
    tr = run.cycles(cycles, trace=True)
    np.testing.assert_array_equal(idx, tr["idx"])
    np.testing.assert_array_equal(acc, tr["acc"])
    # rounding: 64 atoms of up to 40 features, each a sum of some hundred terms
    assert np.abs(de - tr["de"]).max() <= 1e-11 * (np.abs(run.en_tot).max() + 1.0)
    x, en, _ = eng.state(0)
    np.testing.assert_array_equal(x, run.x)
    np.testing.assert_allclose(en, pt.nnp2_energies(pot, x)[0], rtol=1e-11, atol=1e-12)
    eng.close()


@pytest.mark.parametrize("n1,n2,etas,zetas,n_rad,hidden,act", [
    (4, 3, tuple(np.geomspace(0.002, 0.08, 11)), POW2[:2], 1, (17, 16), (2, 1)),
    (5, 3, (0.004, 0.03), MANY, 1, (16, 33), (1, 2)),
    (3, 5, (0.006, 0.05), GENERAL, 3, (20, 20), (2, 2)),
    (1, 1, (0.02,), POW2[:1], 2, (4, 4), (2, 2)),
    (50, 14, (0.008, 0.03), POW2, 2, (20, 20), (2, 2)),
])
def test_binary32_moves_follow_oracle(oracle, n1, n2, etas, zetas, n_rad, hidden, act):
    rng = np.random.default_rng(100 * n1 + n2)
    pot = _potential(rng, n1, n2, etas, zetas, n_rad, hidden, act)
    n = n1 + n2
    x0 = _cluster(rng, n).astype(np.float32).astype(np.float64)
    beta = 1.0 / (KB * np.array([2e4, 6e4]))
    cycles = 4 if n < 20 else 1
    eng = pt.PTEngine(pot, pt.NNVT.of([n1, n2], natomswaps=3), pt.SphericalBC(25.0), pt.MCParams(100, 2, n, n_adjust=100),
                      pt.EngineOptions(precision="fp32", exchange="every", seed=9, recompute_every=2, max_displ=(0.6, 0.1)))
    eng.add_run(n, beta, x0[None], pt.SphericalBC(25.0))
    eng.prepare()
    run = oracle.OracleRun(n, beta, x0[None], pot=oracle.make_pot("nnp2", nnp2=oracle.NNP2(pot), n1=n1, n_swaps=3),
                           radius=25.0, exchange_mode=1, mode=oracle.engine_mode(), n_adjust=100, seed=9,
                           max_displ=(0.6, 0.1), fp32=True)
    eng.set_trace(cycles)
    eng.cycles(cycles)
    eng.sync()
    de, acc, idx = eng.trace(0, cycles)
    tr = run.cycles(cycles, trace=True, replay_acc=acc)
    np.testing.assert_array_equal(idx, tr["idx"])
    # an energy is at most S = n (|b3| + sum |w3|) in size where the layers end in tanh, and of that order
    # with a linear one; 2e-6 S is 32 rounding units (2^-24) of S, about the square root of the roundings on
    # the way (at most 70 features, some hundred terms each, and two layers)
    w = np.array([pot.nnp1.parameters, pot.nnp2.parameters])
    scale = n * (np.abs(w[:, -1]) + np.abs(w[:, -1 - hidden[1]:-1]).sum(1)).max()
    assert np.abs(de - tr["de"]).max() <= 2e-6 * scale, np.abs(de - tr["de"]).max() / scale
    x, en, _ = eng.state(0)
    np.testing.assert_array_equal(x, run.x)
    assert np.abs(en - pt.nnp2_energies(pot, x)[0]).max() <= 2e-6 * scale
    eng.close()
