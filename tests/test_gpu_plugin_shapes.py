"""energy_update of the network potential where its device kernels change
shape: atoms around the lanes given to a configuration (a row of 16 up to 4 atoms,
a wave up to 8) and to a target (16 lanes up to 16 atoms, one above 128), a
configuration that fails the hard-core test, one to ten functions of an eta (eight are done together), inactive
functions, hidden layers around the workgroup's split.  Against the FP64 oracle,
which sums in the reference's order: features to 1e-12 of the largest (sums of
up to N^2 / 2 terms of both signs, each to a few units of 2^-53), energies
to 1e-11."""
import numpy as np
import pytest

from conftest import GOLDEN, gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no GPU visible", allow_module_level=True)

import paralleltemperingmontecarlo as pt  # noqa: E402
from paralleltemperingmontecarlo.api import AngularType3, NeuralNetworkPotential, RuNNerPotential  # noqa: E402
from paralleltemperingmontecarlo.nnp_setup import R_CUT, synthetic_cu55_potential  # noqa: E402


def _potential(n_rad, n_eta, per_eta, h1, h2, seed):
    full = synthetic_cu55_potential(GOLDEN / "nnp" / "scaling.data")
    kinds = [(lam, z) for lam in (1, -1) for z in (1, 2, 4, 8, 16)]
    scale = (2.0, 0.0)  # (maximum, minimum) of the scaling
    # the functions of one eta apart in the table
    ang = [AngularType3(0.002 * (e + 1), *kinds[(k + e) % 10], R_CUT, 111, scale)
           for k in range(per_eta) for e in range(n_eta)]
    nf = n_rad + len(ang)
    w = np.random.default_rng(seed).normal(0.0, 0.2, nf * h1 + h1 + h1 * h2 + h2 + h2 + 1)
    return RuNNerPotential(NeuralNetworkPotential([nf, h1, h2, 1], [1, 2, 2, 1], w), full.radsymfunctions[:n_rad], ang)


@pytest.mark.parametrize("n,n_rad,n_eta,per_eta,h1,h2", [
    (2, 1, 1, 1, 1, 1), (3, 2, 2, 10, 5, 4), (16, 8, 3, 9, 20, 20), (17, 8, 1, 8, 32, 17), (33, 3, 7, 2, 17, 32),
    (64, 1, 2, 10, 20, 20), (65, 8, 5, 1, 20, 20), (129, 4, 2, 9, 31, 3)])
def test_network_update_shapes(oracle, n, n_rad, n_eta, per_eta, h1, h2):
    pot = _potential(n_rad, n_eta, per_eta, h1, h2, n)
    rng = np.random.default_rng(n)
    k = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3), -1).reshape(-1, 3)[:n] * 4.8
    x = np.stack([g - g.mean(0) + rng.uniform(-0.4, 0.4, g.shape) for _ in range(3)])
    idx = np.array([0, n - 1, n // 2], dtype=np.int32)
    trial = x[np.arange(3), idx] + rng.uniform(-0.6, 0.6, (3, 3))
    rad, ang = pot.tables()
    opot = oracle.make_pot("nnp", nnp=oracle.NNP(rad, ang, pot.r_cut, pot.nnp.num_nodes, pot.nnp.activation_functions,
                                                 pot.nnp.parameters, hardcore2=pot.boundary, q10_compat=False))
    plug = pt.PotentialPlugin(pot, pt.NVT(n), pt.SphericalBC(radius=60.0))
    en, ea, v = plug.initialise_energy(x)
    ne, nv, nea = plug.energy_update(x, idx, trial, en, v, en_atom=ea)
    for c in range(3):
        o_en, o_v, o_ea = oracle.plugin_update(opot, x[c], int(idx[c]), trial[c], en[c], vars=v[c])
        assert np.max(np.abs(nv[c] - o_v)) <= 1e-12 * np.max(np.abs(o_v))
        assert np.max(np.abs(nea[c] - o_ea)) <= 1e-11 * np.max(np.abs(o_ea))
        assert ne[c] == pytest.approx(o_en, rel=1e-11, abs=1e-11 * np.abs(o_ea).sum())
    plug.close()


@pytest.mark.parametrize("n,confs", [(2, 1), (3, 6), (4, 5), (5, 3), (8, 3), (9, 3)])
def test_few_atoms_among_other_configurations(oracle, n, confs):
    """Up to four configurations of a wave, the last wave not full, one of them
    with a trial inside another atom: its features and energies stay."""
    pot = _potential(3, 3, 9, 6, 5, n)
    pot.boundary = 1.0  # squared hard-core distance
    rng = np.random.default_rng(n)
    g = np.stack(np.meshgrid(*[np.arange(3)] * 3), -1).reshape(-1, 3)[:n] * 4.8
    x = np.stack([g - g.mean(0) + rng.uniform(-0.4, 0.4, g.shape) for _ in range(confs)])
    idx = rng.integers(0, n, confs).astype(np.int32)
    trial = x[np.arange(confs), idx] + rng.uniform(-0.6, 0.6, (confs, 3))
    bad = 1 if confs > 1 else None
    if bad is not None:
        trial[bad] = x[bad, (idx[bad] + 1) % n] + 1e-3
    rad, ang = pot.tables()
    opot = oracle.make_pot("nnp", nnp=oracle.NNP(rad, ang, pot.r_cut, pot.nnp.num_nodes, pot.nnp.activation_functions,
                                                 pot.nnp.parameters, hardcore2=pot.boundary, q10_compat=False))
    plug = pt.PotentialPlugin(pot, pt.NVT(n), pt.SphericalBC(radius=60.0))
    en, ea, v = plug.initialise_energy(x)
    ne, nv, nea = plug.energy_update(x, idx, trial, en, v, en_atom=ea)
    for c in range(confs):
        o_en, o_v, o_ea = oracle.plugin_update(opot, x[c], int(idx[c]), trial[c], en[c], vars=v[c])
        assert np.max(np.abs(nv[c] - o_v)) <= 1e-12 * np.max(np.abs(o_v))
        assert ne[c] == pytest.approx(o_en, rel=1e-11, abs=1e-11 * np.abs(ea[c]).sum())
    if bad is not None:
        assert ne[bad] == 100.0 and np.array_equal(nv[bad], v[bad])
    plug.close()


def test_more_workgroups_than_a_launch_takes():
    """2^32 work items are a launch's limit: 510,000 clusters of five atoms with 32
    eta ask for 33 workgroups each, more than 2^24 of 256 threads.  Every fifty
    thousandth cluster equals the same cluster in a call of its own."""
    n, confs = 5, 510_000
    pot = _potential(1, 32, 1, 2, 2, 7)
    rng = np.random.default_rng(8)
    site = np.array([[0, 0, 0], [4.8, 0, 0], [0, 4.8, 0], [0, 0, 4.8], [4.8, 4.8, 4.8]])
    x = site + rng.uniform(-0.4, 0.4, (confs, n, 3))
    idx = (np.arange(confs) % n).astype(np.int32)
    trial = x[np.arange(confs), idx] + rng.uniform(-0.3, 0.3, (confs, 3))
    plug = pt.PotentialPlugin(pot, pt.NVT(n), pt.SphericalBC(radius=60.0))
    en, ea, v = plug.initialise_energy(x)
    ne, nv, nea = plug.energy_update(x, idx, trial, en, v, en_atom=ea)
    pick = np.r_[0:confs:50_000, confs - 1]
    en1, ea1, v1 = plug.initialise_energy(x[pick])
    ne1, nv1, nea1 = plug.energy_update(x[pick], idx[pick], trial[pick], en1, v1, en_atom=ea1)
    plug.close()
    assert np.array_equal(ne[pick], ne1) and np.array_equal(nv[pick], nv1) and np.array_equal(nea[pick], nea1)
    assert np.array_equal(v[pick], v1) and not np.array_equal(nv[pick], v1)
