"""energy_update of the network potential where its device kernels change
shape: atoms around the lanes given to a target (16 lanes up to 16 atoms, one
above 128), one to ten functions of an eta (eight are done together), inactive
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
