"""Moves of the network potential at the edges of its device kernels' tiles:
cluster sizes around the 16-atom tiles and the two slot widths, hidden widths
around the 16-column tiles, angular groups from one function to ten, against
the FP64 oracle on replayed positions.

Tolerance: an energy is at most S = N (|b3| + sum |w3|) in size (tanh is
bounded), each of its N terms a sum of h2 products in binary32 on two layers of
sums of at most 88 products; 2e-6 S is 32 rounding units (2^-24) of S, about
the square root of the roundings on the way (88 + 2 x 32 sums of terms, exponentials
and cosines of a few units each)."""
import numpy as np
import pytest

from conftest import GOLDEN, gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no GPU visible", allow_module_level=True)

import paralleltemperingmontecarlo as pt  # noqa: E402
from paralleltemperingmontecarlo.api import NeuralNetworkPotential, PTEngine, RuNNerPotential  # noqa: E402
from paralleltemperingmontecarlo.nnp_setup import synthetic_cu55_potential  # noqa: E402

# atoms, radial and angular functions kept, hidden widths, how far apart the atoms are, temperatures (above 256
# the slots of 33 to 64 atoms take 512 threads)
SHAPES = [s + (2,) for s in (
          (2, 1, 1, 1, 1, 4.5), (3, 8, 80, 20, 20, 4.5), (15, 2, 5, 16, 17, 4.8), (16, 8, 26, 17, 16, 4.8),
          (17, 5, 33, 32, 32, 4.8), (33, 3, 60, 20, 5, 9.0), (49, 8, 80, 20, 20, 5.4), (63, 1, 80, 31, 20, 4.8),
          (64, 8, 79, 20, 20, 4.8), (65, 4, 22, 20, 20, 4.8), (97, 8, 26, 16, 32, 5.4), (128, 2, 9, 20, 17, 4.8))]
SHAPES.append((34, 2, 9, 20, 17, 4.8, 258))


def _cluster(n, spacing, seed):
    """n sites of a simple cubic grid nearest its centre, each moved a little."""
    rng = np.random.default_rng(seed)
    g = np.stack(np.meshgrid(*[np.arange(-3, 4)] * 3), -1).reshape(-1, 3) * spacing
    x = g[np.argsort((g ** 2).sum(1), kind="stable")[:n]] + rng.uniform(-0.2, 0.2, (n, 3))
    return np.ascontiguousarray((x - x.mean(0)).astype(np.float32).astype(np.float64))


@pytest.mark.parametrize("n,n_rad,n_ang,h1,h2,spacing,R", SHAPES)
def test_moves_at_tile_edges(oracle, n, n_rad, n_ang, h1, h2, spacing, R):
    full = synthetic_cu55_potential(GOLDEN / "nnp" / "scaling.data")
    nf = n_rad + n_ang
    n_par = nf * h1 + h1 + h1 * h2 + h2 + h2 + 1
    w = np.random.default_rng(n + 7 * nf).normal(0.0, 0.1, n_par)
    pot = RuNNerPotential(NeuralNetworkPotential([nf, h1, h2, 1], [1, 2, 2, 1], w), full.radsymfunctions[:n_rad],
                          full.angsymfunctions[:n_ang])
    scale = n * (abs(w[-1]) + np.abs(w[-1 - h2:-1]).sum())
    ncyc = 2 if n < 34 else 1
    x0, radius = _cluster(n, spacing, 100 + n), 45.0
    temp = pt.TempGrid(300.0, 30000.0, R)
    eng = PTEngine(pot, pt.NVT(n), pt.SphericalBC(radius), pt.MCParams(10, R, n, n_adjust=5),
                   pt.EngineOptions(precision="fp32", exchange="even_odd", seed=31 + n))
    run = eng.add_run(n, temp.beta_grid, x0[None], pt.SphericalBC(radius), run_key=2)
    eng.prepare()
    eng.set_trace(ncyc)
    eng.start_phase(False)
    eng.cycles(ncyc)
    eng.sync()
    de, acc, idx = eng.trace(run, ncyc)
    rad, ang = pot.tables()
    orc = oracle.OracleRun(n, temp.beta_grid, x0, pot=oracle.make_pot("nnp", nnp=oracle.NNP(
        rad, ang, pot.r_cut, pot.nnp.num_nodes, pot.nnp.activation_functions, pot.nnp.parameters,
        hardcore2=pot.boundary, q10_compat=pot.q10_compat)), radius=radius, mode=oracle.engine_mode(1), fp32=True,
        exchange_mode=2, n_adjust=5, seed=31 + n, run_key=2)
    orc.start_phase(False)
    tr = orc.cycles(ncyc, replay_acc=acc)
    assert np.array_equal(idx, tr["idx"])
    err = np.abs(de - tr["de"])
    assert err.max() <= 2e-6 * scale, (err.max() / scale, int(err.argmax()))
    x_dev, en_dev, _ = eng.state(run)
    assert np.array_equal(x_dev, orc.x.reshape(x_dev.shape))
    assert np.max(np.abs(en_dev - orc.en_tot)) <= 2e-6 * scale
    eng.close()
