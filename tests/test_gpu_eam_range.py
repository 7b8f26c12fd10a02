"""FP64 EAM terms at the ends of their range, bit for bit the oracle's: the
side-by-side evaluation hands distances and exponents past its limits (r^2
subnormal, zero or infinite, |n log r| above 700) to the general one, also where
only some lanes of a wave are past them."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no GPU visible", allow_module_level=True)

import paralleltemperingmontecarlo as pt  # noqa: E402


@pytest.mark.parametrize("far,near,n,m", [(1e25, 3.0, 12.0, 6.0), (1e25, 3.0, 12.5, 5.5), (1e33, 3.0, 12.0, 6.0),
                                          (1e33, 3.0, 9.0, 6.0), (1e160, 3.0, 9.0, 6.0), (20.0, 1e-20, 12.0, 6.0),
                                          (20.0, 1e-30, 12.0, 6.0), (20.0, 1e-160, 9.0, 6.0)])
@pytest.mark.parametrize("lanes", [1, 4])
def test_terms_at_the_ends_of_the_range(oracle, far, near, n, m, lanes):
    x = np.array([[0.0, 0.0, 0.0], [0.0, near, 0.0], [3.1, 0.3, 0.2], [far, 0.0, 0.0], [-2.9, 0.1, 2.0]])
    radius = 1e161 if far > 1e100 else 1e40
    beta = 1.0 / np.array([0.5, 1.0, 4.0])
    eng = pt.PTEngine(pt.EmbeddedAtomPotential(n, m, 0.3, 7.0), pt.NVT(5), pt.SphericalBC(radius=radius),
                      pt.MCParams(10, 3, 5, n_adjust=2),
                      pt.EngineOptions(precision="fp64", lanes_per_replica=lanes, exchange="even_odd", seed=3))
    run = eng.add_run(5, beta, x[None], pt.SphericalBC(radius=radius), run_key=1)
    eng.prepare()
    orc = oracle.OracleRun(5, beta, x, pot=oracle.make_pot("eam", eam=(n, m, 0.3, 7.0)), radius=radius,
                           mode=oracle.engine_mode(eng.lanes_of(run)), exchange_mode=2, n_adjust=2, seed=3, run_key=1)
    assert np.array_equal(eng.energies(run), orc.en_tot, equal_nan=True)
    eng.set_trace(4)
    eng.start_phase(False)
    eng.cycles(4)
    eng.sync()
    de, acc, idx = eng.trace(run, 4)
    orc.start_phase(False)
    tr = orc.cycles(4, trace=True)
    assert np.array_equal(idx, tr["idx"])
    assert np.array_equal(acc, tr["acc"])
    assert np.array_equal(de, tr["de"], equal_nan=True)
    xd, en, _ = eng.state(run)
    assert np.array_equal(xd, orc.x.reshape(xd.shape))
    assert np.array_equal(en, orc.en_tot, equal_nan=True)
    eng.close()
