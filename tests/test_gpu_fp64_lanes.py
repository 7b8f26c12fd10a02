"""Lanes per configuration that FP64 ladders get when none are asked for: the
rule at its edges, and the run on them bit for bit the oracle's with that many
lanes; against one lane (sums in sequence) energies to 1e-13."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no GPU visible", allow_module_level=True)

import paralleltemperingmontecarlo as pt  # noqa: E402

# atoms, temperatures, copies of the run, pair form, lanes
CASES = [(2, 4, 1, "horner", 2), (5, 16, 2, "horner", 8), (13, 16, 1, "horner", 16), (13, 17, 1, "horner", 8),
         (13, 32, 300, "horner", 4), (20, 33, 1, "horner", 4), (20, 65, 1, "horner", 2), (38, 32, 3, "horner", 8),
         (13, 16, 1, "reference", 1), (4, 8, 1, "eam", 4), (13, 32, 2, "eam", 8), (30, 16, 1, "eam", 16),
         (30, 33, 1, "eam", 4)]


@pytest.mark.parametrize("n,temps,copies,form,lanes", CASES)
def test_default_lanes(oracle, ne13, n, temps, copies, form, lanes):
    rng = np.random.default_rng(n + temps)
    k = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3), -1).reshape(-1, 3)[:n] * 6.0
    x = g - g.mean(0) + rng.uniform(-0.2, 0.2, g.shape)
    grid, bc = pt.TempGrid(4.0, 16.0, temps), pt.SphericalBC(radius=25.0)

    eam = (9.0, 6.0, 0.3, 7.0)
    pot = pt.EmbeddedAtomPotential(*eam) if form == "eam" else pt.ELJPotentialEven(ne13["coeff"])
    opot = oracle.make_pot("eam", eam=eam) if form == "eam" else oracle.make_pot("elj_even", ne13["coeff"])

    def engine(asked, runs):
        eng = pt.PTEngine(pot, pt.NVT(n), bc, pt.MCParams(100, temps, n, n_adjust=5),
                          pt.EngineOptions(precision="fp64", pair_form="horner" if form == "eam" else form,
                                           exchange="even_odd", seed=5, lanes_per_replica=asked))
        for key in range(runs):
            eng.add_run(n, grid.beta_grid, x[None], bc, run_key=key)
        eng.prepare()
        return eng

    eng = engine(0, copies)
    assert [eng.lanes_of(r) for r in range(copies)] == [lanes] * copies
    one = engine(1 if n <= 20 else 2, 1)  # more where one lane's slab does not fit LDS
    assert np.allclose(eng.energies(0), one.energies(0), rtol=1e-13, atol=0.0)
    one.close()
    eng.start_phase(False)
    eng.cycles(6)
    eng.sync()
    orc = oracle.OracleRun(n, grid.beta_grid, x, pot=opot, radius=25.0,
                           mode=oracle.REFERENCE if form == "reference" else oracle.engine_mode(lanes),
                           exchange_mode=2, n_adjust=5, seed=5, run_key=0)
    orc.start_phase(False)
    orc.cycles(6)
    xd, en, _ = eng.state(0)
    assert np.array_equal(xd, orc.x.reshape(xd.shape))
    assert np.array_equal(en, orc.en_tot)
    eng.close()
