"""An FP64 run alone, among others, and resumed among others: the same bits where
the lanes per configuration are given; lanes that the engine chooses by the room
on the device change the rounding of the energies only."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no GPU visible", allow_module_level=True)

import paralleltemperingmontecarlo as pt  # noqa: E402


def _run(pot, n, bc, temp, x, copies, cycles, opts, start=None, lanes=0):
    """State and counters of the last of `copies` runs after `cycles` cycles;
    start: (state, counters, cycle) to go on from."""
    eng = pt.PTEngine(pot, pt.NVT(n), bc, pt.MCParams(100, len(temp.beta_grid), n, n_adjust=3), opts)
    for k in range(copies):
        eng.add_run(n, temp.beta_grid, x[None], bc, run_key=7 if k == copies - 1 else 100 + k, lanes=lanes)
    eng.prepare()
    used = eng.lanes_of(copies - 1)
    eng.start_phase(False)
    if start:
        (xs, _, _), c, at = start
        eng.set_state(copies - 1, x=xs, max_displ=c["max_displ"], count_atom=c["count_atom"])
        eng.seek(at, at)
    eng.cycles(cycles)
    eng.sync()
    out = eng.state(copies - 1), eng.counters(copies - 1), cycles
    eng.close()
    return out, used


@pytest.mark.parametrize("lanes", [2, 0])
def test_run_alone_and_in_a_batch(ne13, lanes):
    n, temp = 13, pt.TempGrid(4.0, 16.0, 32)
    bc = pt.SphericalBC(radius=ne13["radius"])
    opts = pt.EngineOptions(precision="fp64", exchange="even_odd", seed=5)
    args = pt.ELJPotentialEven(ne13["coeff"]), n, bc, temp, ne13["pos"]
    (alone, ca, _), wide = _run(*args, 1, 40, opts, lanes=lanes)
    (among, cb, _), narrow = _run(*args, 600, 40, opts, lanes=lanes)
    # the other half of the way in another batch
    half, _ = _run(*args, 1, 20, opts, lanes=lanes)
    (resumed, cc, _), _ = _run(*args, 600, 20, opts, start=half, lanes=lanes)
    assert np.array_equal(alone[0], among[0]) and np.array_equal(alone[0], resumed[0])
    assert np.array_equal(ca["max_displ"], cc["max_displ"])
    assert all(np.array_equal(ca[k], cb[k]) for k in ca if k != "ham")
    if lanes:
        assert wide == narrow == lanes
        assert np.array_equal(alone[1], among[1])
    else:
        # 40 x 13 moves of energies of the order of E round to 2^-53 E each
        assert wide > narrow
        for en in (among[1], resumed[1]):
            np.testing.assert_allclose(en, alone[1], rtol=600 * 2.0**-53, atol=0)
