"""State and counters read back from the device: what set_state wrote, for
every slot layout (lanes per configuration, ladders spread over workgroups,
128-atom slots), precision and box, also where the run is larger than the
staging (1 MiB) and is read in pieces.  Positions are exactly representable in
binary32, so the round trip is exact."""
import numpy as np
import pytest

from conftest import GOLDEN, gpu_available

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no GPU visible", allow_module_level=True)

import paralleltemperingmontecarlo as pt  # noqa: E402
from paralleltemperingmontecarlo.nnp_setup import synthetic_cu55_potential  # noqa: E402

LJ = [-4.0, 0.0, 0.0, 4.0]  # r^-6, r^-8, r^-10, r^-12


def _grid(n, a, rng):
    g = np.stack(np.meshgrid(*[np.arange(6)] * 3), -1).reshape(-1, 3)[:n] * a
    x = g - g.mean(0) + rng.uniform(-0.1, 0.1, (n, 3))
    return x


@pytest.mark.parametrize("kind,precision,atoms,temps,lanes,spread", [
    ("sphere", "fp64", 13, 5, 1, 0), ("sphere", "fp32", 13, 250, 1, 0), ("sphere", "fp32", 33, 17, 8, 64),
    ("cubic", "fp32", 108, 13, 16, 64), ("cubic", "fp64", 108, 3, 16, 0), ("cubic", "fp32", 108, 3, 64, 64),
    ("rhombic", "fp32", 64, 6, 4, 0), ("nnp", "fp32", 13, 3, 0, 0), ("nnp", "fp32", 65, 700, 0, 0)])
def test_state_round_trip(kind, precision, atoms, temps, lanes, spread):
    rng = np.random.default_rng(atoms + temps)
    box = {"sphere": pt.SphericalBC(radius=40.0), "nnp": pt.SphericalBC(radius=60.0), "cubic": pt.CubicBC(14.0),
           "rhombic": pt.RhombicBC(14.0, 12.0)}[kind]
    ens = pt.NVT(atoms) if kind in ("sphere", "nnp") else pt.NPT(atoms, 1e-9)
    pot = synthetic_cu55_potential(GOLDEN / "nnp" / "scaling.data") if kind == "nnp" else pt.ELJPotentialEven(LJ)
    spacing = 4.8 if kind == "nnp" else 1.9
    x0 = np.stack([_grid(atoms, spacing, rng) for _ in range(2)])
    eng = pt.PTEngine(pot, ens, box, pt.MCParams(10, temps, atoms),
                      pt.EngineOptions(precision=precision, exchange="even_odd", workgroup_lanes=spread))
    beta = 1.0 / np.linspace(0.3, 2.0, temps)
    runs = [eng.add_run(atoms, beta, x[None], box, lanes=lanes, pressure=1e-9 if kind in ("cubic", "rhombic") else 0.0)
            for x in x0]
    eng.prepare()
    want = {}
    for r in runs:
        x = np.stack([_grid(atoms, spacing, rng) for _ in range(temps)]).astype(np.float32).astype(np.float64)
        words = dict(max_displ=rng.uniform(0.1, 0.2, (temps, 2)), ham=rng.normal(size=(temps, 2)),
                     **{k: rng.integers(0, 1 << 40, (temps, 2)) for k in ("count_atom", "count_vol", "count_exc")})
        bx = None
        if kind == "cubic":
            bx = rng.uniform(13.0, 15.0, temps)
        elif kind == "rhombic":
            bx = rng.uniform(13.0, 15.0, (temps, 2))
        eng.set_state(r, x=x, box=bx, **words)
        want[r] = (x, bx, words)
    for r in runs:
        x, bx, words = want[r]
        gx, ge, gb = eng.state(r)
        assert np.array_equal(gx, x)
        assert np.array_equal(ge, eng.energies(r)) and np.isfinite(ge).all()
        if bx is not None:
            assert np.array_equal(gb, bx)
        c = eng.counters(r)
        for k, v in words.items():
            assert np.array_equal(c[k], v), k
    eng.close()
