"""Energy and virial of reciprocal space on both routes of the y and z transforms
(kx planes in LDS up to 4,096 points, separate passes beyond), even and odd
grids, against the FP64 oracle.

Bars, of the energy and of the largest virial component: FP32 transforms round by
about 6e-8 per stage of some twenty in random directions: 5e-6; the FP64 path's
inputs differ by the box / 2^32 coordinate grid: 1e-7.  Grids of about one
point per A or finer, where the columns at half the grid, whose sign of m a
convention decides, carry next to nothing (exp(-pi^2 m^2 / kappa^2) < 1e-9)."""
import numpy as np
import pytest

from apocharmm_amd import _lib, systems

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# planes, planes of odd and of radix-7 and -11 lengths, passes, the same
@pytest.mark.parametrize("grid", [(24, 24, 24), (27, 25, 45), (22, 33, 49), (30, 64, 64),
                                  (30, 64, 65), (25, 81, 63), (40, 100, 100)])
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_energy_and_virial_against_oracle(oracle, grid, precision):
    from apocharmm_amd.force_manager import ForceManager
    print("recip virial, grid", grid, precision, flush=True)
    spec = systems.tip3p_box(216, 19.0, 24, seed=7, cutnb=9.0, ctofnb=8.0, ctonnb=7.0)
    spec["box"] = np.array([19.0, 20.5, 23.0])
    spec["fft_grid"] = np.array(grid, np.int32)
    ref = oracle.evaluate(oracle.prepare(spec), systems.xyzq_of(spec), terms=("recip",))
    w = np.asarray(ref["virial"]).reshape(3, 3)
    bar = 5e-6 if precision == "mixed" else 1e-7
    fm = ForceManager(spec, precision).initialize()
    x = torch.tensor(systems.xyzq_of(spec), device="cuda")
    fm.calcForce(x, reset=True, calcEnergy=True, calcVirial=True, terms=_lib.APO_TERM_RECIP)
    e, v = fm.getEnergyComponents()["ewks"], fm.getVirial()
    fm.close()
    assert abs(e - ref["energy"]["ewks"]) <= bar * abs(ref["energy"]["ewks"])
    assert np.abs(v - w).max() <= bar * np.abs(w).max(), (v, w)
