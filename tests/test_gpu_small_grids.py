"""The charge spread on axes shorter than a slab and a stencil together (4 to 8
points), where an atom reaches a slab from both sides, against the FP64 oracle.

Bars, of the reciprocal force's rms: FP32 transforms of a few stages 5e-6; the
FP64 path's inputs differ by the box / 2^32 coordinate grid, 1e-7."""
import numpy as np
import pytest

from apocharmm_amd import _lib, systems

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(4, 4, 4), (5, 4, 7), (6, 5, 4), (8, 6, 5), (64, 6, 64),
                                  (32, 64, 5), (24, 7, 8)])
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_short_axes(oracle, grid, precision):
    from apocharmm_amd.force_manager import ForceManager
    print("grid", grid, precision, flush=True)
    spec = systems.tip3p_box(216, 19.0, 24, seed=7, cutnb=9.0, ctofnb=8.0, ctonnb=7.0)
    spec["fft_grid"] = np.array(grid, np.int32)
    ref = oracle.evaluate(oracle.prepare(spec), systems.xyzq_of(spec), terms=("recip",))
    fm = ForceManager(spec, precision).initialize()
    x = torch.tensor(systems.xyzq_of(spec), device="cuda")
    fm.calcForce(x, reset=True, terms=_lib.APO_TERM_RECIP)
    g = fm.getForces().cpu().numpy()
    err = np.sqrt(np.sum((g - ref["grad"]) ** 2) / np.sum(ref["grad"] ** 2))
    assert err <= (5e-6 if precision == "mixed" else 1e-7), err
    fm.close()
