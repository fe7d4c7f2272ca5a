"""Reciprocal space over grids that use every radix (2 to 13, with the composite
6, 8 and 10), odd and uneven lengths, and both routes of the y and z transforms
(kx planes in LDS up to 64 x 64 points, separate passes beyond), on one stream
and captured in a graph, against the FP64 oracle.

Bars, of the reciprocal force's rms: FP32 transforms round by about 6e-8 per
stage of each pass (some twenty in all) in random directions and the FP64
path's inputs differ by the box / 2^32 coordinate grid: 5e-6 and 1e-7.  The
energy is a sum of squares: 5e-6 and 1e-7 of itself."""
import numpy as np
import pytest

from apocharmm_amd import _lib, systems

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

GRIDS = [(4, 4, 4), (5, 7, 11), (6, 10, 8), (13, 9, 26), (24, 24, 24), (14, 22, 33), (30, 64, 64),
         (30, 64, 65), (21, 5, 100), (27, 36, 40), (49, 63, 98), (100, 50, 60)]


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_grid_against_oracle(oracle, grid, precision):
    from apocharmm_amd.force_manager import ForceManager
    print("grid", grid, precision, flush=True)
    spec = systems.tip3p_box(216, 19.0, 24, seed=7, cutnb=9.0, ctofnb=8.0, ctonnb=7.0)
    spec["box"] = np.array([19.0, 20.5, 23.0])
    spec["fft_grid"] = np.array(grid, np.int32)
    ref = oracle.evaluate(oracle.prepare(spec), systems.xyzq_of(spec), terms=("recip",))
    rms = np.sqrt(np.mean(np.sum(ref["grad"] ** 2, 1)))
    bar = 5e-6 if precision == "mixed" else 1e-7
    fm = ForceManager(spec, precision).initialize()
    x = torch.tensor(systems.xyzq_of(spec), device="cuda")

    def check():
        g = fm.getForces().cpu().numpy()
        err = np.sqrt(np.mean(np.sum((g - ref["grad"]) ** 2, 1))) / rms
        assert err <= bar, err

    fm.calcForce(x, reset=True, terms=_lib.APO_TERM_RECIP)
    check()
    fixed = fm.force.clone()
    fm.calcForce(x, calcEnergy=True, calcVirial=True, terms=_lib.APO_TERM_RECIP)
    check()
    e = fm.getEnergyComponents()["ewks"]
    assert abs(e - ref["energy"]["ewks"]) <= bar * abs(ref["energy"]["ewks"])
    # the whole force call captured: the pair kernel runs beside the chain
    fm.calcForce(x)
    total = fm.force.clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        fm.calcForce(x)
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(fm.force, total)
        fm.calcForce(x, terms=_lib.APO_TERM_RECIP)
        assert torch.equal(fm.force, fixed)
    del graph
    fm.close()
