"""The final energy/virial reduction at the edges of its chunks (1,024 partial
rows, 4,096 atoms of the self energy) and with regions that have no rows,
against the FP64 oracle.

The all-FP64 path runs, so that the reduction itself is what the bars see: its
inputs differ from the oracle's by the box / 2^32 coordinate grid (about 1e-8 of
a force).  Energies within 1e-10 of the sum of all terms' magnitudes, the
virial within 1e-7 of the sum of the terms' own virials (they cancel in the
total)."""
import numpy as np
import pytest

from apocharmm_amd import systems

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _box(n_waters):
    L = max(10.0, (n_waters / systems.WATER_DENSITY) ** (1.0 / 3.0))
    return systems.tip3p_box(n_waters, L, systems.smooth_grid(L), seed=n_waters, cutnb=5.0,
                             ctofnb=4.5, ctonnb=4.0)


# 1 water: one row everywhere; 1,365 and 1,366 waters: 4,095 and 4,098 atoms (one and two
# chunks of the self energy); 5,500 waters: a 56^3 grid, 1,624 reciprocal rows (two chunks)
@pytest.mark.parametrize("n_waters", [1, 33, 1365, 1366, 5500])
def test_reduction_against_oracle(oracle, n_waters):
    from apocharmm_amd.force_manager import ForceManager
    spec = _box(n_waters)
    _check(oracle, spec, ForceManager(spec, "fp64").initialize())


def test_reduction_without_bonded_rows(oracle):
    from apocharmm_amd.force_manager import ForceManager
    spec = _box(33)
    for k, w in (("bonds", 2), ("angles", 3)):
        spec[k] = np.zeros((0, w), np.int32)
    spec["bond_par"] = spec["angle_par"] = np.zeros((0, 2))
    # without bonds nothing is excluded: keep the atoms of a water apart
    spec["xyz"] = systems.lattice_sites(5, 10.0)[: 3 * 33]
    _check(oracle, spec, ForceManager(spec, "fp64").initialize())


def _check(oracle, spec, fm):
    print("reduction, atoms", fm.natom, flush=True)
    x = torch.tensor(systems.xyzq_of(spec), device="cuda")
    fm.energy.fill_(7.0)
    fm.virial.fill_(-3.0)
    fm.calcForce(x, reset=True, calcEnergy=True, calcVirial=True)
    got, vir = fm.getEnergyComponents(), fm.getVirial()
    p, xyzq = oracle.prepare(spec), systems.xyzq_of(spec)
    ref = oracle.evaluate(p, xyzq)
    scale = sum(abs(v) for k, v in ref["energy"].items() if k != "epot")
    for k, r in ref["energy"].items():
        assert abs(got[k] - r) <= 1e-10 * scale, (k, got[k], r)
    wscale = sum(np.abs(oracle.evaluate(p, xyzq, terms=(t,))["virial"]).max()
                 for t in ("bonded", "direct", "pairs14", "recip"))
    assert np.abs(vir - np.asarray(ref["virial"]).reshape(3, 3)).max() <= 1e-7 * wscale
    fm.close()
