"""The pair kernel's Coulomb table and its length unit over the range of
kappa and r_off a caller may give (interval edges from 1/64 A up, 32 to 512
intervals, a cutoff on an interval's edge and inside one), for cubic and uneven
boxes and each layout of the vdW table, against the FP64 oracle.

Bars: FP32 pair arithmetic errs by about 13 roundings of 6e-8 (r^-13) per pair,
below 1e-6 of the pair's force, and pairs' errors are independent: 2e-6 of the
direct force's rms.  The FP64 path differs by the box / 2^32 coordinate grid:
5e-8."""
import numpy as np
import pytest

from apocharmm_amd import _lib, systems

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# kappa, r_off
RANGE = [(1e-4, 12.0), (0.34, 12.0), (0.34, 11.93), (0.2, 4.5), (1.0, 7.0), (3.0, 12.0),
         (0.5, 1.9)]


def _spec(kappa, off, box, ntypes):
    n = 216 if off < 9 else 512
    L = 19.0 if off < 9 else 25.0
    spec = systems.tip3p_box(n, L, 24, seed=int(1000 * kappa) + n, kappa=kappa, cutnb=off + 1.0,
                             ctofnb=off, ctonnb=0.8 * off)
    if box == "uneven":
        spec["box"] = np.array([L, 1.1 * L, 1.3 * L])
    if ntypes > 2:  # one type per atom up to ntypes, near the water values
        rng = np.random.default_rng(ntypes)
        t = np.arange(3 * n) % ntypes
        oxygen = np.arange(3 * n) % 3 == 0
        spec["vdwtype"] = (2 * t + oxygen).astype(np.int32)
        spec["eps"] = np.tile(systems.WATER_EPS, ntypes) * rng.uniform(0.9, 1.1, 2 * ntypes)
        spec["rmin_half"] = np.tile(systems.WATER_RMIN_HALF, ntypes) * rng.uniform(0.97, 1.03,
                                                                                 2 * ntypes)
    return spec


def _check(oracle, spec, precision):
    from apocharmm_amd.force_manager import ForceManager
    fm = ForceManager(spec, precision).initialize()
    x = torch.tensor(systems.xyzq_of(spec), device="cuda")
    p = oracle.prepare(spec)
    ref = oracle.evaluate(p, systems.xyzq_of(spec), terms=("direct",))
    rms = np.sqrt(np.mean(np.sum(ref["grad"] ** 2, 1)))
    mixed = precision == "mixed"
    for ev in (False, True):
        fm.calcForce(x, reset=True, calcEnergy=ev, calcVirial=ev, terms=_lib.APO_TERM_DIRECT)
        g = fm.getForces().cpu().numpy()
        err = np.sqrt(np.mean(np.sum((g - ref["grad"]) ** 2, 1))) / rms
        print("force error", err, flush=True)
        assert err <= (2e-6 if mixed else 5e-8)
    fm.close()


@pytest.mark.parametrize("kappa,off", RANGE)
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_table_range(oracle, kappa, off, precision):
    print("kappa", kappa, "r_off", off, precision, flush=True)
    _check(oracle, _spec(kappa, off, "cubic", 2), precision)


# 2 types (P, Q, A12 table), 24 (square table), 64 (triangle in LDS), 256
# (combination rule in FP32, the global table in FP64)
@pytest.mark.parametrize("box", ["cubic", "uneven"])
@pytest.mark.parametrize("ntypes", [2, 12, 32, 128])
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_table_layouts(oracle, box, ntypes, precision):
    print(box, 2 * ntypes, "types", precision, flush=True)
    _check(oracle, _spec(0.34, 9.0, box, ntypes if ntypes > 2 else 2), precision)
