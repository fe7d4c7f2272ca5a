"""Energies, gradient and virial of single pairs over the range of kappa and
r_off a caller may give, every layout of the vdW table, both precisions, cubic
and uneven boxes, against 40 digits.

Two atoms at coordinates that are exact in float and in the pair kernel's
32-bit grid (boxes of 32 and 64 A, multiples of 2^-10 A), so that nothing but
the kernel's own arithmetic is left.

Bars, x = kappa r and eps = 2^-53.  FP64 energies (both precisions) and the
FP64 path's forces: Coulomb (12 + 3 x^2) eps (about ten roundings, and r^2's,
which weighs x^2) and beyond x = 5 the table's own 2e-13; vdW 64 eps of the sum
of the magnitudes of its terms (r^-12 is about twenty roundings); forces also
the 2^-40 they are stored in; below 2^-1022 a double holds no relative precision.
FP32 forces and virial: vdW 4e-6 of the
magnitudes (r^-13 from a reciprocal root of 6e-8, and type radii of 6e-8 to the
twelfth); Coulomb (2e-6 + 4e-7 x^2), the latter for the roundings of r^2 and of
exp's argument, and 3e-8 of the bare q q / r^2, the table's fit."""
import numpy as np
import pytest

from apocharmm_amd import _lib, systems

torch = pytest.importorskip("torch")
mp = pytest.importorskip("mpmath")
pytestmark = pytest.mark.gpu
EPS, TINY = 2.0 ** -53, 2.0 ** -1022
CCELEC = 332.0716
Q = 30.0


def _spec(kappa, off, box, ntypes, rng):
    spec = systems.tip3p_box(1, 32.0, 8, seed=1, kappa=kappa, cutnb=off + 1.0, ctofnb=off,
                             ctonnb=0.75 * off)
    spec["box"] = np.array(box, np.float64)
    spec["charges"] = np.array([Q, -Q])
    spec["masses"] = np.ones(2)
    for k, w in (("bonds", 2), ("angles", 3)):
        spec[k] = np.zeros((0, w), np.int32)
    spec["bond_par"] = spec["angle_par"] = np.zeros((0, 2))
    spec["waters"] = np.zeros((0, 3), np.int32)
    spec["vdwtype"] = rng.integers(0, ntypes, 2).astype(np.int32)
    spec["eps"] = rng.uniform(0.05, 0.3, ntypes)
    spec["rmin_half"] = off * rng.uniform(0.06, 0.12, ntypes)  # contacts up to (Rmin / r) = 2
    return spec


def _exact(spec, r2):
    """Coulomb and vdW (energy, -r dU/dr / r^2, magnitude) in 40 digits."""
    kappa, off, on = (mp.mpf(float(spec[k])) for k in ("kappa", "ctofnb", "ctonnb"))
    r = mp.sqrt(r2)
    x = kappa * r
    qq = -mp.mpf(CCELEC) * mp.mpf(Q) ** 2
    u = qq * mp.erfc(x) / r
    w = u + qq * 2 * kappa / mp.sqrt(mp.pi) * mp.exp(-x * x)
    tab = np.asarray(systems.lj_table(spec["eps"], spec["rmin_half"]), np.float32)
    a, b = sorted(int(t) for t in spec["vdwtype"])
    c6, c12 = (mp.mpf(float(v)) for v in tab.reshape(-1, 2)[b * (b + 1) // 2 + a])
    k6, k12 = off ** 3 / (off ** 3 - on ** 3), off ** 6 / (off ** 6 - on ** 6)
    i3, i6, o3, o6 = r ** -3, r ** -6, off ** -3, off ** -6
    if r > on:
        parts = [k12 * c12 * t for t in (i6 * i6, -2 * o6 * i6, o6 * o6)]
        parts += [-k6 * c6 * t for t in (i6, -2 * o3 * i3, o3 * o3)]
        forces = [12 * k12 * c12 * i6 * i6, -12 * k12 * c12 * o6 * i6, -6 * k6 * c6 * i6,
                  6 * k6 * c6 * o3 * i3]
    else:
        parts = [c12 * i6 * i6, -c12 * o6 / on ** 6, -c6 * i6, c6 * o3 / on ** 3]
        forces = [12 * c12 * i6 * i6, -6 * c6 * i6]
    return (u, w / r2, x), (mp.fsum(parts), mp.fsum(forces) / r2, mp.fsum(map(abs, parts)),
                            mp.fsum(map(abs, forces)) / r2)


def _check(kappa, off, box, ntypes, precision):
    from apocharmm_amd.force_manager import ForceManager
    print("pairs: kappa", kappa, "r_off", off, "box", box, "types", ntypes, precision, flush=True)
    rng = np.random.default_rng(int(1000 * kappa + 10 * off) + ntypes)
    spec = _spec(kappa, off, box, ntypes, rng)
    fm = ForceManager(spec, precision).initialize()
    mixed = precision == "mixed"
    # separations from a close contact to the cutoff, across the boundary too
    for r in np.concatenate([np.linspace(0.12, 0.999, 9), [0.74, 0.76]]) * off:
        d = rng.normal(size=3)
        d = np.round(d / np.linalg.norm(d) * r * 1024) / 1024
        if d @ d >= off * off:
            continue
        x0 = np.round(rng.random(3) * spec["box"] * 1024) / 1024
        xyzq = np.zeros((2, 4), np.float32)
        xyzq[:, 3] = spec["charges"]
        xyzq[0, :3], xyzq[1, :3] = x0, np.mod(x0 - d, spec["box"])
        x = torch.tensor(xyzq, device="cuda")
        with mp.workdps(40):
            (u, fc, kr), (uv, fv, muv, mfv) = _exact(spec, mp.mpf(float(d @ d)))
            cb = (12 + 3 * float(kr) ** 2) * EPS + (2e-13 if kr > 5 else 0.0)
            if mixed:
                bare = CCELEC * Q * Q / float(d @ d) ** 1.5
                scale = (2e-6 + 4e-7 * float(kr) ** 2) * abs(fc) + 3e-8 * bare + 4e-6 * mfv
            else:
                scale = cb * abs(fc) + 64 * EPS * mfv
            got = None
            for ev in ((False, False), (True, True), (True, False), (False, True)):
                fm.calcForce(x, reset=True, calcEnergy=ev[0], calcVirial=ev[1],
                             terms=_lib.APO_TERM_DIRECT)
                g = fm.getForces().cpu().numpy()
                # dU/dx of atom 0: -(fc + fv) d
                for a in range(3):
                    want = -(fc + fv) * float(d[a])
                    bar = float(scale * abs(float(d[a]))) + 2.0 ** -39
                    assert abs(g[0, a] - want) <= bar, (ev, float(kr), g[0, a], float(want))
                assert np.array_equal(g[1], -g[0])
                if ev[0]:
                    e = fm.getEnergyComponents()
                    got = got or e
                    assert e == got
                    assert abs(e["elec"] - u) <= cb * abs(u) + TINY, (float(kr), e["elec"], float(u))
                    assert abs(e["vdw"] - uv) <= 64 * EPS * muv + TINY, (float(r), e["vdw"], float(uv))
                if ev[1]:
                    vir = fm.getVirial()
                    for a in range(3):
                        for b in range(3):
                            want = (fc + fv) * float(d[a] * d[b])
                            bar = float(scale * abs(float(d[a] * d[b])))
                            assert abs(vir[a, b] - want) <= bar + TINY, (a, b, vir, float(want))
    fm.close()


@pytest.mark.parametrize("kappa", [0.34, 3.0])
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_atoms_at_one_place(kappa, precision):
    """An infinite Coulomb energy of the product's sign, as 1 / r gives it."""
    from apocharmm_amd.force_manager import ForceManager
    print("coincident atoms", kappa, precision, flush=True)
    spec = _spec(kappa, 12.0, (32.0, 32.0, 32.0), 2, np.random.default_rng(1))
    fm = ForceManager(spec, precision).initialize()
    x = torch.full((2, 4), 5.0, device="cuda")
    for q, want in ((-Q, -np.inf), (Q, np.inf)):
        x[0, 3], x[1, 3] = Q, q
        fm.calcForce(x, reset=True, calcEnergy=True, terms=_lib.APO_TERM_DIRECT)
        assert fm.getEnergyComponents()["elec"] == want
    fm.close()


RANGE = [(1e-4, 12.0), (0.1, 12.0), (0.34, 12.0), (0.34, 11.93), (0.34, 15.0), (0.4, 9.0),
         (0.5, 12.0), (0.5, 1.9), (1.0, 12.0),
         # without a table: kappa above 1, kappa r_off above 12
         (0.9, 14.0), (2.0, 7.0), (3.0, 12.0), (3.0, 1.9), (5.0, 12.0), (8.0, 4.5)]


@pytest.mark.parametrize("kappa,off", RANGE)
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_pairs_over_the_range(kappa, off, precision):
    _check(kappa, off, (32.0, 32.0, 32.0), 2, precision)


# 2 types: switched coefficients per type pair; 24: square table; 64: triangle;
# 200: combination rule (FP32) or the global table (FP64)
@pytest.mark.parametrize("ntypes", [2, 24, 64, 200])
@pytest.mark.parametrize("box", [(32.0, 32.0, 32.0), (32.0, 64.0, 32.0)])
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_pairs_of_every_layout(box, ntypes, precision):
    for kappa, off in ((0.34, 12.0), (3.0, 12.0)):
        _check(kappa, off, box, ntypes, precision)


def test_steps_and_batches_without_a_table():
    """The prune variant and the batched kernel of a system without a table: its
    gradient after ten steps, alone with a pruned list, against a fresh list
    (float sums in another order: 1e-6 of the rms); in a batch with a system that
    has a table, bit for bit its lone trajectory."""
    from apocharmm_amd.force_manager import ForceManager
    from apocharmm_amd.integrator import (LangevinBatch, LangevinThermostatIntegrator,
                                          maxwell_velocities)

    def make(kappa, prune=0):
        spec = systems.tip3p_box(343, 21.7, 24, seed=3, kappa=kappa, cutnb=10.0, ctofnb=8.0,
                                 ctonnb=7.0)
        fm = ForceManager(spec).initialize()
        lt = LangevinThermostatIntegrator(0.002, friction=1.0, temperature=300.0, seed=9)
        lt.setListPruneFrequency(prune)
        lt.setCharmmContext(fm, np.asarray(spec["xyz"], np.float64) - 0.5 * 21.7,
                            maxwell_velocities(spec["masses"], 300.0, 5))
        return spec, fm, lt

    for prune in (0, 5):
        spec, fm, lt = make(3.0, prune)
        lt.propagate(10)
        st = lt.getState()
        lone = st["xyz"] if prune == 0 else lone
        x = torch.tensor(systems.xyzq_of(spec, st["xyz"] - st["dprev"]), device="cuda")
        fm.calcForce(x, reset=True)
        g = fm.getForces().cpu().numpy()
        err = np.sqrt(np.mean((g - st["grad"]) ** 2) / np.mean(g ** 2))
        print("prune", prune, "gradient against a fresh list", err, flush=True)
        assert err <= 1e-6
        lt.close()
        fm.close()
    runs = [make(0.34), make(3.0)]
    batch = LangevinBatch([lt for _, _, lt in runs])
    batch.propagate(10)
    torch.cuda.synchronize()
    assert np.array_equal(runs[1][2].getState()["xyz"], lone)
    batch.close()
    for _, fm, lt in runs:
        lt.close()
        fm.close()
