"""Energies, virial and gradient of one system and one list have the same bits however a
call runs: on one stream or forked, captured in a graph (replayed with eager work
in between), with kernel timers, as a member of a batch, and for the reciprocal
term on its own.  Their sums are ordered by the kernels' blocks, so the route of
the transforms must not depend on any of these."""
import os

import numpy as np
import pytest

from apocharmm_amd import _lib, charmm_io, systems

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DATA = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "charmm")


def _water(n, ntypes=2):
    L = max(26.0, (n / systems.WATER_DENSITY) ** (1.0 / 3.0))
    spec = systems.tip3p_box(n, L, min(systems.smooth_grid(L), 60), seed=n)
    if ntypes > 2:  # a vdW triangle in LDS
        rng = np.random.default_rng(ntypes)
        half = ntypes // 2
        t = np.arange(3 * n) % half
        spec["vdwtype"] = (2 * t + (np.arange(3 * n) % 3 == 0)).astype(np.int32)
        spec["eps"] = np.tile(systems.WATER_EPS, half) * rng.uniform(0.9, 1.1, 2 * half)
        spec["rmin_half"] = np.tile(systems.WATER_RMIN_HALF, half) * rng.uniform(0.97, 1.03,
                                                                               2 * half)
    return spec


def _protein():
    f = lambda n: os.path.join(DATA, n + ".gz")
    return charmm_io.charmm_system(f("jac_5dhfr.psf"),
                                   [f("par_all22_prot.prm"), f("toppar_water_ions.str")],
                                   f("jac_5dhfr.crd"), (62.23,) * 3, 64, name="dhfr")


# below and above the sizes from which eager calls fork (25,000 atoms with
# energies, 33,000 without), planes that fit beside the pair kernel's tables
# (2 types) and not (64 types, the protein)
CASES = {"water 3k": lambda: _water(1000), "64 types 12k": lambda: _water(4000, 64),
         "protein": _protein, "water 27k": lambda: _water(9000),
         "64 types 27k": lambda: _water(9000, 64), "64 types 34k": lambda: _water(11400, 64)}


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_energies_and_virial_of_every_route(name, precision):
    from apocharmm_amd.force_manager import ForceManager
    spec = CASES[name]()
    print("energy bits:", name, precision, len(spec["charges"]), flush=True)
    fm = ForceManager(spec, precision).initialize()
    x = torch.tensor(systems.xyzq_of(spec), device="cuda")
    fm.resetNeighborList(x)

    def call(energy=True, virial=True, **kw):
        fm.calcForce(x, calcEnergy=energy, calcVirial=virial, **kw)

    call()
    want, vir, grad = fm.getEnergyComponents(), fm.getVirial(), fm.force.clone()
    assert np.isfinite(want["epot"])

    def check(what, energy=True, virial=True):
        torch.cuda.synchronize()
        assert torch.equal(fm.force, grad), what
        if energy:
            assert fm.getEnergyComponents() == want, what
        if virial:
            assert np.array_equal(fm.getVirial(), vir), what

    call(virial=False)
    check("energies alone", virial=False)
    call(energy=False, virial=False)
    check("forces alone", energy=False, virial=False)
    _lib.check(_lib.lib().apo_nb_profile(fm._handle, 1))
    call()
    _lib.check(_lib.lib().apo_nb_profile(fm._handle, 0))
    check("kernel timers")
    call(terms=_lib.APO_TERM_RECIP)
    assert fm.getEnergyComponents()["ewks"] == want["ewks"]
    wk = fm.getVirial()
    call(energy=False, terms=_lib.APO_TERM_RECIP)
    assert np.array_equal(fm.getVirial(), wk)
    for energy, virial in ((True, True), (True, False), (False, True)):
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            call(energy, virial)
        call(energy, virial)
        torch.cuda.synchronize()
        v1 = fm.getVirial()
        for _ in range(3):
            fm.energy.fill_(1.0)
            fm.virial.fill_(1.0)
            g.replay()
            torch.cuda.synchronize()
            if energy:
                assert fm.getEnergyComponents() == want
            if virial:
                assert np.array_equal(fm.getVirial(), v1)
            call()
            check("eager between replays")
        del g
    fm.close()


def test_energies_of_a_batch_member():
    from apocharmm_amd.force_manager import ForceManager
    from apocharmm_amd.integrator import (LangevinBatch, LangevinThermostatIntegrator,
                                          maxwell_velocities)
    spec = _water(9000, 64)
    print("energy bits of a batch member", flush=True)
    fm = ForceManager(spec).initialize()
    x = torch.tensor(systems.xyzq_of(spec), device="cuda")
    fm.calcForce(x, reset=True, calcEnergy=True, calcVirial=True)
    want, vir = fm.getEnergyComponents(), fm.getVirial()
    lt = LangevinThermostatIntegrator(0.002, friction=1.0, temperature=300.0, seed=1)
    lt.setCharmmContext(fm, np.asarray(spec["xyz"], np.float64),
                        maxwell_velocities(spec["masses"], 300.0, 2))
    batch = LangevinBatch([lt])
    fm.calcForce(x, reset=True, calcEnergy=True, calcVirial=True)
    assert fm.getEnergyComponents() == want and np.array_equal(fm.getVirial(), vir)
    batch.close()
    lt.close()
    fm.close()
