"""A system in a batch runs the batched instantiations of its step kernels: its
trajectory has to be bit for bit the one it has alone, for uneven boxes, every
layout of the vdW table and bonded solutes too (the boxes of the other batch
tests are cubic water)."""
import numpy as np
import pytest

from apocharmm_amd import systems

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CUBIC, UNEVEN = (21.7, 21.7, 21.7), (21.7, 22.9, 25.3)


def _water(box, ntypes):
    spec = systems.tip3p_box(343, 21.7, 24, seed=3, cutnb=10.0, ctofnb=8.0, ctonnb=7.0)
    spec["box"] = np.array(box)
    if ntypes > 2:
        rng = np.random.default_rng(ntypes)
        half = ntypes // 2
        t = np.arange(1029) % half
        spec["vdwtype"] = (2 * t + (np.arange(1029) % 3 == 0)).astype(np.int32)
        spec["eps"] = np.tile(systems.WATER_EPS, half) * rng.uniform(0.9, 1.1, 2 * half)
        spec["rmin_half"] = np.tile(systems.WATER_RMIN_HALF, half) * rng.uniform(0.97, 1.03,
                                                                               2 * half)
    return spec


def _chain(box):
    spec = systems.solvated_chain(150, 450, 25.4, 27)
    spec.update(cutnb=11.0, ctofnb=10.0, ctonnb=9.0, box=np.array(box))
    return spec


SYSTEMS = {
    "water": lambda: _water(UNEVEN, 2),
    "water, odd grid": lambda: dict(_water(UNEVEN, 2), fft_grid=np.array([25, 27, 33], np.int32)),
    "24 types": lambda: _water(UNEVEN, 24),
    "64 types": lambda: _water(UNEVEN, 64),
    "200 types": lambda: _water(UNEVEN, 200),
    "200 types, cubic": lambda: _water(CUBIC, 200),
    "chain": lambda: _chain((25.4, 26.1, 27.3)),
    "chain, cubic": lambda: _chain((25.4, 25.4, 25.4)),
}


def _make(spec):
    from apocharmm_amd.force_manager import ForceManager
    from apocharmm_amd.integrator import LangevinThermostatIntegrator, maxwell_velocities
    fm = ForceManager(spec).initialize()
    lt = LangevinThermostatIntegrator(0.002, friction=1.0, temperature=300.0, seed=9)
    lt.setCharmmContext(fm, np.asarray(spec["xyz"], np.float64) - 0.5 * np.asarray(spec["box"]),
                        maxwell_velocities(spec["masses"], 300.0, 5))
    return fm, lt


@pytest.mark.parametrize("name", SYSTEMS)
def test_batch_of_one_is_the_lone_trajectory(name):
    from apocharmm_amd.integrator import LangevinBatch
    print("batch of one:", name, flush=True)
    fm, lt = _make(SYSTEMS[name]())
    lt.propagate(25)
    lone = lt.getState()
    lt.close()
    fm.close()
    fm, lt = _make(SYSTEMS[name]())
    batch = LangevinBatch([lt])
    batch.propagate(25)
    torch.cuda.synchronize()
    got = lt.getState()
    for k in ("xyz", "vel", "grad"):
        assert np.array_equal(got[k], lone[k]), (k, np.abs(got[k] - lone[k]).max())
    batch.close()
    lt.close()
    fm.close()
