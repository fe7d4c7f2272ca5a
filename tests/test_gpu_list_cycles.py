"""List cycles run as recorded graphs or, the first time at given launch constants,
step by step: every mix of the two has to give the trajectory of eager stepping
bit for bit, also where the prune interval does not divide the list interval."""
import numpy as np
import pytest

from apocharmm_amd import systems

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

NB = 8


def _run(pieces, prune, comfreq, graph=True, setting=0):
    from apocharmm_amd.force_manager import ForceManager
    from apocharmm_amd.integrator import LangevinThermostatIntegrator, maxwell_velocities
    spec = systems.tip3p_box(343, 21.7, 24, seed=3, cutnb=10.0, ctofnb=8.0, ctonnb=7.0)
    fm = ForceManager(spec).initialize()
    lt = LangevinThermostatIntegrator(0.002, friction=1.0, temperature=300.0, seed=9)
    lt.setNonbondedListUpdateFrequency(NB)
    lt.setListPruneFrequency(prune)
    lt.setRemoveCenterOfMassFrequency(comfreq)
    lt.setLaunchSetting(setting)
    lt.setUseGraph(graph)
    lt.setCharmmContext(fm, np.asarray(spec["xyz"], np.float64) - 0.5 * np.asarray(spec["box"]),
                        maxwell_velocities(spec["masses"], 300.0, 5))
    for k in pieces:
        lt.propagate(k)
    st = lt.getState()
    th = lt._state(())["thermo"]
    lt.close()
    fm.close()
    return [np.asarray(st[k]).tobytes() for k in ("xyz", "vel", "dprev", "grad")] + [
        np.asarray(th, np.float64).tobytes()]


@pytest.mark.parametrize("prune,comfreq", [(0, 0), (4, 0), (3, 0), (4, 20)])
@pytest.mark.parametrize("pieces", [(5 * NB,), (NB,) * 5, (NB, 3 * NB, NB), (2 * NB, 3 * NB)])
def test_stepped_and_recorded_cycles(pieces, prune, comfreq):
    assert _run(pieces, prune, comfreq) == _run(pieces, prune, comfreq, graph=False)


def test_the_trial_of_launch_settings():
    # 16 trial cycles, then one step by step, then recorded ones
    assert _run((20 * NB,), 4, 0, setting=None) == _run((20 * NB,), 4, 0, graph=False)
