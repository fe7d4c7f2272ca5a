"""SHAKE groups at the edges of their blocks (48 groups each) and of the step
kernel's water blocks (64 units), with 1, 2 and 3 hydrogens mixed, with and
without waters and free atoms: initialisation and three steps against the
oracle's integrator driven by the gradients the GPU used.

Bars: both are FP64 and meet the bond equations to 1e-13 or better, so
coordinates agree to 1e-10 A, velocities (displacements over 0.04 AKMA) to 1e-8,
and every bond's squared length holds to 1e-12."""
import numpy as np
import pytest

from apocharmm_amd import systems

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _spec(groups, waters, free):
    n_sites = groups + waters + free
    m = max(4, int(np.ceil(n_sites ** (1.0 / 3.0))))
    L = 5.5 * m
    sites = systems.lattice_sites(m, L)[:n_sites] - 0.5 * L
    spec = systems.tip3p_box(max(waters, 1), L, systems.smooth_grid(L), seed=1, cutnb=10.0,
                             ctofnb=9.0, ctonnb=8.0)
    rng = np.random.default_rng(groups)
    dirs = np.array([[1, 1, 1], [1, -1, -1], [-1, 1, -1]]) / np.sqrt(3.0)
    xyz, q, mass, typ, bonds, sg = [], [], [], [], [], []
    for k in range(groups):
        nh, a = 1 + k % 3, len(xyz)
        xyz += [sites[k]] + [sites[k] + 1.09 * dirs[h] for h in range(nh)]
        q += [-0.1 * nh] + [0.1] * nh
        mass += [12.011] + [1.008] * nh
        typ += [1] + [0] * nh
        bonds += [(a, a + 1 + h) for h in range(nh)]
        sg.append([a] + [a + 1 + h if h < nh else -1 for h in range(3)])
    w0 = len(xyz)
    if waters:
        w = systems.water_positions(sites[groups:groups + waters], rng).reshape(-1, 3)
        xyz += list(w)
        q += [-0.834, 0.417, 0.417] * waters
        mass += [15.9994, 1.008, 1.008] * waters
        typ += [1, 0, 0] * waters
    xyz += list(sites[groups + waters:])
    q += [0.0] * free
    mass += [39.948] * free
    typ += [1] * free
    wb, wbp, wa, wap = systems.water_topology(waters, first=w0)
    spec.update(
        xyz=np.array(xyz), charges=np.array(q), masses=np.array(mass),
        vdwtype=np.array(typ, np.int32),
        bonds=np.concatenate([np.array(bonds, np.int32).reshape(-1, 2), wb]),
        bond_par=np.concatenate([np.tile([[1.09, 320.0]], (len(bonds), 1)), wbp]),
        angles=wa, angle_par=wap,
        waters=(w0 + 3 * np.arange(waters)[:, None] + np.arange(3)).astype(np.int32),
        shake_groups=np.array(sg, np.int32).reshape(-1, 4),
        shake_r2=np.full(groups, 1.09 ** 2))
    return spec


@pytest.mark.parametrize("groups,waters,free", [
    (1, 0, 0), (2, 0, 3), (47, 0, 1), (48, 63, 1), (49, 64, 0), (96, 65, 2), (97, 0, 64)])
def test_groups_match_oracle(oracle, groups, waters, free):
    from apocharmm_amd.force_manager import ForceManager
    from apocharmm_amd.integrator import LangevinThermostatIntegrator, maxwell_velocities
    sp = _spec(groups, waters, free)
    print(groups, "groups", waters, "waters", free, "free atoms", flush=True)
    x = np.array(sp["xyz"])
    v = maxwell_velocities(sp["masses"], 300.0, 5)
    fm = ForceManager(sp).initialize()
    lt = LangevinThermostatIntegrator(0.002, friction=1.0, temperature=300.0, seed=3)
    lt.setCharmmContext(fm, x, v)
    lt.initialize()
    st = lt.getState()
    g, r2 = sp["shake_groups"], sp["shake_r2"]
    ol = oracle.Langevin(1.0 / sp["masses"], sp["waters"], 0.002, 300.0, 1.0, 3, shake=(g, r2))
    xo, vo = x.copy(), v.copy()
    ol.init_constrain(xo, vo)
    dprev = ol.init_backstep(st["grad"], xo, vo)
    assert np.abs(st["xyz"] - xo).max() < 1e-10
    assert np.abs(st["dprev"] - dprev).max() < 1e-10
    for s in range(3):
        lt.propagate(1)
        st = lt.getState()
        if s == 0:
            ol.remove_com(dprev)
        ke = ol.step(st["grad"], xo, dprev, vo, s)
        assert np.abs(st["xyz"] - xo).max() < 1e-10
        assert np.abs(st["vel"] - vo).max() < 1e-8
        assert np.abs(st["thermo"][:2] / ke - 1).max() < 1e-7
    for k in range(1, 4):
        m = g[:, k] >= 0
        if m.any():
            d2 = np.sum((st["xyz"][g[m, 0]] - st["xyz"][g[m, k]]) ** 2, 1)
            assert np.abs(d2 / r2[m] - 1).max() < 1e-12
    lt.close()
    fm.close()
