"""Performance cases: the force calls and MD runs a user of this package makes.

A force call is ForceManager.calcForce and what the caller reads after it (the
gradient on the device; energies and the virial on the host when asked for).
An MD case is LangevinThermostatIntegrator.propagate over two list cycles.
Water is a piece of an equilibrated 50 A TIP3P liquid (the water box of the
tests), repeated or cut to the wanted edges; the protein is the 23,558-atom
DHFR benchmark system; the chain is the solvated random walk of
apocharmm_amd.systems.  The seed moves and turns every water a little, moves
every other atom a little and draws the velocities.

Mixed-precision results are handed on in single precision, the precision they
are computed in; the all-FP64 path's stay in double.
"""
import functools
import math
import os

import numpy as np
import torch

from apocharmm_amd import charmm_io, systems
from apocharmm_amd.force_manager import ForceManager
from apocharmm_amd.integrator import LangevinThermostatIntegrator, maxwell_velocities

DATA = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tests", "golden",
                    "charmm")
LIQUID_EDGE = 50.0     # the equilibrated water box
SEAM = 2.5             # smallest O-O distance left across a cut (A)
ATOMS_PER_A3 = 0.094   # TIP3P liquid
MD_STEPS = 40          # two list cycles
WIDE = (14.0, 12.0, 10.0)  # cutnb, ctofnb, ctonnb of the benchmark systems
SHORT = (10.0, 9.0, 8.0)   # of boxes too small for them


def water(lx, ly=None, lz=None, grid=None, cut=WIDE):
    ly, lz = ly or lx, lz or lx
    g = grid or tuple(systems.smooth_grid(e) for e in (lx, ly, lz))
    return dict(system="water", lx=lx, ly=ly, lz=lz, kx=g[0], ky=g[1], kz=g[2], cutnb=cut[0],
                ctofnb=cut[1], ctonnb=cut[2])


def protein(grid=64, cut=WIDE):
    return dict(system="protein", lx=62.23, ly=62.23, lz=62.23, kx=grid, ky=grid, kz=grid,
                cutnb=cut[0], ctofnb=cut[1], ctonnb=cut[2])


def chain(nchain, nwater, edge, grid):
    return dict(system="chain", nchain=nchain, nwater=nwater, lx=edge, ly=edge, lz=edge, kx=grid,
                ky=grid, kz=grid, cutnb=WIDE[0], ctofnb=WIDE[1], ctonnb=WIDE[2])


def force(energy=False, virial=False, reset=False, precision="mixed"):
    return dict(call="force", energy=energy, virial=virial, reset=reset, precision=precision)


def md(prune=0):
    return dict(call="md", steps=MD_STEPS, prune=prune, precision="mixed")


def listed():
    return [
        # the smallest periodic box of the smoke test: a caller that steps a
        # small system itself and wants only forces; latency and launches
        dict(name="force_1k", **water(21.7, grid=(24, 24, 24), cut=SHORT), **force()),
        # energy and virial of the 31 A benchmark box: what a Monte-Carlo or
        # barostat loop reads on every call
        dict(name="energy_virial_3k", **water(31.04, grid=(32, 32, 32)),
             **force(energy=True, virial=True)),
        # every call on coordinates the list has not seen (scoring separate
        # frames of a trajectory): list build and forces
        dict(name="rebuild_force_12k", **water(LIQUID_EDGE, grid=(48, 48, 48)),
             **force(reset=True)),
        # the all-FP64 path as the reference result of a mid-sized system
        dict(name="fp64_energy_virial_12k", **water(LIQUID_EDGE, grid=(48, 48, 48)),
             **force(energy=True, virial=True, precision="fp64")),
        # protein in water, every bonded term and 35 vdW types, with energies
        dict(name="energy_virial_protein_24k", **protein(), **force(energy=True, virial=True)),
        # one vdW type per solute atom: more types than any table in LDS holds
        dict(name="force_chain_24k", **chain(2489, 7023, 62.23, 64), **force()),
        # an uneven box with odd grid edges, forces and the virial (constant
        # pressure steps of a caller's own integrator)
        dict(name="virial_uneven_28k", **water(48.7, 62.9, 97.3, grid=(49, 63, 98)),
             **force(virial=True)),
        # the largest water box: forces alone ...
        dict(name="force_94k", **water(2 * LIQUID_EDGE, grid=(100, 100, 100)), **force()),
        # ... and a fresh list with energies and virial (the first call on new
        # coordinates, and the report of an analysis run)
        dict(name="rebuild_energy_virial_94k", **water(2 * LIQUID_EDGE, grid=(100, 100, 100)),
             **force(energy=True, virial=True, reset=True)),
        # Langevin/SETTLE dynamics of the small box
        dict(name="md_3k", **water(31.04, grid=(32, 32, 32)), **md()),
        # ... of the protein, with SHAKE on its bonds to hydrogen
        dict(name="md_protein_24k", **protein(), **md()),
        # ... and of the largest box, with the list pruned between builds as
        # the benchmark runs it
        dict(name="md_94k", **water(2 * LIQUID_EDGE, grid=(100, 100, 100)), **md(prune=10)),
    ]


def draw(rng):
    """Boxes of 21.7 to 100 A (1,000 to 94,000 atoms, a third of them uneven),
    grids of about one point per A, the call and its options."""
    call = rng.choice(["force", "force", "force", "force", "md"])
    kind = rng.choice(["water", "water", "water", "protein", "chain"])
    if call == "md" and kind == "chain":
        kind = "water"
    if kind == "protein":
        off = round(rng.uniform(9.0, 12.0), 2)
        sys_ = protein(rng.choice([60, 63, 64, 65, 66, 70]), (off + 2.0, off, off - 2.0))
    elif kind == "chain":
        n = int(math.exp(rng.uniform(math.log(150), math.log(1200))))
        edge = round(32.0 * (n / 300.0) ** (1.0 / 3.0), 2)
        edge = max(edge, 24.6)
        sys_ = chain(n, 3 * n, edge, systems.smooth_grid(edge))
    else:
        lo, hi = math.log(21.7), math.log(99.9)
        edges = [round(math.exp(rng.uniform(lo, hi)), 2)] * 3
        if rng.random() < 1.0 / 3.0:
            edges = [round(math.exp(rng.uniform(lo, hi)), 2) for _ in range(3)]
        cut = WIDE if min(edges) > 24.2 else SHORT
        spacing = rng.uniform(0.95, 1.1)
        sys_ = water(*edges, grid=tuple(systems.smooth_grid(e, spacing) for e in edges), cut=cut)
    volume = sys_["lx"] * sys_["ly"] * sys_["lz"]
    if call == "md":
        return dict(**sys_, **md(rng.choice([0, 10]) if volume > 2.5e5 else 0))
    fp64 = rng.random() < 0.15 and volume < 2.5e5
    return dict(**sys_, **force(energy=rng.random() < 0.4, virial=rng.random() < 0.4,
                                reset=rng.random() < 0.35,
                                precision="fp64" if fp64 else "mixed"))


# ---- systems ----------------------------------------------------------------
def _file(name):
    return os.path.join(DATA, name + ".gz")


@functools.lru_cache(maxsize=1)
def _liquid():
    """(3916, 3, 3) coordinates of the equilibrated water box."""
    crd = charmm_io.CharmmCrd(_file("waterbox.crd"))
    return np.asarray(crd.coords, np.float64).reshape(-1, 3, 3)


@functools.lru_cache(maxsize=4)
def _water_coords(lx, ly, lz):
    """Whole waters whose oxygen lies in [0, L) of the repeated liquid, less
    those that would touch another one across a cut."""
    L = np.array([lx, ly, lz])
    w = _liquid()
    w = w - LIQUID_EDGE * np.floor(w[:, :1] / LIQUID_EDGE)
    n = np.ceil(L / LIQUID_EDGE - 1e-9).astype(int)
    rep = np.stack(np.meshgrid(*[np.arange(k) for k in n], indexing="ij"), -1).reshape(-1, 1, 1, 3)
    w = (w[None] + LIQUID_EDGE * rep).reshape(-1, 3, 3)
    w = w[np.all(w[:, 0] < L, 1)]
    cut = np.abs(L - LIQUID_EDGE * n) > 1e-9
    o = w[:, 0]
    edge = np.nonzero(np.any(((o < SEAM) | (o > L - SEAM)) & cut, 1))[0]
    drop = np.zeros(len(w), bool)
    for a in range(0, len(edge), 512):
        i = edge[a:a + 512]
        d = o[i][:, None] - o[edge][None]
        shift = np.round(d / L)
        d -= L * shift
        near = (np.einsum("ijk,ijk->ij", d, d) < SEAM ** 2) & np.any((shift != 0) & cut, 2)
        near &= i[:, None] > edge[None]
        drop[i[np.any(near, 1)]] = True
    return w[~drop]


@functools.lru_cache(maxsize=6)
def _spec(system, lx, ly, lz, kx, ky, kz, cutnb, ctofnb, ctonnb, nchain, nwater):
    """The system without its seed: topology, parameters, coordinates."""
    if system == "protein":
        s = charmm_io.charmm_system(_file("jac_5dhfr.psf"),
                                    [_file("par_all22_prot.prm"), _file("toppar_water_ions.str")],
                                    _file("jac_5dhfr.crd"), (lx, ly, lz), kx, name="dhfr")
    elif system == "chain":
        s = systems.solvated_chain(nchain, nwater, lx, kx)
    else:
        w = _water_coords(lx, ly, lz)
        s = systems.tip3p_box(len(w), max(lx, ly, lz), kx)
        s["xyz"] = w.reshape(-1, 3)
    s["box"] = np.array([lx, ly, lz])
    s["fft_grid"] = np.array([kx, ky, kz], np.int32)
    s.update(cutnb=cutnb, ctofnb=ctofnb, ctonnb=ctonnb)
    return s


def _system(case):
    return _spec(*[case[k] for k in ("system", "lx", "ly", "lz", "kx", "ky", "kz", "cutnb",
                                     "ctofnb", "ctonnb")],
                 case.get("nchain", 0), case.get("nwater", 0))


def _coordinates(case, seed):
    """The seed's coordinates: waters moved by ~0.03 A and turned by ~2
    degrees as wholes, other atoms moved by ~0.01 A.  MD starts from rigid
    waters."""
    spec = _system(case)
    rng = np.random.default_rng(seed)
    x = np.array(spec["xyz"], np.float64)
    waters = np.asarray(spec["waters"], np.int64)
    other = np.ones(len(x), bool)
    other[waters.reshape(-1)] = False
    x[other] += rng.normal(0.0, 0.01, (int(other.sum()), 3))
    w = x[waters]
    if case["call"] == "md":
        o, m = w[:, 0], 0.5 * (w[:, 1] + w[:, 2])
        ey = (m - o) / np.linalg.norm(m - o, axis=1)[:, None]
        ex = w[:, 1] - w[:, 2]
        ex -= np.sum(ex * ey, 1)[:, None] * ey
        ex /= np.linalg.norm(ex, axis=1)[:, None]
        f = systems.water_frame()
        w = o[:, None] + f[None, :, :1] * ex[:, None] + f[None, :, 1:2] * ey[:, None]
    t = rng.normal(0.0, 0.03, (len(w), 3))
    d = w - w[:, :1]
    w = w[:, :1] + d + np.cross(t[:, None], d)
    if case["call"] == "md":  # the turn above is first order: restore the lengths
        d = w - w[:, :1]
        d[:, 1:] *= systems.TIP3P["roh"] / np.linalg.norm(d[:, 1:], axis=2)[:, :, None]
        w = w[:, :1] + d
    x[waters] = w + rng.normal(0.0, 0.03, (len(w), 1, 3))
    return spec, x


class _DeviceArray:
    """A device address of the integrator as an array torch can read."""

    def __init__(self, address, shape):
        self.__cuda_array_interface__ = dict(data=(address, False), shape=shape, typestr="<f4",
                                             version=2)


def prepare(case, seed):
    spec, x = _coordinates(case, seed)
    fm = ForceManager(spec, case["precision"]).initialize()
    if case["call"] == "md":
        lt = LangevinThermostatIntegrator(0.002, friction=1.0, temperature=300.0, seed=seed)
        lt.setNonbondedListUpdateFrequency(20)
        lt.setListPruneFrequency(case["prune"])
        x = x - (0.0 if case["system"] == "protein" else 0.5 * spec["box"])
        lt.setCharmmContext(fm, x, maxwell_velocities(spec["masses"], 300.0, seed))
        lt.initialize()
        view = torch.as_tensor(_DeviceArray(lt.getXYZQ(), (fm.natom, 4)), device="cuda")
        return dict(case=case, lt=lt, fm=fm, xyzq=view)
    xyzq = torch.tensor(systems.xyzq_of(spec, x), device="cuda")
    if not case["reset"]:
        fm.resetNeighborList(xyzq)
    return dict(case=case, fm=fm, xyzq=xyzq)


def run(state):
    case, fm = state["case"], state["fm"]
    if case["call"] == "md":
        state["lt"].propagate(case["steps"])
        return state["xyzq"].clone()
    fm.calcForce(state["xyzq"], reset=case["reset"], calcEnergy=case["energy"],
                 calcVirial=case["virial"])
    mixed = case["precision"] == "mixed"
    out = dict(gradient=fm.getForces().float() if mixed else fm.getForces())
    if case["energy"]:
        out["energy"] = fm.getEnergyComponents()
    if case["virial"]:
        v = fm.getVirial()
        out["virial"] = v.astype(np.float32) if mixed else v
    return out


def work(case):
    """Coordinates in and the gradient out; 61 flops per pair inside r_off (100
    with the energy), the PME stencils (64 points twice per atom) and two 3-D
    real FFTs.  An MD step also reads and writes x, v and the displacements."""
    volume = case["lx"] * case["ly"] * case["lz"]
    n = ATOMS_PER_A3 * volume
    grid = case["kx"] * case["ky"] * case["kz"]
    pairs = 0.5 * n * ATOMS_PER_A3 * 4.0 / 3.0 * math.pi * case["ctofnb"] ** 3
    flops = pairs * (100 if case.get("energy") else 61) + n * 64 * 12
    flops += 2 * 2.5 * grid * math.log2(grid) + 10 * grid
    bytes_ = 16 * n + 24 * n
    if case["call"] == "md":
        return dict(bytes=case["steps"] * (bytes_ + 2 * 72 * n), flops=case["steps"] * flops)
    return dict(bytes=bytes_, flops=flops)


# ---- the same results from the formulas, in 64 bits -------------------------
CCELEC = 332.0716


def _exclusions(n, bonds):
    """Sorted keys i * n + j (i < j) of the excluded pairs (1-2, 1-3, 1-4), and
    the 1-4 and 1-2/1-3 pair lists."""
    b = np.asarray(bonds, np.int64).reshape(-1, 2)
    e = np.unique(np.concatenate([b, b[:, ::-1]]), axis=0)
    start = np.searchsorted(e[:, 0], np.arange(n + 1))

    def join(p):
        cnt = start[p[:, 1] + 1] - start[p[:, 1]]
        first = np.repeat(p[:, 0], cnt)
        at = np.repeat(start[p[:, 1]] - (np.cumsum(cnt) - cnt), cnt) + np.arange(cnt.sum())
        q = np.stack([first, e[at, 1]], 1)
        return np.unique(q[q[:, 0] != q[:, 1]], axis=0)

    key = lambda p: np.unique(p[p[:, 0] < p[:, 1]] @ np.array([n, 1]))
    p13 = join(e)
    k12, k13 = key(e), key(p13)
    k14 = np.setdiff1d(key(join(p13)), np.union1d(k12, k13))
    kex = np.union1d(k12, k13)
    pairs = lambda k: np.stack([k // n, k % n], 1)
    return np.union1d(kex, k14), pairs(k14), pairs(kex)


def _f32(a):
    return np.asarray(a, np.float32).astype(np.float64)


class _Exact:
    def __init__(self, spec, xyzq):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.s = spec
        q = self.t(np.asarray(xyzq, np.float32).astype(np.float64))
        self.x, self.q = q[:, :3].contiguous(), q[:, 3].contiguous()
        self.n = len(q)
        self.L = self.t(spec["box"])
        self.kappa = float(spec["kappa"])
        self.g = torch.zeros_like(self.x)
        self.w = self.t(np.zeros((3, 3)))
        self.e = {k: 0.0 for k in ("bond", "angle", "ureyb", "dihe", "imdihe", "ewks", "ewse",
                                   "ewex", "elec", "vdw")}
        self.type = self.t(np.asarray(spec["vdwtype"], np.int64))
        off, on = float(spec["ctofnb"]), float(spec["ctonnb"])
        self.off, self.on = off, on
        self.k6 = off ** 3 / (off ** 3 - on ** 3)
        self.k12 = off ** 6 / (off ** 6 - on ** 6)

    def t(self, a):
        return torch.as_tensor(np.ascontiguousarray(a), device=self.dev)

    def lj(self, i, j, fourteen):
        """(c6, c12) of the pairs."""
        s, a, b = self.s, self.type[i], self.type[j]
        name = "vdwtab14" if fourteen else "vdwtab"
        if name in s:
            hi, lo = torch.maximum(a, b), torch.minimum(a, b)
            c = self.t(_f32(s[name])).reshape(-1, 2)[hi * (hi + 1) // 2 + lo]
            return c[:, 0], c[:, 1]
        eps = s.get("eps14", s["eps"]) if fourteen else s["eps"]
        rh = s.get("rmin_half14", s["rmin_half"]) if fourteen else s["rmin_half"]
        eps, rh = self.t(np.asarray(eps, np.float64)), self.t(np.asarray(rh, np.float64))
        e = torch.sqrt(eps[a] * eps[b])
        r6 = (rh[a] + rh[b]) ** 6
        return (2.0 * e * r6).float().double(), (e * r6 * r6).float().double()

    def pairs(self, i, j, d, coulomb, fourteen=None):
        """Adds pairs (i, j) with differences d: coulomb is the name of the
        energy and the constant of qq (erfc(kappa r) + c) / r; fourteen False /
        True also adds the switched vdW term with that table."""
        name, c = coulomb
        r2 = torch.sum(d * d, 1)
        r = torch.sqrt(r2)
        qq = CCELEC * self.q[i] * self.q[j]
        u = qq * (torch.special.erfc(self.kappa * r) + c) / r
        du = -u / r - qq * 2.0 * self.kappa / math.sqrt(math.pi) * torch.exp(-(self.kappa * r) ** 2) / r
        self.e[name] += float(u.sum())
        if fourteen is not None:
            c6, c12 = self.lj(i, j, fourteen)
            r3, o3 = 1.0 / (r * r2), 1.0 / self.off ** 3
            n3, n6 = 1.0 / self.on ** 3, 1.0 / self.on ** 6
            outer = r > self.on
            a6 = torch.where(outer, self.k6 * (r3 - o3) ** 2, r3 ** 2 - n3 * o3)
            a12 = torch.where(outer, self.k12 * (r3 ** 2 - o3 ** 2) ** 2, r3 ** 4 - n6 * o3 ** 2)
            b6 = torch.where(outer, -6.0 * self.k6 * (r3 - o3) * r3, -6.0 * r3 ** 2) / r
            b12 = torch.where(outer, -12.0 * self.k12 * (r3 ** 2 - o3 ** 2) * r3 ** 2,
                              -12.0 * r3 ** 4) / r
            self.e["vdw"] += float((c12 * a12 - c6 * a6).sum())
            du = du + c12 * b12 - c6 * b6
        f = (du / r)[:, None] * d
        self.g.index_add_(0, i, f)
        self.g.index_add_(0, j, -f)
        self.w -= d.T @ f

    def direct(self, excluded):
        excl = self.t(excluded)
        step = max(1, int(2e7) // self.n)
        off2 = self.off ** 2
        for a in range(0, self.n, step):
            b = min(self.n, a + step)
            r2 = torch.zeros((b - a, self.n - a), dtype=torch.float64, device=self.dev)
            for k in range(3):
                d = self.x[a:b, k, None] - self.x[None, a:, k]
                d -= self.L[k] * torch.round(d / self.L[k])
                r2 += d * d
            i, j = torch.nonzero(r2 < off2, as_tuple=True)
            keep = i < j
            i, j = i[keep] + a, j[keep] + a
            if len(excl):
                key = i * self.n + j
                at = torch.searchsorted(excl, key).clamp(max=len(excl) - 1)
                keep = excl[at] != key
                i, j = i[keep], j[keep]
            d = self.x[i] - self.x[j]
            d -= self.L * torch.round(d / self.L)
            self.pairs(i, j, d, ("elec", 0.0), False)

    def listed_pairs(self, pairs, coulomb, fourteen=None):
        if len(pairs):
            i, j = self.t(pairs[:, 0]), self.t(pairs[:, 1])
            self.pairs(i, j, self.x[i] - self.x[j], coulomb, fourteen)

    def bonded(self):
        s = self.s
        x = self.x.clone().requires_grad_(True)
        terms = {}

        def rows(idx, par):
            idx = np.asarray(s[idx], np.int64)
            return self.t(idx).T, self.t(_f32(s[par])).T

        for name, idx, par in (("bond", "bonds", "bond_par"), ("ureyb", "ureyb", "ub_par")):
            if len(s[idx]):
                (i, j), (b0, kb) = rows(idx, par)
                terms[name] = kb * (torch.linalg.norm(x[i] - x[j], dim=1) - b0) ** 2
        if len(s["angles"]):
            (i, j, k), (t0, kt) = rows("angles", "angle_par")
            u, v = x[i] - x[j], x[k] - x[j]
            c = (u * v).sum(1) / (torch.linalg.norm(u, dim=1) * torch.linalg.norm(v, dim=1))
            terms["angle"] = kt * (torch.acos(c.clamp(-0.999, 0.999)) - t0) ** 2
        for name, idx, par in (("dihe", "dihe", "dihe_par"), ("imdihe", "imp", "imp_par")):
            if not len(s[idx]):
                continue
            (i, j, k, l), (n, kc, delta) = rows(idx, par)
            F, G, H = x[i] - x[j], x[j] - x[k], x[l] - x[k]
            A, B = torch.linalg.cross(F, G), torch.linalg.cross(H, G)
            phi = torch.atan2(torch.linalg.norm(G, dim=1) * (A * H).sum(1), (A * B).sum(1))
            wrapped = torch.remainder(phi - delta + math.pi, 2.0 * math.pi) - math.pi
            cosine = kc * (1.0 + torch.cos(n * phi - delta))
            flat = kc * wrapped ** 2 if name == "imdihe" else kc + 0.0 * phi
            terms[name] = torch.where(n != 0, cosine, flat)
        if terms:
            g, = torch.autograd.grad(sum(v.sum() for v in terms.values()), x)
            self.g += g
            self.w -= self.x.T @ g
            for k, v in terms.items():
                self.e[k] = float(v.detach().sum())

    def recip(self):
        K = [int(k) for k in self.s["fft_grid"]]
        th, dth, at = [], [], []
        for k in range(3):
            f = self.x[:, k] / self.L[k] + 0.5
            f = K[k] * (f - torch.floor(f))
            i = torch.floor(f)
            w = f - i
            th.append(torch.stack([(1 - w) ** 3, 4 - 6 * w ** 2 + 3 * w ** 3,
                                   1 + 3 * w + 3 * w ** 2 - 3 * w ** 3, w ** 3], 1) / 6.0)
            dth.append(torch.stack([-(1 - w) ** 2, -4 * w + 3 * w ** 2, 1 + 2 * w - 3 * w ** 2,
                                    w ** 2], 1) / 2.0)
            at.append((i.long()[:, None] + torch.arange(4, device=self.dev)) % K[k])
        idx = ((at[2][:, :, None, None] * K[1] + at[1][:, None, :, None]) * K[0] +
               at[0][:, None, None, :])
        prod = lambda a, b, c: a[:, None, None, :] * b[:, None, :, None] * c[:, :, None, None]
        Q = torch.zeros(K[0] * K[1] * K[2], dtype=torch.float64, device=self.dev)
        Q.index_add_(0, idx.reshape(-1),
                     (self.q[:, None, None, None] * prod(th[0], th[1], th[2])).reshape(-1))
        Qk = torch.fft.rfftn(Q.reshape(K[2], K[1], K[0]))
        m, pre = [], []
        for k in range(3):
            c = torch.arange(K[k], dtype=torch.float64, device=self.dev)
            pre.append(((4.0 + 2.0 * torch.cos(2.0 * math.pi * c / K[k])) / 6.0) ** -2)
            half = K[k] // 2 + K[k] % 2
            m.append(torch.where(c >= half, c - K[k], c) / self.L[k])
        H = K[0] // 2 + 1
        mx, my, mz = m[0][None, None, :H], m[1][None, :, None], m[2][:, None, None]
        msq = mx ** 2 + my ** 2 + mz ** 2
        msq[0, 0, 0] = 1.0
        V = float(torch.prod(self.L))
        fac = math.pi ** 2 / self.kappa ** 2
        e = torch.exp(-fac * msq) / (math.pi * V * msq)
        e = e * pre[0][None, None, :H] * pre[1][None, :, None] * pre[2][:, None, None]
        e[0, 0, 0] = 0.0
        t = e * (Qk.real ** 2 + Qk.imag ** 2)
        t[:, :, 1:] *= 2.0  # the half grid's columns stand for both halves
        self.e["ewks"] = 0.5 * CCELEC * float(t.sum())
        v = 2.0 * (fac + 1.0 / msq)
        mm = (mx, my, mz)
        for a in range(3):
            for b in range(3):
                y = t * (v * mm[a] * mm[b] - (1.0 if a == b else 0.0))
                self.w[a, b] -= 0.5 * CCELEC * y.sum()
        phi = torch.fft.irfftn(Qk * e, s=(K[2], K[1], K[0])).reshape(-1) * (K[0] * K[1] * K[2])
        p = phi[idx]
        for k in range(3):
            f = [dth[c] if c == k else th[c] for c in range(3)]
            self.g[:, k] += self.q * CCELEC * K[k] / self.L[k] * (p * prod(*f)).sum((1, 2, 3))

    def all(self):
        excluded, in14, ex14 = _exclusions(self.n, self.s["bonds"])
        self.direct(excluded)
        self.listed_pairs(in14, ("elec", float(self.s["e14fac"]) - 1.0), True)
        self.listed_pairs(ex14, ("ewex", -1.0))
        self.bonded()
        self.recip()
        self.e["ewse"] = -self.kappa * CCELEC / math.sqrt(math.pi) * float((self.q ** 2).sum())
        self.e["epot"] = sum(self.e.values())
        return self


def exact(case, seed):
    if case["call"] == "md":
        return None  # a trajectory is no closed form
    spec, x = _coordinates(case, seed)
    r = _Exact(spec, systems.xyzq_of(spec, x)).all()
    out = dict(gradient=r.g)
    if case["energy"]:
        out["energy"] = {k: torch.tensor(v, dtype=torch.float64) for k, v in r.e.items()}
    if case["virial"]:
        out["virial"] = r.w
    return out
