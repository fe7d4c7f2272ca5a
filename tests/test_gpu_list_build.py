"""The pairs in the built list against a count over all pairs in float64.

The list's distance test works in float32 on 32-bit fixed-point coordinates:
each difference, square and sum rounds once (relative 6e-8), so a pair is
decided as in exact arithmetic unless its distance is within 5e-6 A of the
cutoff (r up to 17 A, five roundings).  The count has to lie between those of
the two cutoffs that far apart."""
import numpy as np
import pytest

from apocharmm_amd import _lib, systems

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
BAND = 5e-6


def _excluded(n, bonds):
    """Pairs one to three bonds apart."""
    adj = [set() for _ in range(n)]
    for a, b in bonds:
        adj[a].add(int(b))
        adj[b].add(int(a))
    out = set()
    for i in range(n):
        seen, edge = {i}, {i}
        for _ in range(3):
            edge = set().union(*(adj[k] for k in edge)) - seen
            seen |= edge
        out |= {(i, j) for j in seen if j > i}
    return np.array(sorted(out), np.int64).reshape(-1, 2)


def _dist(a, b, box):
    d = a - b
    d -= box * torch.round(d / box)
    return torch.sqrt(torch.sum(d * d, dim=-1))


def _counts(x, box, radii, ex):
    """Pairs closer than each radius, less the excluded ones."""
    x, box, ex = (torch.tensor(a, device="cuda") for a in (x, box, ex))
    c = [0] * len(radii)
    for i in range(0, len(x), 256):
        d = _dist(x[i:i + 256, None], x[None], box)
        for k, r in enumerate(radii):
            c[k] += int((d < r).sum()) - len(d)
    d = _dist(x[ex[:, 0]], x[ex[:, 1]], box)
    return [c[k] // 2 - int((d < r).sum()) for k, r in enumerate(radii)]


# box edges, list cutoff: one image per cell or not; equal and uneven edges;
# more candidate tiles than the masks in LDS hold; columns of 1,000 atoms;
# atoms piled up in z; more partner cells of exclusions than their table holds
CASES = {
    "wrapped": ((27.6, 27.6, 27.6), 13.0),
    "one_image": ((40.4, 40.4, 40.4), 14.0),
    "uneven": ((33.0, 46.0, 38.0), 12.5),
    "one_cell_row": ((21.0, 64.0, 23.0), 10.0),
    "many_tiles": ((46.0, 46.0, 46.0), 17.0),
    "tall": ((24.0, 24.0, 170.0), 11.0),
    "flat": ((40.4, 40.4, 40.4), 14.0),
    "exclusions": ((40.4, 40.4, 40.4), 14.0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_pairs_in_list(name):
    from apocharmm_amd.force_manager import ForceManager
    print("list build", name, flush=True)
    edges, cut = CASES[name]
    rng = np.random.default_rng(11)
    nw = int(np.prod(edges) * systems.WATER_DENSITY)
    spec = systems.tip3p_box(nw, 60.0, 32, seed=3, cutnb=cut, ctofnb=cut - 2.0, ctonnb=cut - 4.0)
    spec["box"] = np.array(edges, np.float64)
    n = 3 * nw
    # positions of no particular order (pairs are only counted)
    x = rng.random((n, 3)) * np.array(edges) - 0.3 * np.array(edges)
    if name == "flat":
        x[:, 2] *= 0.02
    if name == "exclusions":
        more = rng.integers(0, n, (n, 2))
        more = more[more[:, 0] != more[:, 1]]
        bonds = np.asarray(spec["bonds"]).reshape(-1, 2)
        spec["bonds"] = np.concatenate([bonds, more]).astype(bonds.dtype)
        par = np.asarray(spec["bond_par"]).reshape(-1, 2)
        spec["bond_par"] = np.concatenate([par, np.repeat(par[:1], len(more), 0)])
    xyzq = systems.xyzq_of(spec, x.astype(np.float32))
    fm = ForceManager(spec).initialize()
    t = torch.tensor(xyzq, device="cuda")
    stats = []
    for reset in (True, True):  # the build that sizes the buffers, and one into them
        fm.calcForce(t, reset=reset, terms=_lib.APO_TERM_DIRECT)
        stats.append(fm.listStats())
    fm.resetNeighborList(t)
    stats.append(fm.listStats())
    fm.close()
    assert stats[0] == stats[1] == stats[2], stats
    ex = _excluded(n, np.asarray(spec["bonds"]).reshape(-1, 2))
    x = np.asarray(xyzq, np.float64).reshape(-1, 4)[:, :3]
    box = np.array(edges)
    lo, hi = _counts(x, box, (cut - BAND, cut + BAND), ex)
    assert lo <= stats[0]["pairs_in_list"] <= hi, (lo, stats[0], hi)
