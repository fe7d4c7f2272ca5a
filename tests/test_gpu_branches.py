"""Every way a force call may run its branches gives the same gradient bits: on
one stream, forked, captured in a graph, with the bonded and 1-4 terms in the
pair kernel's launch or in their own, and as separate calls per group of terms.
All sums are int64, so the comparison is exact."""
import ctypes

import numpy as np
import pytest

from apocharmm_amd import _lib, systems

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# atoms: below and above the sizes at which captured calls stop merging (10,000)
# and eager calls start to fork (33,000 without energies)
@pytest.mark.parametrize("n_waters", [40, 3300, 3400, 11300])
def test_branch_plans_give_the_same_bits(n_waters):
    from apocharmm_amd.force_manager import ForceManager
    L = max(26.0, (n_waters / systems.WATER_DENSITY) ** (1.0 / 3.0))
    spec = systems.tip3p_box(n_waters, L, systems.smooth_grid(L), seed=n_waters)
    print("branch plans, atoms", 3 * n_waters, flush=True)
    fm = ForceManager(spec).initialize()
    x = torch.tensor(systems.xyzq_of(spec), device="cuda")
    fm.calcForce(x, reset=True)
    eager = fm.force.clone()
    # with energies and the virial: other kernels, the bonded terms on their own
    fm.calcForce(x, calcEnergy=True, calcVirial=True)
    assert torch.equal(fm.force, eager)
    # group by group
    total = torch.zeros_like(eager)
    for t in (_lib.APO_TERM_DIRECT, _lib.APO_TERM_RECIP, _lib.APO_TERM_BONDED,
              _lib.APO_TERM_PAIRS14):
        fm.calcForce(x, terms=t)
        total += fm.force
    assert torch.equal(total, eager)
    for t in (_lib.APO_TERM_DIRECT | _lib.APO_TERM_BONDED,
              _lib.APO_TERM_RECIP | _lib.APO_TERM_PAIRS14):
        fm.calcForce(x, terms=t)
        total -= fm.force
    assert not total.any()
    # accumulated onto a caller's own entries
    fm.force.fill_(5)
    _lib.check(_lib.lib().apo_nb_calc_force(
        fm._handle, ctypes.c_void_p(x.data_ptr()), 1 << 3, ctypes.c_void_p(fm.force.data_ptr()),
        fm.stride, None, None, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    n = fm.natom
    rows = fm.force.view(3, fm.stride)[:, :n]
    assert torch.equal(rows, eager.view(3, fm.stride)[:, :n] + 5)
    # with kernel timers on
    _lib.check(_lib.lib().apo_nb_profile(fm._handle, 1))
    fm.calcForce(x)
    _lib.check(_lib.lib().apo_nb_profile(fm._handle, 0))
    assert torch.equal(fm.force, eager)
    # captured, replayed with eager work in between
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        fm.calcForce(x)
    for _ in range(3):
        fm.force.fill_(7)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(fm.force, eager)
        fm.calcForce(x, calcEnergy=True)
        assert np.isfinite(fm.getPotentialEnergy())
    del g
    fm.close()
