"""GPU paths of the Verlet-list kernels that are chosen by the system's size, against the CPU
oracle: at the sizes where the choice changes and with remainders."""
import numpy as np
import pytest

import oracle_bind as ob
from conftest import product

pytestmark = pytest.mark.gpu

FORCE_RTOL = 1e-12  # FP64 sums of ~60 pair forces in another order (normwise relative)
MIXED = dict(ntypes=2, epsilon_per_type=[1.0, 0.5], sigma_per_type=[1.0, 0.88])


def _oracle_force(sim, st, half):
    a = sim.atom
    nl, nall = a.Nlocal, a.Nlocal + a.Nghost
    nt = a.ntypes
    types = np.zeros(nall, np.int32)
    types[:nl] = sim.types()
    types[nl:] = types[st["border_map"]]
    tab = [np.ctypeslib.as_array(getattr(a, k), (nt * nt,)).copy()
           for k in ("epsilon", "sigma6", "cutforcesq")]
    f, e, w = ob.force_lj(nl, st["x"], types, nt, *tab, st["numneigh"], st["neighbors"], half)
    return f[:3 * nl], e, w


def _ghosts_follow_owners(sim, st):
    """x of every ghost = its owner's x plus its shift times the box, the same FP64 operations."""
    nl = st["nlocal"]
    p = sim.param
    x = st["x"].reshape(-1, 3)
    pbc = st["pbc"].reshape(-1, 3)
    want = x[st["border_map"]] + pbc * np.array([p.xprd, p.yprd, p.zprd])
    np.testing.assert_array_equal(x[nl:], want)


@pytest.mark.parametrize("mixed", [0, 1], ids=["uniform", "types"])
@pytest.mark.parametrize("dims", [(4, 4, 4), (5, 9, 8), (11, 11, 11), (13, 11, 9), (21, 17, 18),
                                  (29, 27, 27)], ids=str)
def test_full_list_forces_at_each_lane_count(dims, mixed):
    """64, 64, 32, 16, 8 and 4 lanes per atom; a fused run leaves the ghosts with their owners."""
    P = product()
    print(dims, mixed, flush=True)
    sim = P.VLSim(nx=dims[0], ny=dims[1], nz=dims[2], reneigh_every=5, **(MIXED if mixed else {}))
    try:
        sim.run(13)
        st = sim.state()
        want, _, _ = _oracle_force(sim, st, 0)
        assert np.linalg.norm(want) > 10.0
        assert np.linalg.norm(st["f"] - want) < FORCE_RTOL * np.linalg.norm(want)
        _ghosts_follow_owners(sim, st)
        # the fused call itself, without a ghost update after it
        L = P.lib()
        L.computeForceFinalInitialGFX950(sim.param_p, sim.atom_p, sim.neighbor_p, sim.stats_p)
        _ghosts_follow_owners(sim, sim.state())
    finally:
        sim.close()
