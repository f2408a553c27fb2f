"""GPU paths of the Verlet-list kernels that are chosen by the system's size, against the CPU
oracle: at the sizes where the choice changes and with remainders."""
import ctypes as C

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


@pytest.mark.parametrize("mixed", [0, 1], ids=["uniform", "types"])
@pytest.mark.parametrize("resort", [0, 10], ids=["lattice", "sorted"])
def test_staged_positions_of_large_full_lists(resort, mixed):
    """The size from which a block's neighbours are staged in LDS, with a last block of 92 atoms;
    in the bin sort's order most blocks name more atoms than the stage holds."""
    P = product()
    print(resort, mixed, flush=True)
    sim = P.VLSim(nx=53, ny=57, nz=51, reneigh_every=10, resort_every=resort,
                  **(MIXED if mixed else {}))
    try:
        sim.run(13)
        st = sim.state()
        assert st["nlocal"] == 616284
        want, _, _ = _oracle_force(sim, st, 0)
        assert np.linalg.norm(want) > 10.0
        assert np.linalg.norm(st["f"] - want) < FORCE_RTOL * np.linalg.norm(want)
        _ghosts_follow_owners(sim, st)
    finally:
        sim.close()


@pytest.mark.parametrize("mixed", [0, 1], ids=["uniform", "types"])
@pytest.mark.parametrize("dims", [(4, 4, 4), (13, 13, 15), (15, 14, 16), (21, 17, 18),
                                  (29, 27, 27)], ids=str)
def test_half_list_forces_at_each_lane_count(dims, mixed):
    """32, 16, 16, 8 and 4 lanes per atom; the fused run moves atoms and ghosts; energies."""
    P = product()
    print(dims, mixed, flush=True)
    sim = P.VLSim(nx=dims[0], ny=dims[1], nz=dims[2], half_neigh=1, reneigh_every=5,
                  **(MIXED if mixed else {}))
    try:
        sim.run(13)
        st = sim.state()
        want, e, w = _oracle_force(sim, st, 1)
        assert np.linalg.norm(want) > 10.0
        assert np.linalg.norm(st["f"] - want) < FORCE_RTOL * np.linalg.norm(want)
        _ghosts_follow_owners(sim, st)
        L = P.lib()
        L.requestEnergyVirialGFX950(1)
        sim.compute_force()
        eg, wg = sim.energy_virial()
        L.requestEnergyVirialGFX950(0)
        assert abs(eg - e) <= 1e-11 * abs(e) and abs(wg - w) <= 1e-11 * abs(w)
        assert np.linalg.norm(sim.state(lists=False)["f"] - want) < \
            FORCE_RTOL * np.linalg.norm(want)
        L.computeForceFinalInitialGFX950(sim.param_p, sim.atom_p, sim.neighbor_p, sim.stats_p)
        _ghosts_follow_owners(sim, sim.state())
    finally:
        sim.close()


def test_half_list_run_follows_full_list_run():
    """The same trajectory from a half and a full list (FP64 sums in different orders), with the
    half list's in-place integration against the full list's two buffers."""
    P = product()
    out = []
    for half in (0, 1):
        sim = P.VLSim(nx=6, ny=7, nz=5, half_neigh=half, reneigh_every=7)
        try:
            sim.run(10)
            sim.run(15)
            st = sim.state(lists=False)
            out.append([st[k][:3 * st["nlocal"]] for k in ("x", "v", "f")])
        finally:
            sim.close()
    for a, b in zip(*out):
        np.testing.assert_allclose(a, b, rtol=0, atol=1e-10 * max(1.0, np.abs(b).max()))


@pytest.mark.parametrize("n", [300, 5000])
def test_half_list_of_scattered_neighbours(n):
    """Random lists (main-stub's rand pattern): a block's atoms touch more others than its LDS
    table holds, so the rest go to memory; first and last atom against the oracle."""
    import ctypes
    P = product()
    nn = 38
    res = P.stub_run("rand", n, nn, 1, ntimes=2, half=1)
    libc = ctypes.CDLL(None)
    libc.srand(1)
    for _ in range(n):
        libc.rand()  # the types
    lists = np.empty((n, nn), np.int32)
    for i in range(n):
        seen = set()
        for k in range(nn):
            j = libc.rand() % n
            while j == i or j in seen:
                j = libc.rand() % n
            seen.add(j)
            lists[i, k] = j
    x = np.repeat(np.arange(n) * 1e-5, 3)
    one = np.ones(16)
    f, _, _ = ob.force_lj(n, x, np.zeros(n, np.int32), 4, one, one, one * 1e12,
                          np.full(n, nn, np.int32), lists.reshape(-1), 1)
    # a handful of close pairs make up each sum: 1e-11 relative covers its reordering
    assert abs(res["f0"] - f[0]) <= 1e-11 * abs(f[0])
    assert abs(res["flast"] - f[3 * (n - 1)]) <= 1e-11 * abs(f[3 * (n - 1)])


@pytest.mark.parametrize("dims", [(4, 4, 5), (11, 11, 11), (17, 17, 15), (20, 19, 21),
                                  (22, 22, 21)], ids=str)
def test_eam_forces_and_energies_at_each_lane_count(dims, tmp_path):
    """64, 32, 16, 8 lanes per atom with the rows from L2, and the LDS-table passes; the energy
    passes beside them; ghosts moved by the fused call."""
    P = product()
    print(dims, flush=True)
    path = str(tmp_path / "cu.eam")
    P.lib().mdbWriteFuncflSynthetic(path.encode())
    tab = ob.EamTables(path)
    sim = P.VLSim(nx=dims[0], ny=dims[1], nz=dims[2], force_field=1, lattice_a=3.615, temp=1600.0,
                  maxwell_seed=5, reneigh_every=5, eam_file=path)
    try:
        sim.run(13)
        st = sim.state()
        nl = st["nlocal"]
        cut = sim.param.cutforce ** 2
        want, ea = ob.force_eam_atom(tab, nl, st["x"], st["border_map"], cut, st["numneigh"],
                                     st["neighbors"])
        want = want[:3 * nl]
        assert np.linalg.norm(want) > 10.0
        assert np.linalg.norm(st["f"] - want) < FORCE_RTOL * np.linalg.norm(want)
        _ghosts_follow_owners(sim, st)
        e = sim.eam_atom_energy()
        assert np.linalg.norm(e - ea) < FORCE_RTOL * np.linalg.norm(ea)
        assert np.linalg.norm(sim.state(lists=False)["f"] - want) < \
            FORCE_RTOL * np.linalg.norm(want)
        P.lib().computeForceFinalInitialGFX950(sim.param_p, sim.atom_p, sim.neighbor_p,
                                               sim.stats_p)
        _ghosts_follow_owners(sim, sim.state())
    finally:
        sim.close()


@pytest.mark.parametrize("half", [0, 1])
@pytest.mark.parametrize("case", [dict(nx=4, ny=4, nz=4), dict(nx=19, ny=18, nz=17),
                                  dict(nx=19, ny=18, nz=19), dict(nx=5, ny=5, nz=5, skin=3.0),
                                  dict(nx=7, ny=6, nz=8, squeeze=0.5)], ids=str)
def test_lists_equal_the_oracles_on_moved_atoms(case, half):
    """Both list builds (one block or one wavefront per bin): small, below and above the size
    where the choice changes, stencils of many columns, bins of more than 32 atoms."""
    P = product()
    print(case, half, flush=True)
    x0, _, _ = P.create_lattice(**{k: case[k] for k in ("nx", "ny", "nz")})
    squeeze = case.get("squeeze", 1.0)  # all atoms in one corner of the box
    sim = P.VLSim(half_neigh=half, reneigh_every=1000,
                  **{k: v for k, v in case.items() if k != "squeeze"})
    try:
        n = sim.atom.Nlocal
        L = P.lib()
        p = sim.param
        prd = np.array([p.xprd, p.yprd, p.zprd])
        rng = np.random.default_rng(9)
        x = x0.reshape(-1, 3) + rng.uniform(-0.15, 0.15, (n, 3))
        x = squeeze * np.where(x < 0, x + prd, np.where(x >= prd, x - prd, x))
        host = np.ctypeslib.as_array(sim.atom.x, (3 * n,))
        host[:] = x.reshape(-1)
        nghost, sim.atom.Nghost = sim.atom.Nghost, 0  # the host copies hold the local atoms only
        L.copyDataToGFX950Device(sim.param_p, sim.atom_p)
        L.updateAtomsPbcGFX950(sim.atom_p, sim.param_p, True)
        L.setupPbcGFX950(sim.atom_p, sim.param_p)
        L.updatePbcGFX950(sim.atom_p, sim.param_p, True)
        L.buildNeighborGFX950(sim.atom_p, sim.neighbor_p)
        st = sim.state()
        np.testing.assert_array_equal(st["x"][:3 * n], x.reshape(-1))
        _ghosts_follow_owners(sim, st)
        g = ob.vl_grid(case["nx"], case["ny"], case["nz"], p.lattice, p.cutneigh)
        start, atoms = sim.bins()
        nn, nb = ob.build_neighbor(g, n, st["x"], np.zeros(n + st["nghost"], np.int32), 4,
                                   np.full(16, p.cutneigh ** 2), half, cap_per_atom=2000)
        np.testing.assert_array_equal(st["numneigh"], nn)
        np.testing.assert_array_equal(st["neighbors"], nb)
        if "squeeze" in case:
            assert np.diff(start).max() > 32
        if "skin" in case:
            assert nghost > 0 and nn.max() > 200
    finally:
        sim.close()


@pytest.mark.parametrize("half", [0, 1])
@pytest.mark.parametrize("case", [dict(nx=4, ny=4, nz=4), dict(nx=10, ny=10, nz=10),
                                  dict(nx=12, ny=13, nz=13), dict(nx=13, ny=13, nz=13),
                                  dict(nx=25, ny=24, nz=11), dict(nx=5, ny=5, nz=5, squeeze=0.2),
                                  dict(nx=13, ny=13, nz=13, squeeze=(0.12, 1.0, 1.0))], ids=str)
def test_lists_of_a_runs_rebuild(case, half):
    """The rebuild inside a run, in few launches or many by the size; squeezed into a corner (or a slab)
    the atoms have seven (or about two) images each, more than there was room for, and the lists
    outgrow theirs too."""
    P = product()
    print(case, half, flush=True)
    dims = {k: case[k] for k in ("nx", "ny", "nz")}
    sim = P.VLSim(half_neigh=half, reneigh_every=1 if "squeeze" in case else 3, **dims)
    try:
        n = sim.atom.Nlocal
        p = sim.param
        ghosts0 = sim.atom.Nghost
        if "squeeze" in case:
            x0, _, _ = P.create_lattice(**dims)
            np.ctypeslib.as_array(sim.atom.x, (3 * n,))[:] = \
                (np.array(case["squeeze"]) * x0.reshape(-1, 3)).reshape(-1)
            sim.atom.Nghost = 0  # the host copies hold the local atoms only
            P.lib().copyDataToGFX950Device(sim.param_p, sim.atom_p)
            sim.run(1)
        else:
            sim.run(3)
        st = sim.state()
        _ghosts_follow_owners(sim, st)
        if "squeeze" in case:
            assert st["nghost"] > 1.5 * ghosts0
        nn, nb = ob.build_neighbor(ob.vl_grid(case["nx"], case["ny"], case["nz"], p.lattice,
                                              p.cutneigh), n, st["x"],
                                   np.zeros(n + st["nghost"], np.int32), 4,
                                   np.full(16, p.cutneigh ** 2), half, cap_per_atom=2500)
        np.testing.assert_array_equal(st["numneigh"], nn)
        np.testing.assert_array_equal(st["neighbors"], nb)
    finally:
        sim.close()


@pytest.mark.parametrize("kind", ["lj", "lj-half", "eam", "eam-table"])
def test_atoms_at_one_place(kind):
    """Two atoms at distance zero: the fast kernels' reciprocals have no special cases, so their forces
    have to be no numbers where the strict kernels' are, and the other atoms' the strict ones."""
    P = product()
    print(kind, flush=True)
    n = 22 if kind == "eam-table" else 6
    kw = dict(force_field=1, lattice_a=3.615, temp=300.0, maxwell_seed=5) if "eam" in kind else \
        dict(half_neigh=int(kind == "lj-half"))
    sim = P.VLSim(nx=n, ny=n, nz=n, reneigh_every=1000, **kw)
    L = P.lib()
    try:
        nl = sim.atom.Nlocal
        x = sim.state(lists=False)["x"][:3 * nl].copy()
        x[300:303] = x[0:3]
        np.ctypeslib.as_array(sim.atom.x, (3 * nl,))[:] = x
        sim.atom.Nghost = 0  # the host copies hold the local atoms only
        L.copyDataToGFX950Device(sim.param_p, sim.atom_p)
        L.updateAtomsPbcGFX950(sim.atom_p, sim.param_p, True)
        L.setupPbcGFX950(sim.atom_p, sim.param_p)
        L.buildNeighborGFX950(sim.atom_p, sim.neighbor_p)
        sim.compute_force()
        fast = sim.state(lists=False)["f"].reshape(-1, 3)
        L.mdgfx950SetStrict(1)
        sim.compute_force()
        strict = sim.state(lists=False)["f"].reshape(-1, 3)
        bad = ~np.isfinite(strict)
        assert bad.any(axis=1).sum() == 2 and bad[0].all() and bad[100].all()
        np.testing.assert_array_equal(~np.isfinite(fast), bad)
        assert np.linalg.norm((fast - strict)[~bad]) < FORCE_RTOL * np.linalg.norm(strict[~bad])
    finally:
        L.mdgfx950SetStrict(0)
        sim.close()


@pytest.mark.parametrize("dims", [(18, 17, 17), (22, 22, 21)], ids=str)
def test_eam_tables_too_long_for_lds(dims, tmp_path):
    """2400 rows: 8 and 4 lanes per atom with the rows from L2."""
    P = product()
    print(dims, flush=True)
    path = tmp_path / "cu.eam"
    P.lib().mdbWriteFuncflSynthetic(str(path).encode())
    lines = path.read_text().split("\n")
    nrho, drho, nr, dr, rc = lines[2].split()
    n, m = int(nr), 2400
    vals = np.array(" ".join(lines[3:]).split(), float).reshape(3, n)
    fine = np.arange(m) * float(dr) * n / m
    rows = [vals[0]] + [np.interp(fine, np.arange(n) * float(dr), v) for v in vals[1:]]
    path.write_text("\n".join(lines[:2] + ["%s %s %d %.16e %s" % (nrho, drho, m, fine[1], rc)] +
                              ["%.16e" % v for r in rows for v in r]) + "\n")
    tab = ob.EamTables(str(path))
    sim = P.VLSim(nx=dims[0], ny=dims[1], nz=dims[2], force_field=1, lattice_a=3.615, temp=1600.0,
                  maxwell_seed=5, reneigh_every=5, eam_file=str(path))
    try:
        sim.run(6)
        st = sim.state()
        want, _ = ob.force_eam_atom(tab, st["nlocal"], st["x"], st["border_map"],
                                    sim.param.cutforce ** 2, st["numneigh"], st["neighbors"])
        want = want[:3 * st["nlocal"]]
        assert np.linalg.norm(want) > 10.0
        assert np.linalg.norm(st["f"] - want) < FORCE_RTOL * np.linalg.norm(want)
        _ghosts_follow_owners(sim, st)
    finally:
        sim.close()


def _put(sim, x):
    """The sim's local atoms to x, without ghosts."""
    nl = sim.atom.Nlocal
    np.ctypeslib.as_array(sim.atom.x, (3 * nl,))[:] = x
    sim.atom.Nghost = 0  # the host copies hold the local atoms only
    product().lib().copyDataToGFX950Device(sim.param_p, sim.atom_p)


@pytest.mark.parametrize("call", ["calls", "run"])
@pytest.mark.parametrize("dims", [(4, 4, 4), (10, 10, 10), (16, 16, 16), (19, 18, 19)], ids=str)
def test_atom_outside_the_grid_is_an_error(dims, call):
    """An atom many boxes away is in no bin, so its list would stay the last one: the rebuild says so,
    by the separate calls and inside a run, at each of the binnings and list builds; no force call
    follows it.  With the atom back the next rebuild gives the oracle's lists."""
    P = product()
    L = P.lib()
    print(dims, call, flush=True)
    sim = P.VLSim(nx=dims[0], ny=dims[1], nz=dims[2], reneigh_every=1)
    try:
        p = sim.param
        nl = sim.atom.Nlocal
        good = sim.state(lists=False)["x"][:3 * nl].copy()
        far = good.copy()
        far[3 * 7 + 2] += 50 * p.zprd

        def rebuild():
            if call == "run":
                return L.mdbVLRun(sim.h, 1, None)
            L.updateAtomsPbcGFX950(sim.atom_p, sim.param_p, True)
            L.setupPbcGFX950(sim.atom_p, sim.param_p)
            L.updatePbcGFX950(sim.atom_p, sim.param_p, True)
            L.buildNeighborGFX950(sim.atom_p, sim.neighbor_p)
            return P.status()[0]

        _put(sim, far)
        assert rebuild() == 2  # MDG_ERR_BIN
        assert "outside the bin grid" in P.status()[1]
        L.mdgfx950ClearStatus()
        _put(sim, good)
        assert rebuild() == 0, P.status()
        st = sim.state()
        nn, nb = ob.build_neighbor(ob.vl_grid(*dims, p.lattice, p.cutneigh), nl, st["x"],
                                   np.zeros(nl + st["nghost"], np.int32), 4,
                                   np.full(16, p.cutneigh ** 2), 0, cap_per_atom=2000)
        np.testing.assert_array_equal(st["numneigh"], nn)
        np.testing.assert_array_equal(st["neighbors"], nb)
    finally:
        L.mdgfx950ClearStatus()
        sim.close()


def _hip():
    hip = C.CDLL("libamdhip64.so.7")  # the runtime libmdgfx950.so is linked against
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    return hip


@pytest.mark.parametrize("fused", [0, 1])
@pytest.mark.parametrize("dims", [(4, 4, 4), (15, 14, 16), (29, 27, 27)], ids=str)
def test_half_list_call_leaves_zero_forces_on_ghosts(dims, fused):
    """A half-list call gives every atom's row of the device's forces: a ghost's is zero, whatever the
    buffer held."""
    P = product()
    L = P.lib()
    hip = _hip()
    print(dims, fused, flush=True)
    sim = P.VLSim(nx=dims[0], ny=dims[1], nz=dims[2], half_neigh=1, reneigh_every=5)
    try:
        nl, ng = sim.atom.Nlocal, sim.atom.Nghost
        f = np.full(3 * (nl + ng), np.nan)
        L.mdgfx950Synchronize()
        fx = C.cast(sim.atom.d_atom.fx, C.c_void_p)
        assert hip.hipMemcpy(fx, f.ctypes.data, f.nbytes, 1) == 0
        if fused:
            L.computeForceFinalInitialGFX950(sim.param_p, sim.atom_p, sim.neighbor_p, sim.stats_p)
        else:
            sim.compute_force()
        L.mdgfx950Synchronize()
        assert hip.hipMemcpy(f.ctypes.data, fx, f.nbytes, 2) == 0
        assert ng > 0 and np.isfinite(f[:3 * nl]).all()
        np.testing.assert_array_equal(f[3 * nl:], 0.0)
    finally:
        sim.close()


@pytest.mark.parametrize("half", [0, 1])
@pytest.mark.parametrize("nx,wide", [(6, 1.0), (8, 1.5), (8, 4.0), (20, 1.0)])
def test_lists_in_boxes_of_many_bins(nx, wide, half, tmp_path):
    """Boxes read from a file (bins of half the list cutoff, none to a few atoms each), and a droplet in
    a box whose bins are mostly empty, around the number of bins where the list build changes: the
    lists name the pairs inside the cutoff, at setup and after a run's rebuild."""
    from scipy.spatial import cKDTree
    P = product()
    print(nx, wide, half, flush=True)
    x, v, t = P.create_lattice(nx=nx, ny=nx, nz=nx)
    side = nx * (4 / 0.8442) ** (1 / 3) * wide
    rng = np.random.default_rng(nx)
    x = np.mod(x + rng.uniform(-0.2, 0.2, x.size) + side / 3, side)
    path = str(tmp_path / "a.dmp")
    P.write_dmp(path, x, 0.01 * v, t, [0.0, side] * 3)
    sim = P.VLSim(input_file=path, half_neigh=half, reneigh_every=2, dt=1e-5)
    try:
        bins = sim.bins()[0].size - 1
        assert (bins > 16384) == ((nx, wide) != (6, 1.0))
        for steps in (0, 2):
            if steps:
                sim.run(steps)
            st = sim.state()
            pos = st["x"].reshape(-1, 3)
            nl = st["nlocal"]
            _ghosts_follow_owners(sim, st)
            cn = sim.param.cutneigh ** 2
            near = cKDTree(pos[:nl]).query_ball_tree(cKDTree(pos), sim.param.cutneigh * (1 + 1e-9))
            i = np.repeat(np.arange(nl), [len(q) for q in near])
            j = np.concatenate([np.asarray(q, np.int64) for q in near])
            d = pos[i] - pos[j]
            rsq = d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]
            keep = (i != j) & (rsq <= cn) & ((j > i) if half else True)
            want = np.sort(i[keep] * (1 << 32) + j[keep])
            got = np.repeat(np.arange(nl), st["numneigh"]) * (1 << 32) + st["neighbors"]
            np.testing.assert_array_equal(np.sort(got), want)
    finally:
        sim.close()


@pytest.mark.parametrize("dims", [(6, 6, 6), (7, 6, 6), (9, 9, 9), (13, 13, 14), (14, 14, 14)], ids=str)
def test_eam_energies_at_each_lane_count(dims, tmp_path):
    """32, 16, 16, 8 and 4 lanes per atom in the passes with energies."""
    P = product()
    L = P.lib()
    print(dims, flush=True)
    path = str(tmp_path / "cu.eam")
    L.mdbWriteFuncflSynthetic(path.encode())
    tab = ob.EamTables(path)
    sim = P.VLSim(nx=dims[0], ny=dims[1], nz=dims[2], force_field=1, lattice_a=3.615, temp=1600.0,
                  maxwell_seed=5, reneigh_every=5, eam_file=path)
    try:
        sim.run(13)
        st = sim.state()
        want, ea = ob.force_eam_atom(tab, st["nlocal"], st["x"], st["border_map"],
                                     sim.param.cutforce ** 2, st["numneigh"], st["neighbors"])
        want = want[:3 * st["nlocal"]]
        L.requestEnergyVirialGFX950(1)
        e = sim.eam_atom_energy()
        total, _ = sim.energy_virial()
        L.requestEnergyVirialGFX950(0)
        assert np.linalg.norm(e - ea) < FORCE_RTOL * np.linalg.norm(ea)
        assert abs(total - ea.sum()) < 1e-11 * abs(ea.sum())
        assert np.linalg.norm(sim.state(lists=False)["f"] - want) < \
            FORCE_RTOL * np.linalg.norm(want)
    finally:
        L.requestEnergyVirialGFX950(0)
        sim.close()


def test_foreign_list_under_staging_tables():
    """A list uploaded over one that was built with staging tables (same size, so the tables stay): its
    entries in another order, some dropped, some rows emptied or made of far atoms; the forces are
    that list's."""
    P = product()
    L = P.lib()
    sim = P.VLSim(nx=51, ny=51, nz=51, reneigh_every=1000)
    nb = sim.neighbor
    host = (nb.neighbors, nb.numneigh)
    try:
        sim.run(2)
        st = sim.state()
        nl, mn = st["nlocal"], nb.maxneighs
        assert nl == 530604  # above the size from which the lists have tables
        start = np.concatenate([[0], np.cumsum(st["numneigh"], dtype=np.int64)])
        row = np.repeat(np.arange(nl), st["numneigh"])
        k = np.arange(row.size) - start[row]
        keep = (k % 7 != 3) & (row % 1000 != 5)
        count = np.bincount(row[keep], minlength=nl).astype(np.int32)
        at = np.arange(keep.sum()) - np.concatenate([[0], np.cumsum(count, dtype=np.int64)])[row[keep]]
        lists = np.zeros((nl, mn), np.int32)
        # backwards, so that every entry is in another place
        lists[row[keep], count[row[keep]] - 1 - at] = st["neighbors"][keep]
        for i in range(9, nl, 5000):
            count[i] = min(mn, 40)
            lists[i, :count[i]] = (i + 7919 * np.arange(1, count[i] + 1)) % nl
        csr = lists[np.arange(mn) < count[:, None]]
        nb.neighbors = lists.ctypes.data_as(C.POINTER(C.c_int))
        nb.numneigh = count.ctypes.data_as(C.POINTER(C.c_int))
        L.uploadNeighborGFX950.argtypes = [C.c_void_p, C.c_void_p]
        L.uploadNeighborGFX950(sim.atom_p, sim.neighbor_p)
        assert nb.maxneighs == mn
        sim.compute_force()
        one = np.ones(16)
        want, _, _ = ob.force_lj(nl, st["x"], np.zeros(nl + st["nghost"], np.int32), 4, one, one,
                                 one * 6.25, count, csr, 0)
        want = want[:3 * nl]
        got = sim.state(lists=False)["f"]
        assert np.linalg.norm(want) > 10.0
        assert np.linalg.norm(got - want) < FORCE_RTOL * np.linalg.norm(want)
        np.testing.assert_array_equal(got.reshape(-1, 3)[5::1000][count[5::1000] == 0], 0.0)
    finally:
        nb.neighbors, nb.numneigh = host
        sim.close()
