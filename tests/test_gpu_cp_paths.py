"""GPU paths of the cluster-pair kernels that are chosen by size, precision and list type, against
the CPU oracle and against the separate calls they replace."""
import ctypes as C

import numpy as np
import pytest

from conftest import product
from test_gpu_cp import KA, _live_slots, _oracle_forces, _thermalised_atoms

pytestmark = pytest.mark.gpu

MIX = dict(KA)


@pytest.mark.parametrize("N", [4, 8])
@pytest.mark.parametrize("nx", [5, 8])
def test_fp64_full_list_forces_equal_oracle(N, nx):
    """The wavefront-per-cluster FP64 kernel adds in the reference's order: equal to the bit."""
    x, v, t, lat = _thermalised_atoms(nx)
    sim = product().CPSim(nx=nx, ny=nx, nz=nx, cluster_m=4, cluster_n=N, precision=1, ntimes=0)
    try:
        sim.set_atoms(x, v, t)
        _, f64, e64, w64 = _oracle_forces(sim, 4, N, 0, lat, nx)
        live = _live_slots(sim.get("ci_natoms"), 4)
        np.testing.assert_array_equal(sim.get("slot_f").reshape(-1, 3)[live],
                                      f64.reshape(-1, 3)[live])
        e, w = sim.energy_virial()
        assert abs(e - e64) <= 1e-11 * abs(e64) and abs(w - w64) <= 1e-11 * abs(w64)
    finally:
        sim.close()


@pytest.mark.parametrize("mixture", [0, 1], ids=["lj", "ka"])
@pytest.mark.parametrize("N", [4, 8])
@pytest.mark.parametrize("nx", [4, 9])
def test_fp64_half_list_forces_equal_full_list_forces(nx, N, mixture):
    """The same clusters with half and with full lists: sums of the same ~60 FP64 pair forces in
    another order (atomics), energies of the same pairs."""
    out = []
    for half in (0, 1):
        sim = product().CPSim(nx=nx, ny=nx + 1, nz=nx, cluster_m=4, cluster_n=N, precision=1, ntimes=0,
                              half_neigh=half, **(MIX if mixture else dict(temp=0.5)))
        try:
            if half:
                sim.set_atoms(*atoms)
            else:
                sim.run(15)
                sim.run(1)
                product().lib().updateSingleAtomsGFX950(C.c_void_p(sim.param_p),
                                                        C.c_void_p(sim.atom_p))
                atoms = [sim.get("atoms_" + k).copy() for k in ("x", "v", "type")]
                sim.set_atoms(*atoms)
            live = _live_slots(sim.get("ci_natoms"), 4)
            out.append((sim.get("slot_f").reshape(-1, 3)[live], *sim.energy_virial()))
        finally:
            sim.close()
    (ff, ef, wf), (fh, eh, wh) = out
    assert np.linalg.norm(ff) > 10.0
    assert np.linalg.norm(fh - ff) < 1e-12 * np.linalg.norm(ff)
    assert abs(eh - ef) <= 1e-11 * abs(ef) and abs(wh - wf) <= 1e-11 * max(abs(wf), abs(ef))


@pytest.mark.parametrize("mixture", [0, 1], ids=["lj", "ka"])
@pytest.mark.parametrize("N", [4, 8])
def test_fp64_fused_run_equals_traced_run(N, mixture):
    """The kicks and the drift inside the FP64 force call are the separate calls' operations (a
    traced run makes those): positions, velocities and forces equal to the bit over rebuilds."""
    out = []
    for trace in (False, True):
        sim = product().CPSim(nx=6, ny=5, nz=7, cluster_m=4, cluster_n=N, precision=1, ntimes=0,
                              reneigh_every=6, **(MIX if mixture else {}))
        try:
            sim.run(10, trace=trace)
            sim.run(9, trace=trace)
            live = _live_slots(sim.get("ci_natoms"), 4)
            out.append([sim.get(k).reshape(-1, 3)[live] for k in ("slot_x", "slot_v", "slot_f")])
        finally:
            sim.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("mixture", [0, 1], ids=["lj", "ka"])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("N", [4, 8])
@pytest.mark.parametrize("nx", [4, 22, 23])
def test_fused_run_equals_traced_run_around_the_small_size(nx, N, precision, mixture):
    """Up to 12000 i-clusters (22^3 cells) a wavefront takes one i-cluster and the fused call
    moves the ghosts; above, four, and a launch of their own does.  Either way a traced run,
    which integrates and moves ghosts separately, gives the same bits, ghosts included."""
    out = []
    for trace in (False, True):
        sim = product().CPSim(nx=nx, ny=nx, nz=nx, cluster_m=4, cluster_n=N, ntimes=0,
                              precision=precision, reneigh_every=6, **(MIX if mixture else {}))
        try:
            sim.run(8, trace=trace)
            sim.run(5, trace=trace)
            i = sim.info()
            cjn = sim.get("cj_natoms")
            slots = (np.arange(cjn.size)[:, None] * N + np.arange(N))[np.arange(N) < cjn[:, None]]
            live = _live_slots(sim.get("ci_natoms"), 4)
            out.append([sim.get("slot_x").reshape(-1, 3)[slots]] +
                       [sim.get(k).reshape(-1, 3)[live] for k in ("slot_v", "slot_f")])
            assert (i["nci"] <= 12000) == (nx < 23)
        finally:
            sim.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


def test_precision_change_between_runs_keeps_one_trajectory():
    """FP32 and FP64 calls in turn on one simulation share the position buffers: the FP64 forces
    after an FP32 stretch equal those of a simulation set to the same atoms."""
    P = product()
    sim = P.CPSim(nx=5, ny=5, nz=5, precision=0, ntimes=0, reneigh_every=1000)
    try:
        for precision in (1, 0, 1, 0):
            P.lib().setClusterPrecisionGFX950(precision, 0)
            sim.run(3)
        live = _live_slots(sim.get("ci_natoms"), 4)
        f32 = sim.get("slot_f").reshape(-1, 3)[live]
        P.lib().setClusterPrecisionGFX950(1, 0)
        sim.compute_force()
        f64 = sim.get("slot_f").reshape(-1, 3)[live]
        assert np.linalg.norm(f32 - f64) < 1e-6 * np.linalg.norm(f64)
    finally:
        P.lib().setClusterPrecisionGFX950(0, 0)
        sim.close()


class _AtomHead(C.Structure):
    """The leading fields of the cluster-pair Atom (include/mdbench_cp.h)."""
    _fields_ = [(n, C.c_int) for n in ("Natoms", "Nlocal", "Nghost", "Nmax", "Nclusters_local",
                                       "Nclusters_ghost", "Nclusters_max", "NmaxGhost", "ncj")] + \
               [(n, C.POINTER(C.c_double)) for n in ("x", "y", "z", "vx", "vy", "vz")] + \
               [("border_map", C.POINTER(C.c_int)), ("type", C.POINTER(C.c_int))]


@pytest.mark.parametrize("nx", [5, 36])
def test_atoms_to_and_from_the_device(nx):
    """Small copies and copies of many chunks (186,624 atoms: 4.5 MB of positions): the arrays
    arrive whole, and the host struct follows the atoms it was given."""
    P = product()
    L = P.lib()
    sim = P.CPSim(nx=nx, ny=nx, nz=nx, ntimes=0)
    try:
        x, v, t = P.create_lattice(nx=nx, ny=nx, nz=nx)
        n = t.size
        rng = np.random.default_rng(nx)
        x = np.clip(x + rng.uniform(0, 0.1, 3 * n), 0.0, nx * (4 / 0.8442) ** (1 / 3) - 1e-6)
        v = v + rng.standard_normal(3 * n)
        t = rng.integers(0, 4, n).astype(np.int32)
        sim.set_atoms(x, v, t)
        head = _AtomHead.from_address(sim.atom_p)

        def host():
            g = lambda p, k: np.ctypeslib.as_array(p, (k,))  # noqa: E731
            return (g(head.x, 3 * n), np.stack([g(head.vx, n), g(head.vy, n), g(head.vz, n)], 1),
                    g(head.type, n))

        def device():
            return sim.get("atoms_x"), sim.get("atoms_v").reshape(-1, 3), sim.get("atoms_type")

        want = (x, v.reshape(-1, 3), t)
        for got in (device(), host()):
            for a, b in zip(got, want):
                np.testing.assert_array_equal(a, b)
        for p, k in ((head.x, 3 * n), (head.vx, n), (head.vy, n), (head.vz, n), (head.type, n)):
            np.ctypeslib.as_array(p, (k,))[:] = 0
        L.copyAtomsFromClusterGFX950Device(C.c_void_p(sim.atom_p))
        for a, b in zip(host(), want):
            np.testing.assert_array_equal(a, b)
        np.ctypeslib.as_array(head.vy, (n,))[:] += 1.5
        np.ctypeslib.as_array(head.type, (n,))[:] = t[::-1]
        L.copyAtomsToClusterGFX950Device(C.c_void_p(sim.atom_p))
        want = (x, v.reshape(-1, 3) + [0.0, 1.5, 0.0], t[::-1])
        for a, b in zip(device(), want):
            np.testing.assert_array_equal(a, b)
    finally:
        sim.close()


def _pair_at(rsq, rng):
    """A separation whose squared length, as the kernels and the oracle add it up, is rsq exactly."""
    r = np.sqrt(rsq)
    while True:
        d = rng.standard_normal(3)
        d[2] *= 1e-3
        d = np.round(d * r / np.linalg.norm(d) * 2.0 ** 49) * 2.0 ** -49
        d[1] = np.round(np.sqrt(max(rsq - d[0] ** 2 - 1e-5, 0.0)) * 2.0 ** 49) * 2.0 ** -49
        rest = rsq - (d[0] * d[0] + d[1] * d[1])
        if not 1e-6 < rest < 1e-4:
            continue
        z = np.round(np.sqrt(rest) * 2.0 ** 49)
        for k in range(-64, 65):
            d[2] = (z + k) * 2.0 ** -49
            if d[0] * d[0] + d[1] * d[1] + d[2] * d[2] == rsq:
                return d


@pytest.mark.parametrize("N", [4, 8])
def test_fp64_forces_equal_oracle_where_reciprocals_round_hardest(N):
    """Squared distances a few units in the last place below a power of two, whose reciprocals lie next
    to the middle of two doubles: two Newton steps from an estimate give the wrong one."""
    nx, rho = 6, 0.1
    x, v, t = product().create_lattice(nx=nx, ny=nx, nz=nx, rho=rho)
    x = np.round(x.reshape(-1, 3) * 2.0 ** 10) * 2.0 ** -10
    rng = np.random.default_rng(4)
    lat = (4 / rho) ** (1 / 3)
    inner = np.flatnonzero(((x > 2 * lat) & (x < 4 * lat)).all(axis=1))
    outer = np.flatnonzero(~((x > lat) & (x < 5 * lat)).all(axis=1))
    targets = [p * (1.0 - m * 2.0 ** -53) for p in (1.0, 2.0) for m in (1, 3, 5, 7, 9, 11, 13)]
    assert inner.size >= len(targets)
    for a, b, rsq in zip(inner, outer, targets):
        d = _pair_at(rsq, rng)
        x[b] = x[a] + d
        got = x[a] - x[b]
        assert got[0] * got[0] + got[1] * got[1] + got[2] * got[2] == rsq
    sim = product().CPSim(nx=nx, ny=nx, nz=nx, rho=rho, cluster_m=4, cluster_n=N, precision=1, ntimes=0)
    try:
        sim.set_atoms(x.reshape(-1), v, t)
        _, f64, _, _ = _oracle_forces(sim, 4, N, 0, lat, nx)
        live = _live_slots(sim.get("ci_natoms"), 4)
        assert np.abs(f64.reshape(-1, 3)[live]).max() > 10.0
        np.testing.assert_array_equal(sim.get("slot_f").reshape(-1, 3)[live],
                                      f64.reshape(-1, 3)[live])
    finally:
        sim.close()
