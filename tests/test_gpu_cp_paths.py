"""GPU paths of the cluster-pair kernels that are chosen by size, precision and list type, against
the CPU oracle and against the separate calls they replace."""
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
