"""Performance cases of the gfx950 short-range force step, through its public entry points.

Every pass starts from atoms that the caller holds (another configuration each time), as a program
does that runs many configurations, samples snapshots or restarts from stored frames:

  kind "vl"    Verlet-list scheme (LJ or EAM).  The atoms are device tensors, written into the
               simulation's DeviceAtom arrays; ghosts, bins and lists are rebuilt, then the run
               loop takes `steps` timesteps (rebuilding every 20 steps for LJ, every 10 for EAM).
               Positions, velocities and forces come back as device tensors.  snapshot: per-atom
               energies and the whole state (lists and ghost map too) are downloaded, as the
               training-set capture does.
  kind "cp"    cluster-pair scheme.  Its atoms enter and leave through host arrays (set_atoms,
               the atom download), with 19 steps between: one rebuild interval, after which the
               atoms still have the order of the rebuild that started it.
  kind "sur"   the learned EAM surrogate on packed snapshot frames: energies and forces
               (op "predict") or one training step (op "train": gradients and updated weights).

A process holds one simulation at a time (the library's own rule), so the simulation object of a
configuration is made once and kept here, and a state holds the atoms.

Positions are the fcc lattice with uniform displacements of up to 0.12 sigma (LJ) or 0.2 A
(copper) per axis, a crystal's thermal disorder without overlaps; velocities are normal, without
centre-of-mass motion, at the workload's temperature.
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

LJ = dict(rho=0.8442, temp=1.44, dt=0.005, cut=2.5, skin=0.3, every=20, disp=0.12)
KA = dict(ntypes=2, pair_epsilon=[1.0, 1.5, 1.5, 0.5], pair_sigma=[1.0, 0.8, 0.8, 0.88],
          pair_cutoff=[2.5, 2.0, 2.0, 2.2], rho=1.2, temp=0.8, type1_fraction=0.2, type_seed=4711)
MIXED = dict(ntypes=2, epsilon_per_type=[1.0, 0.5], sigma_per_type=[1.0, 0.88])
CU = dict(a=3.615, cut=4.95, skin=1.0, dt=0.001, every=10, mass=63.55, mvv2e=1.036427e-04,
          kb=8.617343e-05, disp=0.2)
CP_STEPS = 19  # with a rebuild every 20 steps: the interval from one rebuild to the next


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest calls: 256 atoms, where a step is a few launches (unit cells of the
        # regression runs, many small replicas)
        {"name": "vl-lj-4", "kind": "vl", "nx": 4, "ny": 4, "nz": 4, "half": 0, "mixed": 0,
         "eam": 0, "steps": 100, "snapshot": 0, "temp": 1.44},
        # an ordinary box of odd, unequal sides, a half list and a two-type mixture
        {"name": "vl-lj-half-mix-21x17x25", "kind": "vl", "nx": 21, "ny": 17, "nz": 25, "half": 1,
         "mixed": 1, "eam": 0, "steps": 40, "snapshot": 0, "temp": 1.44},
        # the Verlet-list benchmark's size: 1,048,576 atoms, full list
        {"name": "vl-lj-64", "kind": "vl", "nx": 64, "ny": 64, "nz": 64, "half": 0, "mixed": 0,
         "eam": 0, "steps": 40, "snapshot": 0, "temp": 1.44},
        # training-set capture: 4000 copper atoms, 50 steps, energies, lists and state downloaded
        {"name": "eam-capture-10", "kind": "vl", "nx": 10, "ny": 10, "nz": 10, "half": 0,
         "mixed": 0, "eam": 1, "steps": 50, "snapshot": 1, "temp": 900.0},
        # the EAM benchmark's sizes: 131,072 atoms with one odd side, and 1,048,576 atoms
        {"name": "eam-32x31x33", "kind": "vl", "nx": 32, "ny": 31, "nz": 33, "half": 0,
         "mixed": 0, "eam": 1, "steps": 40, "snapshot": 0, "temp": 1600.0},
        {"name": "eam-64", "kind": "vl", "nx": 64, "ny": 64, "nz": 64, "half": 0, "mixed": 0,
         "eam": 1, "steps": 20, "snapshot": 0, "temp": 1600.0},
        # cluster pair, FP32-mixed, full list: a small box and the headline benchmark's box
        {"name": "cp-lj-6", "kind": "cp", "nx": 6, "ny": 6, "nz": 6, "n": 4, "half": 0,
         "precision": 0, "ka": 0},
        {"name": "cp-lj-64", "kind": "cp", "nx": 64, "ny": 64, "nz": 64, "n": 4, "half": 0,
         "precision": 0, "ka": 0},
        # the wide j-clusters with a half list, in an ordinary box of unequal sides
        {"name": "cp-lj-4x8-half-27x30x25", "kind": "cp", "nx": 27, "ny": 30, "nz": 25, "n": 8,
         "half": 1, "precision": 0, "ka": 0},
        # the Kob-Andersen mixture (type-pair table), and the FP64 kernel
        {"name": "cp-f64-ka-20x23x19", "kind": "cp", "nx": 20, "ny": 23, "nz": 19, "n": 4,
         "half": 0, "precision": 1, "ka": 1},
        # the surrogate: inference over 32 frames of 864 atoms, and a training step over the
        # 16 frames of 4000 atoms that the training run takes per batch
        {"name": "sur-predict-32x864", "kind": "sur", "op": "predict", "cells": 6, "frames": 32},
        {"name": "sur-train-16x4000", "kind": "sur", "op": "train", "cells": 10, "frames": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["vl", "vl", "eam", "cp", "cp", "sur"])
    if kind == "sur":
        return {"kind": "sur", "op": rng.choice(["predict", "train"]), "cells": rng.randint(4, 10),
                "frames": rng.randint(1, 15)}
    n = _log_int(rng, 5, 56)
    dims = [max(4, min(64, n + rng.randint(-max(1, n // 6), max(1, n // 6)))) for _ in range(3)]
    box = {"nx": dims[0], "ny": dims[1], "nz": dims[2]}
    if kind == "cp":
        return dict(box, kind="cp", n=rng.choice([4, 4, 8]), half=rng.choice([0, 0, 1]),
                    precision=rng.choice([0, 0, 0, 1]), ka=rng.choice([0, 0, 1]))
    if kind == "eam":
        small = max(dims) <= 12
        return dict(box, kind="vl", half=0, mixed=0, eam=1, steps=rng.randint(10, 20),
                    snapshot=int(small and rng.random() < 0.5), temp=float(rng.randint(300, 2000)))
    return dict(box, kind="vl", half=rng.choice([0, 0, 0, 1]), mixed=rng.choice([0, 0, 1]), eam=0,
                steps=rng.randint(20, 40), snapshot=0, temp=1.44)


# ------------------------------------------------------------------ the library
_modules = {}


def _module(name):
    if name not in _modules:
        if name not in sys.modules:
            path = os.path.join(REPO, "md-bench_amd", name + ".py")
            spec = importlib.util.spec_from_file_location(name, path)
            mod = importlib.util.module_from_spec(spec)
            sys.modules[name] = mod
            spec.loader.exec_module(mod)
        _modules[name] = sys.modules[name]
    return _modules[name]


_live = {"key": None, "sim": None}


def _simulation(case):
    """The process's simulation, of this case's configuration."""
    key = tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "steps", "snapshot")))
    if _live["key"] == key:
        return _live["sim"]
    if _live["sim"] is not None:
        _live["sim"].close()
        _live["key"] = _live["sim"] = None
    md = _module("mdbench_gfx950")
    box = dict(nx=case["nx"], ny=case["ny"], nz=case["nz"])
    if case["kind"] == "cp":
        sim = md.CPSim(cluster_m=4, cluster_n=case["n"], half_neigh=case["half"],
                       precision=case["precision"], reneigh_every=20,
                       **box, **(KA if case["ka"] else {}))
    elif case["eam"]:
        sim = md.VLSim(force_field=md.FF_EAM, lattice_a=CU["a"], temp=case["temp"],
                       maxwell_seed=1600, reneigh_every=CU["every"], **box)
    else:
        sim = md.VLSim(half_neigh=case["half"], reneigh_every=LJ["every"],
                       **box, **(MIXED if case["mixed"] else {}))
    _live["key"], _live["sim"] = key, sim
    return sim


class _Span:
    """n values of a device array of the library, for torch.as_tensor (which keeps this object,
    and with it the array's owner)."""

    def __init__(self, pointer, n, typestr, owner):
        self.owner = owner
        address = ctypes.cast(pointer, ctypes.c_void_p).value
        self.__cuda_array_interface__ = {"shape": (int(n),), "typestr": typestr, "version": 2,
                                         "data": (address, False)}


def _tensor(pointer, n, typestr, owner=None):
    return torch.as_tensor(_Span(pointer, n, typestr, owner), device="cuda")


# ------------------------------------------------------------------ inputs
def _fcc(nx, ny, nz):
    """Lattice sites in half cells, in the 8 x 8 x 8 block order of the library's own lattice."""
    z, y, x = np.meshgrid(np.arange(2 * nz), np.arange(2 * ny), np.arange(2 * nx), indexing="ij")
    keep = (x + y + z) % 2 == 0
    x, y, z = x[keep], y[keep], z[keep]
    order = np.lexsort((x, y, z, x // 8, y // 8, z // 8))
    return np.stack([x, y, z], 1)[order].astype(np.float64)


def _box(case):
    if case["kind"] == "vl" and case["eam"]:
        return CU["a"]
    rho = KA["rho"] if case.get("ka") else LJ["rho"]
    return (4.0 / rho) ** (1.0 / 3.0)


def _atoms(case, seed):
    """Positions in the box, velocities and types of a configuration, as host arrays."""
    rng = np.random.default_rng([seed, case["nx"], case["ny"], case["nz"]])
    a = _box(case)
    prd = a * np.array([case["nx"], case["ny"], case["nz"]], np.float64)
    x = _fcc(case["nx"], case["ny"], case["nz"]) * (0.5 * a)
    eam = case["kind"] == "vl" and case["eam"]
    disp = CU["disp"] if eam else LJ["disp"] * (0.75 if case.get("ka") else 1.0)
    x += rng.uniform(-disp, disp, x.shape)
    x = np.where(x < 0.0, x + prd, x)
    x = np.where(x >= prd, x - prd, x)
    v = rng.standard_normal(x.shape)
    v -= v.mean(0)
    unit, mass = (CU["mvv2e"] / CU["kb"], CU["mass"]) if eam else (1.0, 1.0)
    temp = case["temp"] if case["kind"] == "vl" else (KA["temp"] if case["ka"] else LJ["temp"])
    v *= math.sqrt(temp * (3 * len(x) - 3) / (mass * unit * (v * v).sum()))
    if case.get("ka"):
        t = (rng.random(len(x)) < KA["type1_fraction"]).astype(np.int32)
    else:
        ntypes = 2 if case.get("mixed") else 4
        t = (np.zeros(len(x), np.int32) if eam else rng.integers(0, ntypes, len(x), np.int32))
    return x, v, t, prd


def prepare(case, seed):
    if case["kind"] == "sur":
        return _prepare_sur(case, seed)
    _simulation(case)
    x, v, t, _ = _atoms(case, seed)
    if case["kind"] == "cp":
        return {"case": case, "x": x.reshape(-1), "v": v.reshape(-1), "t": t}
    return {"case": case, "x": torch.from_numpy(x.reshape(-1)).cuda(),
            "v": torch.from_numpy(v.reshape(-1)).cuda(), "t": torch.from_numpy(t).cuda()}


# ------------------------------------------------------------------ passes
def run(state):
    kind = state["case"]["kind"]
    return {"vl": _run_vl, "cp": _run_cp, "sur": _run_sur}[kind](state)


def _run_vl(state):
    case = state["case"]
    sim = _simulation(case)
    lib = _module("mdbench_gfx950").lib()
    n = sim.atom.Nlocal
    d = sim.atom.d_atom
    _tensor(d.x, 3 * n, "<f8").copy_(state["x"])
    _tensor(d.vx, 3 * n, "<f8").copy_(state["v"])
    _tensor(d.type, n, "<i4").copy_(state["t"])
    torch.cuda.current_stream().synchronize()  # the library works on a stream of its own
    lib.updateAtomsPbcGFX950(sim.atom_p, sim.param_p, True)
    lib.setupPbcGFX950(sim.atom_p, sim.param_p)
    lib.updatePbcGFX950(sim.atom_p, sim.param_p, True)
    lib.buildNeighborGFX950(sim.atom_p, sim.neighbor_p)
    sim.compute_force()
    sim.run(case["steps"])
    if case["snapshot"]:
        e = sim.eam_atom_energy()
        out = sim.state()
        return {"x": out["x"][:3 * n], "v": out["v"], "f": out["f"], "e": e,
                "numneigh": out["numneigh"]}
    lib.mdgfx950Synchronize()
    d = sim.atom.d_atom
    return {"x": _tensor(d.x, 3 * n, "<f8").clone(), "v": _tensor(d.vx, 3 * n, "<f8").clone(),
            "f": _tensor(d.fx, 3 * n, "<f8").clone()}


def _run_cp(state):
    sim = _simulation(state["case"])
    lib = _module("mdbench_gfx950").lib()
    sim.set_atoms(state["x"], state["v"], state["t"])
    sim.run(CP_STEPS)
    lib.updateSingleAtomsGFX950(ctypes.c_void_p(sim.param_p), ctypes.c_void_p(sim.atom_p))
    # FP32-mixed runs are kept as single-precision frames, as trajectory files are
    kind = np.float64 if state["case"]["precision"] else np.float32
    return {"x": sim.get("atoms_x").astype(kind, copy=False),
            "v": sim.get("atoms_v").astype(kind, copy=False), "t": sim.get("atoms_type")}


# ------------------------------------------------------------------ the surrogate
SUR = dict(rc=4.95, nr=24, mu0=1.9, dmu=0.13, eta=1.0 / (2.0 * 0.16 ** 2), na=4, amu0=2.5,
           admu=0.6, aeta=1.0 / (2.0 * 0.35 ** 2), nd=32, h=64, r_core=2.0, k_core=30.0)


def _theta():
    """The network's weights before training: normal, scaled by the fan-in, no biases."""
    rng = np.random.default_rng(7)
    h, nd = SUR["h"], SUR["nd"]
    return np.concatenate([rng.normal(0, nd ** -0.5, h * nd), np.zeros(h),
                           rng.normal(0, h ** -0.5, h * h), np.zeros(h),
                           rng.normal(0, h ** -0.5, h), np.zeros(1)]).astype(np.float32)


def _frame(rng, cells):
    """One snapshot: displaced copper lattice, its ghost images and the list inside the cutoff."""
    prd = CU["a"] * cells
    x = _fcc(cells, cells, cells) * (0.5 * CU["a"])
    x += rng.uniform(-CU["disp"], CU["disp"], x.shape)
    x -= np.floor(x / prd) * prd
    ext, owner = [x], []
    for sx in (-1, 0, 1):
        for sy in (-1, 0, 1):
            for sz in (-1, 0, 1):
                if (sx, sy, sz) == (0, 0, 0):
                    continue
                img = x + prd * np.array([sx, sy, sz])
                near = ((img > -SUR["rc"]) & (img < prd + SUR["rc"])).all(1)
                ext.append(img[near])
                owner.append(np.nonzero(near)[0])
    ext, owner = np.concatenate(ext), np.concatenate(owner).astype(np.int32)
    idx, mask = _neighbours(torch.from_numpy(ext).to(_device()), len(x), SUR["rc"])
    idx, mask = idx.cpu().numpy(), mask.cpu().numpy()
    return dict(nlocal=len(x), x=ext.reshape(-1), owner=owner,
                numneigh=mask.sum(1).astype(np.int32), neighbors=idx[mask].astype(np.int32))


_norm = {}


def _normalisation():
    """Mean and standard deviation of the descriptors over a sample frame."""
    if not _norm:
        fr = _frame(np.random.default_rng(11), 5)
        x, n = torch.from_numpy(fr["x"].reshape(-1, 3)), fr["nlocal"]
        idx, mask = _padded(fr, n)
        d = _descriptors(x, n, idx, mask)
        _norm["mean"] = d.mean(0).numpy().astype(np.float32)
        _norm["std"] = (d.std(0) + 1e-3).numpy().astype(np.float32)
    return _norm["mean"], _norm["std"]


def _frames(case, seed):
    """Frames with labels: energies around the copper table's values, forces of a few eV/A."""
    rng = np.random.default_rng([seed, case["cells"], case["frames"]])
    frames = []
    for _ in range(case["frames"]):
        fr = _frame(rng, case["cells"])
        fr["e_ref"] = -3.5 + 0.1 * rng.standard_normal(fr["nlocal"])
        fr["f_ref"] = 0.8 * rng.standard_normal(3 * fr["nlocal"])
        frames.append(fr)
    return frames


def _prepare_sur(case, seed):
    sur = _module("eam_surrogate")
    mean, std = _normalisation()
    model = sur.Model(_theta(), mean, std, -3.5, 0.5, SUR["r_core"], SUR["k_core"])
    packed = sur.PackedFrames(_frames(case, seed))
    if case["op"] == "train":
        return {"case": case, "trainer": sur.Trainer(packed, packed, model,
                                                     batch_frames=case["frames"]),
                "packed": packed}
    model.upload()
    return {"case": case, "packed": packed, "ws": sur.Workspace(packed.nlocal, packed.maxn)}


def _run_sur(state):
    sur = _module("eam_surrogate")
    n = state["packed"].nlocal
    lib = sur.lib()
    if state["case"]["op"] == "predict":
        ws = state["ws"]
        sur.predict(state["packed"].sys, 0, n, ws)
        return {"e": _tensor(ws.e.ptr, n, "<f4", ws), "f": _tensor(ws.f.ptr, 3 * n, "<f8", ws)}
    tr = state["trainer"]
    lib.surSetParamsDeviceGFX950(tr.theta.ptr)  # the library holds one model: this trainer's
    tr.step(0, n, 2e-3)
    return {"theta": _tensor(tr.theta.ptr, sur.NPARAM, "<f4", tr),
            "grad": _tensor(tr.grad.ptr, sur.NPARAM, "<f4", tr),
            "f": _tensor(tr.ws.f.ptr, 3 * n, "<f8", tr).float()}


# ------------------------------------------------------------------ what a pass cannot do without
def _pairs_per_atom(case, cut):
    if case["kind"] == "sur" or case.get("eam"):
        return 4.0 / CU["a"] ** 3 * 4.0 / 3.0 * math.pi * cut ** 3
    rho = KA["rho"] if case.get("ka") else LJ["rho"]
    return rho * 4.0 / 3.0 * math.pi * cut ** 3


def work(case):
    if case["kind"] == "sur":
        n = 4.0 * case["cells"] ** 3 * case["frames"]
        pairs = n * _pairs_per_atom(case, SUR["rc"])
        # positions and the list in, energies and forces out; per pair about 130 operations for
        # the descriptors and 300 for the force, per atom the network forward and backward
        bytes_, flops = n * (24 + 4 + 28) + pairs * 4, pairs * 430 + n * 4 * 6337
        if case["op"] == "train":
            bytes_, flops = bytes_ + n * 32 + 4 * 4 * 6337, flops + pairs * 200 + n * 8 * 6337
        return {"bytes": bytes_, "flops": flops}
    n = 4.0 * case["nx"] * case["ny"] * case["nz"]
    steps = CP_STEPS if case["kind"] == "cp" else case["steps"]
    cut = CU["cut"] if case.get("eam") else LJ["cut"]
    pairs = n * _pairs_per_atom(case, cut) * (0.5 if case["half"] else 1.0)
    # in and out once (x, v, type; x, v, f); per step position and velocity read and written
    bytes_ = n * (52 + 72) + steps * n * 96.0
    flops = (steps + 1) * pairs * (55.0 if case.get("eam") else 24.0)
    return {"bytes": bytes_, "flops": flops}


# ------------------------------------------------------------------ the same in 64 bits
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _neighbours(ext, nlocal, cut, chunk=60000):
    """For each of the first nlocal rows of ext: the indices of all other rows within cut (padded)
    and which of them count."""
    lo = ext.min(0).values - 1e-6
    cell = ((ext - lo) / cut).floor().long()
    dims = cell.max(0).values + 3
    cell = cell + 1
    ident = (cell[:, 2] * dims[1] + cell[:, 1]) * dims[0] + cell[:, 0]
    total = int(dims.prod().item()) + 1
    order = torch.argsort(ident, stable=True)
    count = torch.bincount(ident, minlength=total)
    start = torch.cumsum(count, 0) - count
    most = int(count.max())
    shifts = torch.tensor([(dz * int(dims[1]) + dy) * int(dims[0]) + dx for dz in (-1, 0, 1)
                           for dy in (-1, 0, 1) for dx in (-1, 0, 1)], device=ext.device)
    slots = torch.arange(most, device=ext.device)
    found, widths = [], []
    for a in range(0, nlocal, chunk):
        b = min(nlocal, a + chunk)
        home = ident[a:b, None] + shifts[None]
        at = start[home][..., None] + slots
        ok = slots < count[home][..., None]
        at, ok = at.reshape(b - a, -1), ok.reshape(b - a, -1)
        j = order[at.clamp_(max=len(order) - 1)]
        d = ext[a:b, None, :] - ext[j]
        ok &= (d * d).sum(-1) <= cut * cut
        ok &= j != torch.arange(a, b, device=ext.device)[:, None]
        rank = torch.cumsum(ok, 1) - 1
        width = int(ok.sum(1).max())
        idx = torch.zeros(b - a, width, dtype=torch.long, device=ext.device)
        row, col = ok.nonzero(as_tuple=True)
        idx[row, rank[row, col]] = j[row, col]
        found.append((idx, ok.sum(1)))
        widths.append(width)
    width = max(widths)
    idx = torch.cat([torch.nn.functional.pad(i, (0, width - i.shape[1])) for i, _ in found])
    number = torch.cat([n for _, n in found])
    return idx, torch.arange(width, device=ext.device) < number[:, None]


def _images(x, prd, cut):
    """Periodic images of the atoms within cut of the box: which atom, and its shift."""
    owner, shift = [], []
    for sx in (-1, 0, 1):
        for sy in (-1, 0, 1):
            for sz in (-1, 0, 1):
                if (sx, sy, sz) == (0, 0, 0):
                    continue
                s = torch.tensor([sx, sy, sz], dtype=x.dtype, device=x.device) * prd
                near = ((x + s >= -cut) & (x + s <= prd + cut)).all(1).nonzero()[:, 0]
                owner.append(near)
                shift.append(s.expand(len(near), 3))
    return torch.cat(owner), torch.cat(shift)


def _list(x, prd, cut):
    """Padded neighbour list over atoms: j, its image's shift, and which entries count."""
    owner, shift = _images(x, prd, cut)
    idx, mask = _neighbours(torch.cat([x, x[owner] + shift]), len(x), cut)
    all_owner = torch.cat([torch.arange(len(x), device=x.device), owner])
    all_shift = torch.cat([torch.zeros_like(x), shift])
    return all_owner[idx], all_shift[idx], mask


def _lj_tables(case):
    if case.get("ka"):
        eps, sig = np.array(KA["pair_epsilon"]), np.array(KA["pair_sigma"])
        return eps, sig ** 6, np.array(KA["pair_cutoff"]) ** 2, 2
    if case.get("mixed"):
        e, s = np.array(MIXED["epsilon_per_type"]), np.array(MIXED["sigma_per_type"])
        return (np.sqrt(np.outer(e, e)).reshape(-1), np.outer(s ** 3, s ** 3).reshape(-1),
                np.full(4, LJ["cut"] ** 2), 2)
    return np.ones(1), np.ones(1), np.array([LJ["cut"] ** 2]), 0


def _lj_force(case, x, t, nbr, chunk=100000):
    j, shift, mask = nbr
    eps, sig6, cut2, nt = _lj_tables(case)
    eps, sig6, cut2 = (torch.from_numpy(a).to(x.device) for a in (eps, sig6, cut2))
    f = torch.empty_like(x)
    for a in range(0, len(x), chunk):
        s = slice(a, a + chunk)
        d = x[s, None, :] - (x[j[s]] + shift[s])
        r2 = torch.where(mask[s], (d * d).sum(-1), 1e30)
        k = t[s, None] * nt + t[j[s]] if nt else torch.zeros_like(j[s])
        ir2 = torch.where(r2 < cut2[k], 1.0 / r2, 0.0)
        ir6 = ir2 ** 3 * sig6[k]
        f[s] = (d * (48.0 * ir6 * (ir6 - 0.5) * ir2 * eps[k])[..., None]).sum(1)
    return f


_eam = {}


def _eam_tables(device):
    """Cubic splines of the synthetic copper tables: F(rho), rho(r) and r phi(r), knots 1 .. 1999,
    each as value coefficients c3, c2, c1, c0 of p in [0, 1] and the spacing."""
    if not _eam:
        n, dr, drho = 2000, 0.0025, 0.02
        r = np.arange(n) * dr
        u = ((r - 4.95) / 0.5) ** 4
        taper = np.where(r >= 4.95, 0.0, u / (1.0 + u))
        z = 0.1776 * np.exp(-1.5 * (r - 2.556)) * taper
        tabs = {"F": (-np.sqrt(np.arange(n) * drho), drho),
                "rho": (np.exp(-3.0 * (r / 2.556 - 1.0)) * taper, dr),
                "z2": (27.2 * 0.529 * z * z, dr)}
        for name, (f, h) in tabs.items():
            f = f[:n - 1]  # the reader keeps one knot less than the file
            g = np.zeros_like(f)
            g[2:-2] = ((f[:-4] - f[4:]) + 8.0 * (f[3:-1] - f[1:-3])) / 12.0
            g[0], g[-1] = f[1] - f[0], f[-1] - f[-2]
            g[1], g[-2] = 0.5 * (f[2] - f[0]), 0.5 * (f[-1] - f[-3])
            c2, c3 = np.zeros_like(f), np.zeros_like(f)
            c2[:-1] = 3.0 * (f[1:] - f[:-1]) - 2.0 * g[:-1] - g[1:]
            c3[:-1] = g[:-1] + g[1:] - 2.0 * (f[1:] - f[:-1])
            _eam[name] = np.stack([c3, c2, g, f]), h
    return {k: (torch.from_numpy(c).to(device), h) for k, (c, h) in _eam.items()}


def _spline(tab, at, first):
    """Value and derivative of a table at `at`; `first`: the lowest knot used."""
    c, h = tab
    n = c.shape[1]
    p = at / h + 1.0
    m = p.floor().clamp_(max=n - 1)
    m = m.clamp(min=first)
    p = (p - m).clamp(max=1.0)
    c = c[:, (m.long() - 1).clamp(min=0)]
    return (((c[0] * p + c[1]) * p + c[2]) * p + c[3],
            ((3.0 * c[0] * p + 2.0 * c[1]) * p + c[2]) / h)


def _eam_force(case, x, t, nbr, energy=False, chunk=100000):
    j, shift, mask = nbr
    tab = _eam_tables(x.device)
    rho = torch.empty_like(x[:, 0])
    for a in range(0, len(x), chunk):
        s = slice(a, a + chunk)
        d = x[s, None, :] - (x[j[s]] + shift[s])
        r2 = (d * d).sum(-1)
        ok = mask[s] & (r2 < CU["cut"] ** 2)
        rho[s] = torch.where(ok, _spline(tab["rho"], torch.where(ok, r2, 4.0).sqrt(), 0)[0],
                             0.0).sum(1)
    emb, fp = _spline(tab["F"], rho, 1)
    f, e = torch.empty_like(x), emb.clone()
    for a in range(0, len(x), chunk):
        s = slice(a, a + chunk)
        d = x[s, None, :] - (x[j[s]] + shift[s])
        r2 = (d * d).sum(-1)
        ok = mask[s] & (r2 < CU["cut"] ** 2)
        r = torch.where(ok, r2, 4.0).sqrt()
        z2, z2p = _spline(tab["z2"], r, 0)
        phi = z2 / r
        force = -((fp[s, None] + fp[j[s]]) * _spline(tab["rho"], r, 0)[1] + z2p / r - phi / r) / r
        f[s] = (d * torch.where(ok, force, 0.0)[..., None]).sum(1)
        e[s] += 0.5 * torch.where(ok, phi, 0.0).sum(1)
    return (f, e) if energy else f


def _exact_vl(case, seed):
    x, v, t, prd = _atoms(case, seed)
    dev = _device()
    x, v, t, prd = (torch.from_numpy(a).to(dev) for a in (x, v, t.astype(np.int64), prd))
    par = CU if case["eam"] else LJ
    force = _eam_force if case["eam"] else _lj_force
    dt = par["dt"]
    kick = 0.5 * dt / CU["mass"] / CU["mvv2e"] if case["eam"] else 0.5 * dt
    nbr = _list(x, prd, par["cut"] + par["skin"])
    f = force(case, x, t, nbr)
    for step in range(1, case["steps"] + 1):
        v = v + kick * f
        x = x + dt * v
        if step % par["every"] == 0:
            x = torch.where(x < 0.0, x + prd, torch.where(x >= prd, x - prd, x))
            nbr = _list(x, prd, par["cut"] + par["skin"])
        f = force(case, x, t, nbr)
        v = v + kick * f
    x, v, f = (a.reshape(-1).cpu().numpy() for a in (x, v, f))
    if not case["snapshot"]:
        return {"x": x, "v": v, "f": f}
    e = force(case, torch.from_numpy(x.reshape(-1, 3)).to(dev), t, nbr, energy=True)[1]
    return {"x": x, "v": v, "f": f, "e": e.cpu().numpy(), "numneigh": None}


def _cluster_order(x, prd, n):
    """The atoms sorted into columns of the box and by z inside a column, the i-cluster of each
    (four atoms, columns padded to whole clusters, to an even number for j-clusters of eight),
    and the columns' sides."""
    sides = [float(p) for p in prd]
    # the ratio of a side to a column is a whole number up to rounding: the same cube root
    side = float(np.cbrt(max(4, n) / (len(x) / (sides[0] * sides[1] * sides[2]))))
    nb = [max(1, math.ceil(sides[d] / side)) for d in (0, 1)]
    cx, cy = ((x[:, d] * (1.0 / (float(prd[d]) / nb[d]))).long() for d in (0, 1))
    column = cy * nb[0] + cx
    order = torch.argsort(x[:, 2], stable=True)
    order = order[torch.argsort(column[order], stable=True)]
    column = column[order]
    count = torch.bincount(column, minlength=nb[0] * nb[1])
    clusters = (count + 3) // 4
    if n == 8:
        clusters = (clusters + 1) // 2 * 2
    first = torch.cumsum(count, 0) - count
    rank = torch.arange(len(x), device=x.device) - first[column]
    ci = (torch.cumsum(clusters, 0) - clusters)[column] + rank // 4
    return order, ci, int(clusters.sum()), [float(prd[d]) / nb[d] for d in (0, 1)]


def _boxes(x, cluster, number):
    lo = torch.full((number, 3), 1e30, dtype=x.dtype, device=x.device)
    hi = torch.full((number, 3), -1e30, dtype=x.dtype, device=x.device)
    at = cluster[:, None].expand(-1, 3)
    return lo.scatter_reduce(0, at, x, "amin"), hi.scatter_reduce(0, at, x, "amax")


def _exact_cp(case, seed):
    """Cluster-pair lists hold whole cluster pairs, so an atom pair acts when its clusters are
    listed: some atom pair within the list cutoff, or boxes closer than the sure distance."""
    x, v, t, prd = _atoms(case, seed)
    dev = _device()
    x, v, t, prd = (torch.from_numpy(a).to(dev) for a in (x, v, t.astype(np.int64), prd))
    n, cut = case["n"], LJ["cut"] + LJ["skin"]
    order, ci, nci, side = _cluster_order(x, prd, n)
    x, v, t = x[order], v[order], t[order]
    per = n // 4
    cj, ncj = ci // per, nci // per
    ilo, ihi = _boxes(x, ci, nci)
    jlo, jhi = _boxes(x, cj, ncj)
    sure = max(0.0, cut - 0.5 * math.hypot(*side))
    idx, shift, mask = _list(x, prd, cut + 1.0)
    row, col = mask.nonzero(as_tuple=True)
    i, j, s = row, idx[row, col], shift[row, col]
    del idx, shift, mask
    d = x[i] - x[j] - s
    near = (d * d).sum(1) < cut * cut
    sign = (s / prd).round().long() + 1
    image = sign[:, 0] + 3 * sign[:, 1] + 9 * sign[:, 2]
    a, b = ci[i], cj[j]
    if case["half"]:  # a pair of local clusters is listed by the lower j-cluster's side
        swap = (image == 13) & (a // per > b)
        a, b = torch.where(swap, ci[j], a), torch.where(swap, cj[i], b)
    gap = torch.maximum(ilo[a] - jhi[b] - s, jlo[b] + s - ihi[a]).clamp(min=0.0)
    near |= (gap * gap).sum(1) < sure * sure
    del d, gap
    key = (a * ncj + b) * 27 + image
    which, back = torch.unique(key, return_inverse=True)
    listed_ = torch.zeros(len(which), dtype=torch.bool, device=dev)
    listed_[back[near]] = True
    keep = listed_[back]
    i, j, s = i[keep], j[keep], s[keep]
    del key, which, back, near, image, a, b
    eps, sig6, cut2, nt = (torch.from_numpy(a).to(dev) if isinstance(a, np.ndarray) else a
                           for a in _lj_tables(case))
    k = t[i] * nt + t[j] if nt else torch.zeros_like(i)
    # one row of slots per atom, so that the sums have an order
    number = torch.bincount(i, minlength=len(x))
    slot = torch.arange(len(i), device=dev) - (torch.cumsum(number, 0) - number)[i]
    width = int(number.max())
    pj = torch.zeros(len(x), width, dtype=torch.long, device=dev)
    ps = torch.zeros(len(x), width, 3, dtype=x.dtype, device=dev)
    pk = torch.zeros(len(x), width, dtype=torch.long, device=dev)
    pj[i, slot], ps[i, slot], pk[i, slot] = j, s, k
    ok = torch.arange(width, device=dev) < number[:, None]
    del i, j, s, k, slot

    def force(x, chunk=100000):
        f = torch.empty_like(x)
        for c in range(0, len(x), chunk):
            q = slice(c, c + chunk)
            d = x[q, None, :] - (x[pj[q]] + ps[q])
            r2 = torch.where(ok[q], (d * d).sum(-1), 1e30)
            ir2 = torch.where(r2 < cut2[pk[q]], 1.0 / r2, 0.0)
            ir6 = ir2 ** 3 * sig6[pk[q]]
            f[q] = (d * (48.0 * ir6 * (ir6 - 0.5) * ir2 * eps[pk[q]])[..., None]).sum(1)
        return f

    f = force(x)
    for _ in range(CP_STEPS):
        v = v + 0.5 * LJ["dt"] * f
        x = x + LJ["dt"] * v
        f = force(x)
        v = v + 0.5 * LJ["dt"] * f
    return {"x": x.reshape(-1).cpu().numpy(), "v": v.reshape(-1).cpu().numpy(), "t": None}


def _padded(fr, n, width=None):
    """A frame's list as padded rows over local and ghost indices."""
    number = torch.from_numpy(fr["numneigh"].astype(np.int64))
    width = width or int(number.max())
    mask = torch.arange(width) < number[:, None]
    idx = torch.zeros(n, width, dtype=torch.long)
    idx[mask] = torch.from_numpy(fr["neighbors"].astype(np.int64))
    return idx, mask


def _descriptors(ext, n, idx, mask):
    """24 Gaussian radial and 2 x 4 angular (l = 1 and l = 2) descriptors per atom."""
    c = SUR
    d = ext[idx] - ext[:n, None, :]
    r2 = (d * d).sum(-1)
    ok = mask & (r2 < c["rc"] ** 2)
    r = torch.where(ok, r2, 1.0).sqrt()
    u = d / r[..., None]
    fc = torch.where(ok, (1.0 - (r / c["rc"]) ** 2) ** 3, 0.0)
    mu = c["mu0"] + c["dmu"] * torch.arange(c["nr"], dtype=ext.dtype, device=ext.device)
    amu = c["amu0"] + c["admu"] * torch.arange(c["na"], dtype=ext.dtype, device=ext.device)
    out = [(torch.exp(-c["eta"] * (r[..., None] - mu) ** 2) * fc[..., None]).sum(1)]
    w = torch.exp(-c["aeta"] * (r[..., None] - amu) ** 2) * fc[..., None]
    m1 = torch.matmul(w.transpose(1, 2), u)
    uu = (u[..., :, None] * u[..., None, :]).reshape(*u.shape[:2], 9)
    m2 = torch.matmul(w.transpose(1, 2), uu)
    trace = m2[..., 0] + m2[..., 4] + m2[..., 8]
    out.append((m1 * m1).sum(-1))
    out.append(1.5 * ((m2 * m2).sum(-1) - trace ** 2 / 3.0))
    return torch.cat(out, 1)


def _network(theta, dn, e0=-3.5, s_e=0.5):
    h, nd = SUR["h"], SUR["nd"]
    w1, b1, w2, b2, w3, b3 = torch.split(theta, [h * nd, h, h * h, h, h, 1])
    a = torch.tanh(dn @ w1.reshape(h, nd).T + b1)
    a = torch.tanh(a @ w2.reshape(h, h).T + b2)
    return s_e * (a @ w3 + b3) + e0


def _exact_sur(case, seed):
    """Energies, forces and the loss gradient by automatic differentiation in 64 bits."""
    dev = _device()
    frames = _frames(case, seed)
    mean, std = (torch.from_numpy(a.astype(np.float64)).to(dev) for a in _normalisation())
    train = case["op"] == "train"
    theta = torch.from_numpy(_theta().astype(np.float64)).to(dev).requires_grad_(train)
    total = sum(fr["nlocal"] for fr in frames)
    es, fs, grad = [], [], 0.0
    for fr in frames:
        n = fr["nlocal"]
        ext = torch.from_numpy(fr["x"].reshape(-1, 3)).to(dev)
        idx, mask = (a.to(dev) for a in _padded(fr, n))
        owner = torch.from_numpy(fr["owner"].astype(np.int64)).to(dev)
        x = ext[:n].clone().requires_grad_(True)
        full = torch.cat([x, x[owner] + (ext[n:] - ext[owner])])
        e = _network(theta, (_descriptors(full, n, idx, mask) - mean) / std)
        core = torch.zeros_like(e)
        if not train:
            d = full[idx] - full[:n, None, :]
            r = torch.where(mask, (d * d).sum(-1), 100.0).sqrt()
            core = 0.5 * SUR["k_core"] * ((SUR["r_core"] - r).clamp(min=0.0) ** 3).sum(1)
        f = -torch.autograd.grad((e + core).sum(), x, create_graph=train)[0]
        if train:
            de = e - torch.from_numpy(fr["e_ref"]).to(dev)
            df = f - torch.from_numpy(fr["f_ref"].reshape(-1, 3)).to(dev)
            loss = (de * de).sum() / total + (df * df).sum() / (3 * total)
            grad = grad + torch.autograd.grad(loss, theta)[0]
        es.append(e.detach())
        fs.append(f.detach().reshape(-1))
    f = torch.cat(fs).cpu().numpy()
    if not train:
        return {"e": torch.cat(es).cpu().numpy(), "f": f}
    g = grad.cpu().numpy()
    # Adam's first step: moments g and g^2 after the bias correction
    theta = theta.detach().cpu().numpy() - 2e-3 * g / (np.abs(g) + 1e-8)
    return {"theta": theta, "grad": g, "f": f}


def exact(case, seed):
    if case["kind"] == "sur":
        return _exact_sur(case, seed)
    return _exact_vl(case, seed) if case["kind"] == "vl" else _exact_cp(case, seed)
