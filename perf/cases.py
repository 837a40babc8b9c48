"""The work that users of this framework have it do, as cases that can be timed and compared.

Each case is one pass through the public surface: a piece of a simulation (``Simulation.run``
and the recording of the frame it reached), a batch of replicas, a training step of the learned
coarse-grained energy, or the kernel drivers of the C interface that a host program calls in
place of its own. The sizes span the range that the tests, the examples and ``bench.py`` use:
from a few thousand particles, where launches and latency count, to about a million.

A trajectory is chaotic: two correct implementations part by the rounding of their force sums
times exp(lambda t). The runs are therefore short (at most a few hundred steps with the steps
taken in ``prepare``), and positions are returned unwrapped, so that a particle that sits on the
face of the box does not jump by its edge.
"""

import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "hoomd-blue_amd"))

import hoomd_amd as hoomd  # noqa: E402
from hoomd_amd import _lib  # noqa: E402
from hoomd_amd.batch import ReplicaBatch, fcc_fill  # noqa: E402
from hoomd_amd.md import mlcg  # noqa: E402

WCA = 2.0 ** (1.0 / 6.0)


def listed():
    return [
        # The reference's how-to benchmark at its own size: a WCA fluid of a few thousand
        # particles. A step is a handful of launches: latency is everything.
        dict(name="wca-2048-bussi", family="run", fluid="wca", N=2048, rho=1.0, kT=1.2, dt=0.001,
             buffer=0.2, method="bussi", steps=100),
        # A small constant-energy LJ run, the size a CPU run is still compared with.
        dict(name="lj-16384-nve", family="run", fluid="lj", N=16384, rho=0.8442, kT=1.2, dt=0.005,
             buffer=0.4, method="nve", steps=50),
        # The how-to benchmark replicated: the ordinary size of a single-GPU study.
        dict(name="wca-131072-bussi", family="run", fluid="wca", N=131072, rho=1.0, kT=1.2,
             dt=0.001, buffer=0.2, method="bussi", steps=100),
        # The LJ liquid at scale (bench.py's default workload).
        dict(name="lj-1048576-bussi", family="run", fluid="lj", N=1048576, rho=0.8442, kT=1.2,
             dt=0.005, buffer=0.4, method="bussi", steps=100),
        # Two species with their own cutoffs, XPLOR smoothing, a box with three different edges,
        # a ragged particle count, and the pressure tensor logged at the end of each piece.
        dict(name="mixture-50021-xplor", family="run", fluid="mixture", N=50021, rho=0.85, kT=1.0,
             dt=0.004, buffer=0.3, method="bussi", steps=100),
        # Bead-spring melt, FENE bonds, exclusions, Langevin (bench.py --kg).
        dict(name="melt-1000000-langevin", family="run", fluid="melt", N=1000000, rho=0.85,
             kT=1.0, dt=0.01, buffer=0.4, method="langevin", steps=50),
        # Production run of a learned coarse-grained model (bench.py --mlcg / --cg-step).
        dict(name="learned-cg-200000", family="run", fluid="cg", N=200000, rho=0.17, kT=1.0,
             dt=0.02, buffer=0.4, method="langevin", steps=50),
        # Force matching of that model: one Adam step on a few frames, as its training loop runs.
        dict(name="train-200000x2", family="train", N=200000, rho=0.17, frames=2),
        # Loss and gradient of one frame of a small ragged system (an outer optimiser's call).
        dict(name="lossgrad-7210", family="lossgrad", N=7210, rho=0.17, frames=1),
        # A sweep of uneven independent replicas as one batch (bench.py --replicas).
        dict(name="replicas-256", family="batch", replicas=256, nmin=500, nmax=20000, steps=100),
        # The pair-force driver in the reference's own array layout, with the virial, as a host
        # program that owns its neighbour list calls it.
        dict(name="pair-driver-100003", family="driver", N=100003, rho=0.8442, tpp=8),
        # Cell list, neighbour list and pair force through the C drivers, one after another.
        dict(name="list-drivers-262144", family="lists", N=262144, rho=0.8442),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above, sizes spread over their logarithm."""
    family = rng.choice(["run"] * 6 + ["batch", "train", "lossgrad", "driver", "lists"])
    if family == "run":
        fluid = rng.choice(["wca", "lj", "lj", "mixture", "melt", "cg"])
        top = {"wca": 700000, "lj": 700000, "mixture": 200000, "melt": 500000, "cg": 150000}
        N = _log_uniform(rng, 1500, top[fluid])
        c = dict(family="run", fluid=fluid, N=N)
        if fluid == "wca":
            c.update(rho=rng.uniform(0.8, 1.0), kT=1.2, dt=0.001, buffer=rng.choice([0.2, 0.3]),
                     method=rng.choice(["bussi", "nve"]))
        elif fluid == "lj":
            c.update(rho=rng.uniform(0.7, 0.9), kT=rng.uniform(0.8, 1.5), dt=0.005,
                     buffer=rng.choice([0.3, 0.4]),
                     method=rng.choice(["bussi", "nve", "langevin"]))
        elif fluid == "mixture":
            c.update(rho=rng.uniform(0.75, 0.9), kT=1.0, dt=0.004, buffer=0.3,
                     method=rng.choice(["bussi", "langevin"]))
        elif fluid == "melt":
            c.update(N=max(2000, N // 50 * 50), rho=0.85, kT=1.0, dt=0.01,
                     buffer=rng.choice([0.3, 0.4]), method="langevin")
        else:
            c.update(N=max(3000, N // 10 * 10), rho=0.17, kT=1.0, dt=0.02, buffer=0.4,
                     method="langevin")
        c["steps"] = 50 if fluid in ("melt", "cg") or c["method"] == "nve" else 100
        return c
    if family == "batch":
        return dict(family="batch", replicas=_log_uniform(rng, 8, 200), nmin=500,
                    nmax=_log_uniform(rng, 2000, 20000), steps=rng.choice([50, 100]))
    if family == "train":
        return dict(family="train", N=_log_uniform(rng, 5000, 150000), rho=0.17,
                    frames=rng.choice([2, 3]))
    if family == "lossgrad":
        return dict(family="lossgrad", N=_log_uniform(rng, 3000, 30000), rho=0.17, frames=1)
    if family == "driver":
        return dict(family="driver", N=_log_uniform(rng, 3000, 250000),
                    rho=rng.uniform(0.7, 0.9), tpp=rng.choice([4, 8, 16]))
    return dict(family="lists", N=_log_uniform(rng, 3000, 250000), rho=rng.uniform(0.7, 0.9))


# ------------------------------------------------------------------------------------- inputs
def _edges(case):
    """Box edges: cubic, except the mixture's (ratios 1 : 0.9 : 1.2)."""
    V = case["N"] / case["rho"]
    r = (1.0, 0.9, 1.2) if case.get("fluid") == "mixture" else (1.0, 1.0, 1.0)
    a = (V / (r[0] * r[1] * r[2])) ** (1.0 / 3.0)
    return np.array([a * x for x in r])


def _wrap(x, L):
    x = x - L * np.floor(x / L + 0.5)
    return np.where(x >= L / 2, -L / 2, x)


def _fluid_positions(N, L, rng, jitter):
    """N sites of an FCC lattice stretched into the box, chosen at random, each moved a little."""
    unit = fcc_fill(N, 1.0, rng)
    return _wrap(unit * L + rng.uniform(-jitter, jitter, (N, 3)), L)


def _velocities(N, kT, mass, rng):
    v = rng.normal(0.0, math.sqrt(kT / mass), (N, 3))
    return v - v.mean(axis=0)


def _chain_positions(N, L, rng):
    """Chains laid along a snake through a cubic lattice that fills the box: consecutive beads
    are neighbours on the lattice, so no bond is stretched."""
    n = int(math.ceil(N ** (1.0 / 3.0) - 1e-9))
    s = np.arange(N)
    row, x = s // n, s % n
    z, y = row // n, row % n
    x = np.where(row % 2 == 1, n - 1 - x, x)
    y = np.where(z % 2 == 1, n - 1 - y, y)
    a = L / n
    p = (np.stack([x, y, z], 1) + 0.5) * a - L / 2
    return _wrap(p + rng.uniform(-0.02, 0.02, p.shape), L)


def _walk_positions(N, per, step, L, rng):
    """Chains of `per` sites as random walks of the given step."""
    m = N // per
    d = rng.normal(size=(m, per, 3))
    d *= step / np.linalg.norm(d, axis=2, keepdims=True)
    start = rng.uniform(-0.5, 0.5, (m, 1, 3)) * L
    return _wrap((start + np.cumsum(d, axis=1)).reshape(-1, 3), L)


def _chain_bonds(N, per):
    idx = np.arange(N).reshape(-1, per)
    return np.stack([idx[:, :-1].ravel(), idx[:, 1:].ravel()], 1).astype(np.uint32)


def _start(case, seed):
    """Positions, velocities, types and bonds that a run case starts from."""
    rng = np.random.default_rng(seed)
    N, L = case["N"], _edges(case)
    fluid = case["fluid"]
    tid, bonds, mass = np.zeros(N, np.uint32), None, 1.0
    if fluid == "melt":
        pos, bonds = _chain_positions(N, L, rng), _chain_bonds(N, 50)
    elif fluid == "cg":
        pos, bonds, mass = _walk_positions(N, 10, 1.7, L, rng), _chain_bonds(N, 10), 5.0
    else:
        pos = _fluid_positions(N, L, rng, 0.03 if fluid == "wca" else 0.05)
        if fluid == "mixture":
            tid = (rng.uniform(size=N) < 0.3).astype(np.uint32)
    return pos, _velocities(N, case["kT"], mass, rng), tid, bonds, mass


class _DeviceView:
    """A device buffer of the framework seen by torch without a copy."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, typestr="<f4",
                                             version=3)


def _mixture_pairs():
    eps = {("A", "A"): 1.0, ("A", "B"): 1.2, ("B", "B"): 0.8}
    sig = {("A", "A"): 1.0, ("A", "B"): 0.95, ("B", "B"): 0.9}
    return eps, sig


def _simulation(case, seed):
    pos, vel, tid, bonds, mass = _start(case, seed)
    N, L = case["N"], _edges(case)
    snap = hoomd.Snapshot()
    snap.configuration.box = [L[0], L[1], L[2], 0, 0, 0]
    snap.particles.N = N
    snap.particles.types = ["A", "B"] if case["fluid"] == "mixture" else ["A"]
    snap.particles.position[:] = pos
    snap.particles.velocity[:] = vel
    snap.particles.typeid[:] = tid
    snap.particles.mass[:] = mass
    if bonds is not None:
        snap.bonds.N = len(bonds)
        snap.bonds.types = ["b"]
        snap.bonds.group[:] = bonds
    sim = hoomd.Simulation(device=hoomd.device.GPU(), seed=seed & 0xffff)
    sim.create_state_from_snapshot(snap)
    excl = ("bond",) if bonds is not None else ()
    nl = hoomd.md.nlist.Cell(buffer=case["buffer"], exclusions=excl)
    fluid = case["fluid"]
    forces = []
    if fluid == "cg":
        net = mlcg.SiteEnergyMLP(nlist=nl, seed=seed & 0xffff,
                                 params=mlcg.init_params(seed & 0xffff) * 0.05)
        r = (np.arange(80) + 0.5) * 0.05
        prior, rc = mlcg.rdf_prior_table(r, np.clip((r - 0.3) / 1.5, 0.0, 1.0))
        net.pair_table = mlcg.regrid_table(prior, rc, net.r_cut, width=600)
        bond = hoomd.md.bond.Harmonic()
        bond.params["b"] = dict(k=2.3, r0=1.74)
        forces = [net, bond]
    else:
        rc, mode = {"wca": (WCA, "none"), "lj": (2.5, "none"), "mixture": (2.5, "xplor"),
                    "melt": (WCA, "shift")}[fluid]
        lj = hoomd.md.pair.LJ(nlist=nl, default_r_cut=rc, mode=mode)
        if fluid == "mixture":
            eps, sig = _mixture_pairs()
            for p in eps:
                lj.params[p] = dict(epsilon=eps[p], sigma=sig[p])
                lj.r_cut[p] = 2.5 * sig[p]
                lj.r_on[p] = 2.0 * sig[p]
        else:
            lj.params[("A", "A")] = dict(epsilon=1.0, sigma=1.0)
        forces = [lj]
        if fluid == "melt":
            fene = hoomd.md.bond.FENEWCA()
            fene.params["b"] = dict(k=30.0, r0=1.5, epsilon=1.0, sigma=1.0, delta=0.0)
            forces.append(fene)
    if case["method"] == "langevin":
        method = hoomd.md.methods.Langevin(filter=hoomd.filter.All(), kT=case["kT"])
        for t in snap.particles.types:
            method.gamma[t] = 5.0 if fluid == "cg" else 1.0
    else:
        thermostat = None
        if case["method"] == "bussi":
            thermostat = hoomd.md.methods.thermostats.Bussi(kT=case["kT"])
        method = hoomd.md.methods.ConstantVolume(hoomd.filter.All(), thermostat=thermostat)
    sim.operations.integrator = hoomd.md.Integrator(dt=case["dt"], forces=forces,
                                                    methods=[method])
    thermo = None
    if fluid == "mixture":
        thermo = hoomd.md.compute.ThermodynamicQuantities(hoomd.filter.All())
        sim.operations.add(thermo)
    return sim, pos, thermo


def _frames(case, seed):
    """Mapped frames as FP32 host arrays: sites off a lattice at the density of the mapped melt,
    and forces of its size."""
    rng = np.random.default_rng(seed)
    N = case["N"]
    L = (N / case["rho"]) ** (1.0 / 3.0)
    n = int(math.ceil(N ** (1.0 / 3.0) - 1e-9))
    out = []
    for _ in range(case["frames"]):
        s = np.sort(rng.choice(n ** 3, N, replace=False))
        p = np.stack([s % n, s // n % n, s // (n * n)], 1) + 0.5
        p = _wrap(p * (L / n) - L / 2 + rng.normal(0.0, 0.45, (N, 3)), np.array([L] * 3))
        p = p.astype(np.float32)
        p[p >= np.float32(L / 2)] = np.float32(-L / 2 * (1 - 1e-6))
        p[p < -np.float32(L / 2)] = np.float32(-L / 2 * (1 - 1e-6))
        out.append((p, rng.normal(0.0, 5.0, (N, 3)).astype(np.float32)))
    return out, L


def _normalization(rho):
    """Mean densities of a structureless fluid and the inverse of their spread."""
    r = (np.arange(3000) + 0.5) * 1e-3
    fc = 0.5 * (np.cos(np.pi * r / 3.0) + 1.0)
    g = np.array([np.sum(rho * 4 * np.pi * r * r * np.exp(-(r - 0.2 * k) ** 2 / 0.08) * fc) * 1e-3
                  for k in range(16)])
    return g, 1.0 / (0.05 + np.sqrt(g))


def _training(case, seed):
    frames, L = _frames(case, seed)
    snap = hoomd.Snapshot()
    snap.configuration.box = [L, L, L, 0, 0, 0]
    snap.particles.N = case["N"]
    snap.particles.types = ["S"]
    snap.particles.position[:] = frames[0][0]
    sim = hoomd.Simulation(device=hoomd.device.GPU(), seed=seed & 0xffff)
    sim.create_state_from_snapshot(snap)
    nl = hoomd.md.nlist.Cell(buffer=0.4)
    net = mlcg.SiteEnergyMLP(nlist=nl, params=mlcg.init_params(seed & 0xffff))
    net.normalization = _normalization(case["rho"])
    sim.operations.integrator = hoomd.md.Integrator(
        dt=0.01, forces=[net], methods=[hoomd.md.methods.ConstantVolume(hoomd.filter.All())])
    sim.operations.tuners.clear()
    sim.run(0)
    fs = mlcg.FrameSet(case["frames"], case["N"])
    for k, (p, f) in enumerate(frames):
        fs.set(k, p, f)
    return dict(sim=sim, net=net, frames=fs, n=case["frames"])


def _driver_positions(case, seed):
    rng = np.random.default_rng(seed)
    L = (case["N"] / case["rho"]) ** (1.0 / 3.0)
    return _fluid_positions(case["N"], np.array([L] * 3), rng, 0.12), L


def _list_args(pos, L, r_cut, r_buff):
    """Buffers and argument blocks of the cell-list and neighbour-list drivers."""
    N = len(pos)
    lib, box = _lib.lib(), _lib.box(L)
    dim = (C.c_uint * 3)()
    _lib.check(lib.hm_cell_dims(C.byref(box), r_cut + r_buff, dim))
    ncell = dim[0] * dim[1] * dim[2]
    n_adj = lib.hm_cell_n_adj(dim)
    cmax, nmax = 64, 160

    def empty(n, dtype):
        return torch.zeros(n, dtype=dtype, device="cuda")

    b = dict(size=empty(ncell, torch.int32), entries=empty(ncell * cmax * 4, torch.float64),
             adj=empty(ncell * n_adj, torch.int32), cond=empty(4, torch.int32),
             nlist=empty(N * nmax, torch.int32), n_neigh=empty(N, torch.int32))
    b["pos"] = empty((N, 4), torch.float64)
    b["pos"][:, :3] = torch.from_numpy(pos)
    torch.cuda.synchronize()
    _lib.check(lib.hm_cell_adj(dim, b["adj"].data_ptr(), None))
    ca, na = _lib.HmCellArgs(), _lib.HmNlistArgs()
    for a in (ca, na):
        a.N, a.pos, a.box, a.cmax = N, b["pos"].data_ptr(), box, cmax
        a.cell_size, a.entries = b["size"].data_ptr(), b["entries"].data_ptr()
        for k in range(3):
            a.dim[k] = dim[k]
    ca.conditions = b["cond"].data_ptr()
    na.cell_adj, na.n_adj, na.ntypes = b["adj"].data_ptr(), n_adj, 1
    na.r_cut[0], na.r_buff, na.nmax = r_cut, r_buff, nmax
    na.nlist, na.n_neigh = b["nlist"].data_ptr(), b["n_neigh"].data_ptr()
    na.conditions = b["cond"].data_ptr() + 12
    return b, ca, na, nmax


def _lj_driver(case, seed):
    """The reference's arrays around its pair driver: Scalar4 positions with the type's bits,
    a head list, the neighbour rows, squared cutoffs."""
    pos, L = _driver_positions(case, seed)
    b, ca, na, nmax = _list_args(pos, L, 2.5, 0.4)
    lib = _lib.lib()
    _lib.check(lib.hm_cell_list_build(C.byref(ca), None))
    _lib.check(lib.hm_nlist_build(C.byref(na), None))
    _lib.check(lib.hm_synchronize())
    N = case["N"]

    class Box(C.Structure):
        _fields_ = [("lo", C.c_double * 3), ("L", C.c_double * 3), ("tilt", C.c_double * 3),
                    ("periodic", C.c_int * 3)]

    class Args(C.Structure):
        _fields_ = [("force", C.c_void_p), ("virial", C.c_void_p), ("pitch", C.c_size_t),
                    ("N", C.c_uint), ("n_max", C.c_uint), ("pos", C.c_void_p),
                    ("charge", C.c_void_p), ("box", Box), ("n_neigh", C.c_void_p),
                    ("nlist", C.c_void_p), ("head", C.c_void_p), ("rcutsq", C.c_void_p),
                    ("ronsq", C.c_void_p), ("size", C.c_size_t), ("ntypes", C.c_uint),
                    ("block", C.c_uint), ("shift", C.c_uint), ("with_virial", C.c_uint),
                    ("tpp", C.c_uint)]

    dev = dict(device="cuda", dtype=torch.float64)
    b["force"], b["virial"] = torch.zeros((N, 4), **dev), torch.zeros((6, N), **dev)
    b["head"] = torch.arange(N, device="cuda", dtype=torch.int64) * nmax
    b["rcutsq"], b["ronsq"] = torch.full((1,), 6.25, **dev), torch.zeros(1, **dev)
    b["params"] = torch.tensor([1.0, 4.0], **dev)
    a = Args()
    a.force, a.virial, a.pitch = b["force"].data_ptr(), b["virial"].data_ptr(), N
    a.N = a.n_max = N
    a.pos, a.n_neigh, a.nlist = b["pos"].data_ptr(), b["n_neigh"].data_ptr(), b["nlist"].data_ptr()
    for k in range(3):
        a.box.lo[k], a.box.L[k], a.box.periodic[k] = -L / 2, L, 1
    a.head, a.rcutsq, a.ronsq = b["head"].data_ptr(), b["rcutsq"].data_ptr(), b["ronsq"].data_ptr()
    a.size, a.ntypes, a.block, a.shift = N * nmax, 1, 256, 1
    a.with_virial, a.tpp = 1, case["tpp"]
    torch.cuda.synchronize()
    return dict(buffers=b, args=a)


def _lj_lists(case, seed):
    pos, L = _driver_positions(case, seed)
    b, ca, na, nmax = _list_args(pos, L, 2.5, 0.4)
    N = case["N"]
    b["force"] = torch.zeros((N, 4), device="cuda")
    pa = _lib.HmPairArgs()
    pa.N, pa.pos, pa.box, pa.ntypes = N, na.pos, na.box, 1
    pa.nlist, pa.nmax, pa.n_neigh = na.nlist, nmax, na.n_neigh
    pa.r_cut[0], pa.force = 2.5, b["force"].data_ptr()
    lj = (_lib.HmLJParams * 1)()
    lj[0].sigma = lj[0].epsilon = 1.0
    torch.cuda.synchronize()
    return dict(buffers=b, cell=ca, nlist=na, pair=pa, lj=lj, nmax=nmax)


# steps of equilibration in `prepare` (off the lattice, launch shapes chosen)
WARM = {"wca": 200, "lj": 100, "mixture": 100, "melt": 100, "cg": 100}


def prepare(case, seed):
    family = case["family"]
    if family == "run":
        sim, pos, thermo = _simulation(case, seed)
        sim.run(0 if case["method"] == "nve" else WARM[case["fluid"]])
        N = case["N"]
        smap = mlcg.SiteMap(np.arange(N + 1), np.arange(N))  # every particle its own site
        smap.attach(sim)
        fs = mlcg.FrameSet(1, N)
        s = dict(sim=sim, frame=fs, steps=case["steps"], thermo=thermo)
        s["pos"] = torch.as_tensor(_DeviceView(fs.d_pos.ptr, (N, 3)), device="cuda")
        s["force"] = torch.as_tensor(_DeviceView(fs.d_force.ptr, (N, 3)), device="cuda")
        s["x0"] = torch.from_numpy(pos.astype(np.float32)).cuda()
        s["L"] = torch.from_numpy(_edges(case).astype(np.float32)).cuda()
        return s
    if family in ("train", "lossgrad"):
        return _training(case, seed)
    if family == "batch":
        R = case["replicas"]
        rng = np.random.default_rng(R)  # the sizes belong to the case, the rest to the seed
        n = np.rint(np.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"]),
                                       R))).astype(int)
        rng = np.random.default_rng(seed)
        rho, kT = rng.uniform(0.7, 0.9, R), rng.uniform(0.8, 1.5, R)
        L = (n / rho) ** (1.0 / 3.0)
        b = ReplicaBatch([fcc_fill(int(n[k]), float(L[k]), rng) for k in range(R)], L, kT,
                         (seed + np.arange(R)) % 65536)
        b.thermalize()
        b.run(50)
        b.tune()
        return dict(batch=b, steps=case["steps"], L=np.repeat(L, n)[:, None])
    if family == "driver":
        return _lj_driver(case, seed)
    return _lj_lists(case, seed)


def run(state):
    if "sim" in state and "frame" in state:
        # a piece of the simulation, then the frame it reached (positions and net forces)
        state["sim"].run(state["steps"])
        state["frame"].record(state["sim"], 0)
        d = state["pos"] - state["x0"]
        out = dict(position=state["x0"] + (d - state["L"] * torch.round(d / state["L"])),
                   force=state["force"].clone())
        if state["thermo"] is not None:
            out["pressure"] = np.array(state["thermo"].pressure_tensor)
        return out
    if "net" in state:
        if state["n"] > 1:
            loss = state["net"].train(state["frames"], 1, lr=5e-4, frames_per_step=state["n"])
            return dict(loss=loss, params=state["net"].params)
        loss, grad = state["net"].loss_grad(state["frames"], 0)
        return dict(loss=np.array([loss]), grad=grad)
    if "batch" in state:
        b = state["batch"]
        b.run(state["steps"])
        x, v, image = (part[0].base for part in b.state())  # every replica's particles at once
        return dict(position=x + image * state["L"], velocity=v)
    lib = _lib.lib()
    if "args" in state:
        b = state["buffers"]
        _lib.check(lib.hm_compute_pair_forces_lj(C.byref(state["args"]), b["params"].data_ptr(),
                                                 None), "pair driver")
        return dict(force=b["force"], virial=b["virial"])
    b = state["buffers"]
    _lib.check(lib.hm_cell_list_build(C.byref(state["cell"]), None), "cells")
    _lib.check(lib.hm_nlist_build(C.byref(state["nlist"]), None), "list")
    _lib.check(lib.hm_pair_lj(C.byref(state["pair"]), state["lj"], None), "pair")
    return dict(n_neigh=b["n_neigh"], rows=b["nlist"], force=b["force"])


# ------------------------------------------------------------------------------------- costs
def work(case):
    """Bytes and operations of one pass. A step reads and writes each particle's position and
    velocity in FP64 (96 bytes); the pairs within the cutoff, each once, cost 27 operations (LJ)
    or 16 Gaussians in both passes (learned energy); its network 20 992 per site."""
    family = case["family"]

    def pairs(rho, rc):
        return 0.5 * rho * 4.0 / 3.0 * math.pi * rc ** 3

    if family == "run":
        N, K = case["N"], case["steps"]
        rc = {"wca": WCA, "melt": WCA, "lj": 2.5, "mixture": 2.4, "cg": 3.0}[case["fluid"]]
        per = pairs(case["rho"], rc) * 27.0 + 60.0
        if case["fluid"] == "cg":
            per = pairs(case["rho"], rc) * 16 * 20.0 + 20992.0 + 60.0
        return dict(bytes=K * N * 96.0 + N * 24.0, flops=K * N * per)
    if family in ("train", "lossgrad"):
        N, K = case["N"], case["frames"]
        return dict(bytes=K * N * 24.0, flops=K * N * (pairs(0.17, 3.0) * 16 * 60.0 + 6 * 10496.0))
    if family == "batch":
        lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
        N = case["replicas"] * (math.exp(hi) - math.exp(lo)) / (hi - lo)
        K = case["steps"]
        return dict(bytes=K * N * 96.0 + N * 60.0, flops=K * N * (pairs(0.8, 2.5) * 27.0 + 60.0))
    N = case["N"]
    row = 8.0 / 3.0 * math.pi * case["rho"] * 2.9 ** 3 / 2.0  # entries of a full row
    f = N * pairs(case["rho"], 2.5) * 27.0 * 2
    if family == "driver":
        return dict(bytes=N * (32.0 + 32.0 + 48.0 + 4.0 + 4.0 * row), flops=f)
    return dict(bytes=N * (32.0 + 16.0 + 4.0 + 4.0 * row), flops=f + N * row * 8.0)


def tolerance(case):
    """Runs and batches: about four times what another order of the FP32 pair sums (2 against 16
    lanes per particle) changed in two passes. Network: bf16 matrix products and dE/dG."""
    family = case["family"]
    if family == "run":
        return {"wca": dict(rel=1e-5, max=1e-3), "lj": dict(rel=2e-3, max=0.4),
                "mixture": dict(rel=1e-3, max=0.1), "melt": dict(rel=6e-4, max=0.02),
                "cg": dict(rel=0.01, max=0.5)}[case["fluid"]]
    if family in ("train", "lossgrad"):
        return dict(rel=0.01, max=0.5)
    if family == "batch":
        return dict(rel=2e-4, max=0.05)
    return dict(rel=2e-6, max=1e-3)


# ------------------------------------------------------------------------------------- 64 bits
def _lj_sums(x, L, rc, shift=False, virial=False):
    """Forces and energies (half of each pair) of LJ, all pairs, FP64."""
    N = len(x)
    out = torch.zeros((N, 4), dtype=torch.float64, device=x.device)
    vir = torch.zeros((6, N), dtype=torch.float64, device=x.device)
    s6 = 1.0 / rc ** 6
    e0 = 4.0 * (s6 * s6 - s6) if shift else 0.0
    chunk = max(1, (1 << 26) // N)
    for a in range(0, N, chunk):
        d = [x[a:a + chunk, k, None] - x[None, :, k] for k in range(3)]
        d = [t - L * torch.round(t / L) for t in d]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        i, j = torch.nonzero((r2 < rc * rc) & (r2 > 0), as_tuple=True)
        r2 = r2[i, j]
        d = torch.stack([t[i, j] for t in d], 1)
        inv = 1.0 / r2
        i6 = inv * inv * inv
        f = inv * i6 * (48.0 * i6 - 24.0)
        e = 0.5 * (4.0 * i6 * (i6 - 1.0) - e0)
        out[a:a + chunk].index_add_(0, i, torch.cat([d * f[:, None], e[:, None]], 1))
        if virial:
            for m, (p, q) in enumerate(((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))):
                vir[m, a:a + chunk].index_add_(0, i, 0.5 * f * d[:, p] * d[:, q])
    return out, vir


def _exact_nve(case, seed):
    pos, vel, _, _, _ = _start(case, seed)
    L = float(_edges(case)[0])
    rc = WCA if case["fluid"] == "wca" else 2.5
    x = torch.from_numpy(pos).cuda()
    v = torch.from_numpy(vel).cuda()
    dt = case["dt"]
    f = _lj_sums(x, L, rc)[0][:, :3]
    for _ in range(case["steps"]):
        v = v + 0.5 * dt * f
        x = x + dt * v
        f = _lj_sums(x, L, rc)[0][:, :3]
        v = v + 0.5 * dt * f
    return dict(position=x, force=f)


def _exact_loss(case, seed):
    """Loss and gradient over the frames' mean by automatic differentiation in FP64."""
    frames, L = _frames(case, seed)
    p = torch.from_numpy(mlcg.init_params(seed & 0xffff)).double().cuda().requires_grad_(True)
    W1, b1 = p[:1024].reshape(64, 16), p[1024:1088]
    W2, b2 = p[1088:5184].reshape(64, 64), p[5184:5248]
    w3, b3 = p[5248:5312], p[5312]
    mean, scale = (torch.from_numpy(a).cuda() for a in _normalization(case["rho"]))
    mu = 0.2 * torch.arange(16, dtype=torch.float64, device="cuda")
    losses, grads = [], []
    for pos, target in frames:
        x = torch.from_numpy(pos).double().cuda().requires_grad_(True)
        N = len(x)
        edges = []
        chunk = max(1, (1 << 26) // N)
        with torch.no_grad():
            for a in range(0, N, chunk):
                r2 = 0.0
                for k in range(3):
                    t = x[a:a + chunk, k, None] - x[None, :, k]
                    r2 = r2 + (t - L * torch.round(t / L)) ** 2
                e = torch.nonzero((r2 < 9.0) & (r2 > 0))
                e[:, 0] += a
                edges.append(e)
        i, j = torch.cat(edges).T
        d = x[i] - x[j]
        d = d - L * torch.round(d.detach() / L)
        r = d.square().sum(1).sqrt()
        phi = torch.exp(-(r[:, None] - mu) ** 2 / 0.08) \
            * (0.5 * (torch.cos(math.pi * r / 3.0) + 1.0))[:, None]
        G = torch.zeros((N, 16), dtype=torch.float64, device="cuda").index_add(0, i, phi)
        silu = torch.nn.functional.silu
        h = silu(silu(((G - mean) * scale) @ W1.T + b1) @ W2.T + b2)
        E = (h @ w3 + b3).sum()
        F = -torch.autograd.grad(E, x, create_graph=True)[0]
        loss = (F - torch.from_numpy(target).double().cuda()).square().sum() / (3.0 * N)
        grads.append(torch.autograd.grad(loss, p)[0])
        losses.append(loss.detach())
    return losses, grads


def exact(case, seed):
    family, N = case["family"], case["N"] if "N" in case else 0
    if family == "run":
        small = case["method"] == "nve" and N <= 40000
        return _exact_nve(case, seed) if small else None
    if family == "lossgrad":
        losses, grads = _exact_loss(case, seed)
        return dict(loss=torch.stack(losses), grad=grads[0])
    if family == "train" and N <= 60000:
        losses, grads = _exact_loss(case, seed)
        return dict(loss=torch.stack(losses).mean().reshape(1), params=None)
    if family in ("driver", "lists"):
        pos, L = _driver_positions(case, seed)
        x = torch.from_numpy(pos).cuda()
        if family == "driver":
            f, v = _lj_sums(x, L, 2.5, shift=True, virial=True)
            return dict(force=f, virial=v)
        return dict(n_neigh=None, rows=None, force=_lj_sums(x, L, 2.5)[0])
    return None
