"""The column form of the list build (csrc/tile.hip) inside the engine: slot rows staged from the relative
positions and index rows staged from the cell entries, with types, exclusions, crowded regions, few cells along
an axis and rows that overflow. The first list is the oracle's, pair for pair, and the forces before and after
rebuilds are those of an FP64 sum. Then the choice between this form and the cell form."""

import numpy as np
import pytest

import oracle as O
from gpu_helpers import rel_rms

pytestmark = pytest.mark.gpu

WCA = 2.0 ** (1.0 / 6.0)
COLUMNS = 5  # hm_sys_nlist_launch


@pytest.fixture(scope="module")
def hoomd():
    import hoomd_amd
    from hoomd_amd import _lib
    assert _lib.lib().hm_device_count() > 0
    return hoomd_amd


def lattice(N, L, seed, jitter=0.05):
    """N sites, chosen at random, of a simple cubic lattice stretched over the box, each moved a little."""
    L = np.asarray(L, float)
    n = np.ceil(L * (N / L.prod()) ** (1.0 / 3.0)).astype(int)
    rng = np.random.default_rng(seed)
    k = rng.choice(n.prod(), N, replace=False)
    x = np.stack([k % n[0], k // n[0] % n[1], k // (n[0] * n[1])], axis=1)
    x = (x + 0.5) * (L / n) - L / 2 + rng.uniform(-jitter, jitter, (N, 3))
    return x, L


def cells(L, r_list):
    return np.floor(np.asarray(L) / r_list).astype(int)


def make(hoomd, pos, L, rc, buff, types=None, bonds=None, kT=0.0, sorter=False, seed=3):
    nt = rc.shape[0]
    d = cells(L, rc.max() + buff)
    # the rule of the column build, so that no case here takes the other form unseen
    assert len(pos) >= 32768 and len(pos) <= 8 * d.prod() and d.min() >= 4
    snap = hoomd.Snapshot()
    snap.configuration.box = [*L, 0, 0, 0]
    snap.particles.N = len(pos)
    snap.particles.types = ["A", "B", "C", "D"][:nt]
    snap.particles.position[:] = pos
    if types is not None:
        snap.particles.typeid[:] = types
    if kT:
        snap.particles.velocity[:] = np.random.default_rng(seed).normal(0, np.sqrt(kT), pos.shape)
    if bonds is not None:
        snap.bonds.N = len(bonds)
        snap.bonds.types = ["b"]
        snap.bonds.group[:] = bonds
    sim = hoomd.Simulation(device=hoomd.device.GPU(), seed=seed)
    sim.create_state_from_snapshot(snap)
    lj = hoomd.md.pair.LJ(nlist=hoomd.md.nlist.Cell(buffer=buff, exclusions=("bond",)))
    for a in range(nt):
        for b in range(nt):
            lj.params[("ABCD"[a], "ABCD"[b])] = dict(epsilon=1.0, sigma=1.0)
            lj.r_cut[("ABCD"[a], "ABCD"[b])] = rc[a, b]
    forces = [lj]
    if bonds is not None:
        h = hoomd.md.bond.Harmonic()
        h.params["b"] = dict(k=1.0, r0=1.0)
        forces.append(h)
    sim.operations.integrator = hoomd.md.Integrator(
        dt=0.002, forces=forces, methods=[hoomd.md.methods.ConstantVolume(hoomd.filter.All())])
    sim.operations.tuners.clear()
    if sorter:
        sim.operations.add(hoomd.tune.ParticleSorter(trigger=20, grid=32))
    return sim, lj


def columns(sim, kind=2):
    """The first list by the cell form, then columns. kind 2: slot rows, 1: index rows."""
    from hoomd_amd import _lib
    sim.run(0)
    if kind != 2:
        _lib.check(_lib.lib().hm_sys_set_pair_kernel(sim._system, kind, 0, 0))
    _lib.check(_lib.lib().hm_sys_set_nlist_launch(sim._system, COLUMNS, 0))
    sim.run(0)


def bonded(N, bonds):
    e = [[] for _ in range(N)]
    for a, b in bonds:
        e[a].append(b)
        e[b].append(a)
    return e


def check(lj, pos, L, rc, buff, types=None, excl=None, pairs=True):
    """Forces of every particle from its own row, and the list's pairs."""
    nt = rc.shape[0]
    nl, nn = O.nlist_binned(O.Box(*L), pos, rc, buff, full=True, types=types, ntypes=nt, excl=excl)
    i = np.repeat(np.arange(len(pos)), nn)
    j = nl[np.arange(nl.shape[1])[None, :] < nn[:, None]].astype(int)
    if pairs:
        got = np.asarray(lj.nlist.pair_list, np.int64)
        half = i < j
        ref = np.sort(i[half] * len(pos) + j[half])
        assert np.array_equal(np.sort(got[:, 0] * len(pos) + got[:, 1]), ref)
    d = pos[i] - pos[j]
    d -= L * np.rint(d / L)
    r2 = (d * d).sum(1)
    t = np.zeros(len(pos), int) if types is None else types
    r2c = rc[t[i], t[j]] ** 2
    inv = 1.0 / r2
    f = np.zeros((len(pos), 3))
    w = np.where(r2 < r2c, inv * inv ** 3 * (48.0 * inv ** 3 - 24.0), 0.0)
    np.add.at(f, i, d * w[:, None])
    assert rel_rms(lj.forces, f) < 1e-5  # the bar of the first forces of every engine test


def one(r):
    return np.array([[float(r)]])


@pytest.mark.parametrize("N,L,rc,buff", [
    (33000, (32.0, 32.1, 32.2), WCA, 0.4),    # 3 a cell, 4 lanes per particle
    (33000, (50.0, 36.0, 45.0), 2.0, 0.4),    # 6.5 a cell, 8 lanes per particle
    (33000, (6.2, 73.0, 73.1), WCA, 0.4),     # 4 cells along x
    (33000, (73.0, 6.2, 73.1), WCA, 0.4),     # along y
    (33000, (73.0, 73.1, 6.2), WCA, 0.4),     # along z: columns of one cell
    (150000, (54.0, 52.0, 54.5), WCA, 0.4),   # columns of several cells
])
@pytest.mark.parametrize("kind", [2, 1])
def test_first_list_and_forces(hoomd, N, L, rc, buff, kind):
    pos, L = lattice(N, L, N)
    sim, lj = make(hoomd, pos, L, one(rc), buff)
    columns(sim, kind)
    check(lj, pos, L, one(rc), buff)


@pytest.mark.parametrize("kind", [2, 1])
def test_types(hoomd, kind):
    pos, L = lattice(34001, (44.0, 45.0, 46.0), 5)
    types = np.random.default_rng(6).integers(0, 3, len(pos)).astype(np.uint32)
    rc = np.array([[1.8, 1.2, 1.5], [1.2, 0.0, 1.7], [1.5, 1.7, 1.6]])
    sim, lj = make(hoomd, pos, L, rc, 0.3, types=types, kT=1.0, sorter=True)
    columns(sim, kind)
    check(lj, pos, L, rc, 0.3, types=types)
    sim.run(60)
    assert lj.nlist.num_builds >= 2
    s = sim.state.get_snapshot().particles
    check(lj, s.position, L, rc, 0.3, types=types, pairs=False)


def near_bonds(pos, L, r, most=4):
    """Bonds between near particles, across the faces too, up to four a particle."""
    nl, nn = O.nlist_binned(O.Box(*L), pos, r, 0.0, full=True)
    left, out = np.full(len(pos), most), []
    for i in range(len(pos)):
        for j in nl[i, :nn[i]]:
            if i < j and left[i] and left[j] and (i + j) % 3:
                out.append((i, int(j)))
                left[i] -= 1
                left[j] -= 1
    return np.array(out, np.uint32), left


@pytest.mark.parametrize("kind", [2, 1])
@pytest.mark.parametrize("L", [(32.0, 32.1, 32.2), (73.0, 73.1, 6.2)])
def test_exclusions(hoomd, L, kind):
    pos, L = lattice(33000, L, 7)
    bonds, left = near_bonds(pos, L, 1.25)
    d = np.abs(pos[bonds[:, 0]] - pos[bonds[:, 1]])
    assert all((d[:, k] > L[k] / 2).sum() > 100 for k in range(3)) and (left == 0).sum() > 100
    excl = bonded(len(pos), bonds)
    sim, lj = make(hoomd, pos, L, one(WCA), 0.4, bonds=bonds, kT=1.0, sorter=True)
    columns(sim, kind)
    check(lj, pos, L, one(WCA), 0.4, excl=excl)
    sim.run(60)
    assert lj.nlist.num_builds >= 2
    check(lj, sim.state.get_snapshot().particles.position, L, one(WCA), 0.4, excl=excl, pairs=False)


def slab(N=40000, seed=8):
    """A liquid at 0.85 in 35 % of the box, the rest empty: 7 particles a cell, 20 in the liquid."""
    pos, l = lattice(N, (21.2, 47.0, 47.3), seed)
    return pos, np.array([60.5, 47.0, 47.3])


@pytest.mark.parametrize("types", [False, True])
def test_crowded_columns(hoomd, types):
    pos, L = slab()
    rc, t = one(2.5), None
    if types:
        rc = np.array([[2.5, 2.2], [2.2, 1.9]])
        t = (np.arange(len(pos)) % 2).astype(np.uint32)
    sim, lj = make(hoomd, pos, L, rc, 0.4, types=t, kT=1.0)
    columns(sim)
    check(lj, pos, L, rc, 0.4, types=t)
    sim.run(60)
    assert lj.nlist.num_builds >= 2
    check(lj, sim.state.get_snapshot().particles.position, L, rc, 0.4, types=t, pairs=False)


@pytest.mark.parametrize("kind", [2, 1])
def test_exclusions_in_crowded_columns(hoomd, kind):
    pos, L = slab()
    bonds, _ = near_bonds(pos, L, 1.25)
    sim, lj = make(hoomd, pos, L, one(2.5), 0.4, bonds=bonds)
    columns(sim, kind)
    check(lj, pos, L, one(2.5), 0.4, excl=bonded(len(pos), bonds))


def test_a_packed_region(hoomd):
    """Cells that hold more than any stage: 27 of them are read from memory."""
    pos, L = lattice(34500, (80.0, 81.0, 82.0), 9)
    rng = np.random.default_rng(10)
    # 4 000 particles within four cells an edge, at least 0.54 apart: 120 a cell
    g = np.stack(np.meshgrid(*[np.arange(16)] * 3), -1).reshape(-1, 3)[:4000]
    pos[:4000] = (g + 0.5) * 0.6 - 0.05 + rng.uniform(-0.03, 0.03, (4000, 3)) - 5.0
    keep = np.abs(pos[4000:]).max(1) > 8.0
    pos = np.concatenate([pos[:4000], pos[4000:][keep]])
    assert len(pos) >= 32768
    sim, lj = make(hoomd, pos, L, one(2.5), 0.4)
    columns(sim)
    check(lj, pos, L, one(2.5), 0.4)


@pytest.mark.parametrize("cmax,nmax", [(2, 256), (64, 8)])
def test_overflow_replays(hoomd, cmax, nmax):
    from hoomd_amd import _lib
    pos, L = lattice(33000, (32.0, 32.1, 32.2), 11)
    sim, lj = make(hoomd, pos, L, one(WCA), 0.4, kT=1.0)
    columns(sim)
    sim.run(5)
    _lib.check(_lib.lib().hm_sys_set_list_capacity(sim._system, cmax, nmax))
    sim.run(20)
    check(lj, sim.state.get_snapshot().particles.position, L, one(WCA), 0.4, pairs=False)


def nlist_launch(sim):
    """Shape in use, whether the cache answered, rows (shape, grid, ms) of the last sweep."""
    from hoomd_amd import _lib
    out, log = np.zeros(3, np.int32), np.zeros((64, 3), np.float32)
    rows = _lib.lib().hm_sys_nlist_launch(sim._system, out.ctypes.data, log.ctypes.data, 64)
    return int(out[0]), bool(out[2]), log[:rows]


def test_tuner_times_both_forms(hoomd):
    """The mean density decides whether the column form can be used, the sweep whether it is."""
    from hoomd_amd import _lib
    for pos, L in (lattice(33000, (32.0, 32.1, 32.2), 12), slab()):
        _lib.lib().hm_tune_cache_clear()
        r = WCA if L[0] < 40 else 2.5
        sim, _ = make(hoomd, pos, L, one(r), 0.4)
        sim.run(0)
        shape, cached, log = nlist_launch(sim)
        print(shape, [(int(a), int(b), round(float(c) * 1e3, 1)) for a, b, c in log], flush=True)
        assert not cached and (log[:, 0] == COLUMNS).sum() == 1 and (log[:, 0] != COLUMNS).sum() >= 2
        assert shape == log[np.argmin(log[:, 2]), 0]


def test_tuner_times_again_where_columns_become_crowded(hoomd):
    """Tuned on a dilute uniform fluid, then the particles lie in a slab: the next runs take the form that is
    faster there, and only once."""
    from hoomd_amd import _lib
    _lib.lib().hm_tune_cache_clear()
    pos, L = lattice(130000, (69.0, 69.1, 69.2), 14)
    sim, lj = make(hoomd, pos, L, one(WCA), 0.4, sorter=True)
    sim.run(10)
    assert nlist_launch(sim)[0] == COLUMNS
    d = np.ascontiguousarray(lattice(len(pos), (29.0, 69.1, 69.2), 15)[0])
    _lib.check(_lib.lib().hm_sys_set_state(sim._system, d.ctypes.data, None, None))
    _lib.check(_lib.lib().hm_sys_set_chunk(sim._system, 10, 1))
    sim.run(60)
    assert lj.nlist.num_builds >= 2
    shape, _, log = nlist_launch(sim)
    print(shape, [(int(a), int(b), round(float(c) * 1e3, 1)) for a, b, c in log], flush=True)
    assert shape != COLUMNS and shape == log[np.argmin(log[:, 2]), 0]


def test_shape_set_by_the_caller_is_kept(hoomd):
    pos, L = slab()
    sim, lj = make(hoomd, pos, L, one(2.5), 0.4, kT=1.0)
    from hoomd_amd import _lib
    columns(sim)
    _lib.check(_lib.lib().hm_sys_set_chunk(sim._system, 10, 1))
    sim.run(60)
    assert lj.nlist.num_builds >= 2 and nlist_launch(sim)[0] == COLUMNS
    _lib.check(_lib.lib().hm_sys_set_nlist_launch(sim._system, 0, 0))
    sim.run(1)
    shape, cached, log = nlist_launch(sim)
    assert cached or shape == log[np.argmin(log[:, 2]), 0]
    assert _lib.lib().hm_sys_set_nlist_launch(sim._system, 6, 0) == -2


def test_tuner_cache_keeps_the_forms_apart(hoomd):
    """33 000 particles may be built over columns, 32 600 may not: the smaller system is swept by itself."""
    from hoomd_amd import _lib
    _lib.lib().hm_tune_cache_clear()
    for N in (33000, 32600):
        pos, L = lattice(33000, (32.0, 32.1, 32.2), 13)
        keep = np.random.default_rng(1).permutation(33000)[:N]
        snap = hoomd.Snapshot()
        snap.configuration.box = [*L, 0, 0, 0]
        snap.particles.N = N
        snap.particles.types = ["A"]
        snap.particles.position[:] = pos[keep]
        sim = hoomd.Simulation(device=hoomd.device.GPU(), seed=1)
        sim.create_state_from_snapshot(snap)
        lj = hoomd.md.pair.LJ(nlist=hoomd.md.nlist.Cell(buffer=0.4), default_r_cut=WCA)
        lj.params[("A", "A")] = dict(epsilon=1.0, sigma=1.0)
        sim.operations.integrator = hoomd.md.Integrator(
            dt=0.002, forces=[lj], methods=[hoomd.md.methods.ConstantVolume(hoomd.filter.All())])
        sim.run(0)
        shape, cached, log = nlist_launch(sim)
        assert not cached and len(log) > 1 and (COLUMNS in log[:, 0]) == (N >= 32768)
