"""Steps inside a chunk (one launch between two steps) against chunks of one step (separate step-one and
step-two launches): the same bits, for each method and each way of forming the Bussi factor."""

import numpy as np
import pytest

from lattices import fcc_lattice, maxwell_boltzmann

pytestmark = pytest.mark.gpu


def final_state(n, method, chunk, steps):
    import hoomd_amd as hoomd
    from hoomd_amd import _lib
    pos, L = fcc_lattice(n)
    snap = hoomd.Snapshot()
    snap.configuration.box = [L, L, L, 0, 0, 0]
    snap.particles.N = len(pos)
    snap.particles.types = ["A"]
    snap.particles.position[:] = pos
    snap.particles.velocity[:] = maxwell_boltzmann(len(pos), 1.2)
    sim = hoomd.Simulation(device=hoomd.device.GPU(), seed=7)
    sim.create_state_from_snapshot(snap)
    lj = hoomd.md.pair.LJ(nlist=hoomd.md.nlist.Cell(buffer=0.4), default_r_cut=2.5)
    lj.params[("A", "A")] = dict(epsilon=1.0, sigma=1.0)
    bussi = hoomd.md.methods.thermostats.Bussi(kT=1.2)
    m = {"nve": lambda: hoomd.md.methods.ConstantVolume(hoomd.filter.All()),
         "bussi": lambda: hoomd.md.methods.ConstantVolume(hoomd.filter.All(), thermostat=bussi),
         "langevin": lambda: hoomd.md.methods.Langevin(hoomd.filter.All(), kT=1.2)}[method]()
    sim.operations.integrator = hoomd.md.Integrator(dt=0.005, forces=[lj], methods=[m])
    sim.run(0)
    # a fixed pair launch: the order of the force sums is the same on both sides
    _lib.check(_lib.lib().hm_sys_set_pair_kernel(sim._system, 2, 8, 128))
    _lib.check(_lib.lib().hm_sys_set_chunk(sim._system, chunk, 1))
    sim.run(steps)
    p = sim.state.get_snapshot().particles
    return p.position, p.velocity, p.image, p.acceleration


# 8: 2 048 particles; 41: 275 684 particles, 1 077 partial sums (the Bussi factor's own launch)
@pytest.mark.parametrize("n,method,chunk,steps", [
    (8, "nve", 7, 40), (8, "bussi", 2, 40), (8, "bussi", 150, 310), (8, "langevin", 100, 60),
    (41, "bussi", 20, 25), (41, "langevin", 3, 8)])
def test_chunk_equals_single_steps(n, method, chunk, steps):
    for a, b in zip(final_state(n, method, chunk, steps), final_state(n, method, 1, steps)):
        assert np.array_equal(a, b)
