"""The launches of the bond phase that carry a stage of the particles' chain: particle bins of every
size the in-bin sort treats apart, bonds dropped by the energy that absorption adds in the same step,
inner friction, and every workgroup size, against the oracle."""
import numpy as np
import pytest

from alien_amd import engine, worlds
from alien_amd.abi import MOTION_COLLISION, MOTION_FLUID
from oracle.pyoracle import from_world

from . import helpers as H
from .test_gpu_parity import assert_identical

pytestmark = pytest.mark.gpu


def world(motion, seed, bonds=True):
    """A mixed world (without bonds: its free cells alone) whose particles crowd some 8x8 bins: 1 to 20
    in a bin each."""
    w = worlds.random_mix(seed, motion=motion, size=(96, 80), num_particles=0, vel_sigma=0.2)
    rng = np.random.default_rng(seed)
    if not bonds:
        w.cells = w.cells[(w.cells["numConnections"] == 0) & (w.cells["barrier"] == 0)].copy()
        w.cells["maxConnections"] = 0
    pos = [np.array([8.0 * (k % 12), 8.0 * (k // 12)]) + rng.uniform(0.1, 7.9, (1 + k % 20, 2)) for k in range(60)]
    pos = np.concatenate(pos)
    parts = H.particles(len(pos))
    parts["pos"] = pos
    parts["vel"] = rng.normal(0, 0.3, pos.shape)
    parts["energy"] = rng.uniform(0.5, 3.0, len(pos))
    parts["color"] = rng.integers(0, 7, len(pos))
    w.particles = parts
    worlds.assign_ids(w.cells, w.particles)
    w.params = H.params(motion, smoothingLength=0.65, innerFriction=0.3, cellMaxBindingEnergy=101.0)
    return w


@pytest.mark.parametrize("threads", [64, 128, 192, 256])
@pytest.mark.parametrize("motion", [MOTION_FLUID, MOTION_COLLISION])
def test_bond_phase_with_particles(motion, threads):
    print("bond phase", motion, threads, flush=True)
    ws = [world(motion, 40 + threads), world(motion, 41 + threads, bonds=False)]
    refs = [from_world(w, precision=32) for w in ws]
    batch = engine.Batch()
    batch.set_block_size(threads)
    for w in ws:
        batch.add(w)
    for steps in (1, 3, 5):
        batch.step(steps)
        for k, ref in enumerate(refs):
            ref.step(steps)
            assert_identical(batch.get_data(k), ref.get_data(), f"world {k} motion {motion} threads {threads}")
    batch.close()


def test_particles_without_bond_work():
    w = world(MOTION_FLUID, 77, bonds=False)
    sim, ref = engine.Simulation.from_world(w), from_world(w, precision=32)
    for steps in (1, 6):
        sim.step(steps)
        ref.step(steps)
        assert_identical(sim.get_data(), ref.get_data(), "fluid world without bonds")
    sim.close()
