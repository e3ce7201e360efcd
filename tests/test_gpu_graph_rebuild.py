"""Particles that die out in the middle of a call: their kernels go while steps captured with them are
still queued, and the rest of the call runs graphs captured anew."""
import numpy as np
import pytest

from alien_amd import engine, worlds
from alien_amd.abi import MOTION_FLUID
from oracle.pyoracle import from_world

from . import helpers as H
from .test_gpu_parity import assert_identical

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bonds", [0, 2])
def test_particles_gone_within_a_call(bonds):
    print("particles gone within a call", bonds, flush=True)
    rng = np.random.default_rng(19 + bonds)
    cells = H.cells(9000)
    cells["connections"]["cellIndex"] = 0
    cells["pos"] = rng.uniform(0, 96, (9000, 2)).astype(np.float32)
    cells["vel"] = rng.normal(0, 0.1, (9000, 2))
    cells["maxConnections"] = bonds
    parts = H.particles(300)
    parts["pos"] = rng.uniform(0, 96, (300, 2)).astype(np.float32)
    parts["vel"] = rng.normal(0, 0.3, (300, 2))
    parts["energy"] = 0.01
    worlds.assign_ids(cells, parts)
    w = worlds.World("dying", (96, 96), H.params(MOTION_FLUID), cells, parts, 5, 0)
    sim, ref = engine.Simulation.from_world(w), from_world(w, precision=32, threads=8)
    for n in (333, 200):  # several calls' worth of queued graphs before the particles are seen gone
        sim.step(n)
        ref.step(n)
        got, want = sim.get_data(), ref.get_data()
        assert_identical(got, want, f"bonds={bonds} after {n} more steps")
    assert len(want[1]) == 0
    sim.close()
