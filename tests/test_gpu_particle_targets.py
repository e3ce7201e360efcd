"""The particles' search for what they fuse with and what absorbs them: bins at the far edges (up to 15 units
wide where the side is no multiple of eight), worlds smaller than a bin, several particles and cells in a slot,
against the oracle."""
import numpy as np
import pytest

from alien_amd import engine, worlds
from alien_amd.abi import MOTION_COLLISION, MOTION_FLUID
from oracle.pyoracle import from_world

from . import helpers as H
from .test_gpu_parity import assert_identical

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("motion", [MOTION_FLUID, MOTION_COLLISION])
@pytest.mark.parametrize("size", [(6, 7), (7, 31), (15, 15), (29, 23), (64, 47), (111, 95)])
def test_targets(size, motion):
    print("particle targets", size, motion, flush=True)
    rng = np.random.default_rng(size[0] * 100 + size[1] + motion)
    area = size[0] * size[1]
    cells = H.cells(max(3, area // 6))
    cells["connections"]["cellIndex"] = 0
    cells["pos"] = np.minimum((rng.uniform(0, 1, (len(cells), 2)) * size).astype(np.float32),
                              np.nextafter(np.float32(size), np.float32(0)))
    cells["vel"] = rng.normal(0, 0.2, (len(cells), 2))
    cells["maxConnections"] = 0
    cells["barrier"][::7] = 1
    parts = H.particles(max(12, area // 3))
    pos = rng.uniform(0, 1, (len(parts), 2)) * size
    pos[: len(parts) // 3] = np.floor(pos[: len(parts) // 3] / 4) * 4 + rng.uniform(0, 0.6, (len(parts) // 3, 2))
    parts["pos"] = np.minimum(pos.astype(np.float32), np.nextafter(np.float32(size), np.float32(0)))
    parts["vel"] = rng.normal(0, 0.5, (len(parts), 2))
    parts["energy"] = rng.uniform(0.3, 4.0, len(parts))
    worlds.assign_ids(cells, parts)
    w = worlds.World("targets", size, H.params(motion, smoothingLength=0.65), cells, parts, 5, 3)
    sim, ref = engine.Simulation.from_world(w), from_world(w, precision=32)
    for steps in (1, 1, 5):
        sim.step(steps)
        ref.step(steps)
        assert_identical(sim.get_data(), ref.get_data(), f"{size} after {steps} more steps")
    sim.close()
