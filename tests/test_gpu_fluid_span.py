"""The fluid pass at the sizes where its waves change their number of cells (16, 32, 64), in a thin fluid and
in crowds whose pairs exceed a wave's records, with a crowd on the torus' edge columns, against the oracle."""
import numpy as np
import pytest

from alien_amd import engine, worlds
from alien_amd.abi import MOTION_FLUID
from oracle.pyoracle import from_world

from . import helpers as H
from .test_gpu_parity import assert_identical

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bonds", [False, True])
@pytest.mark.parametrize("cells", [16384, 16416, 32767, 32832, 65535, 66000])
def test_cells_per_wave(cells, bonds):
    print("fluid span", cells, bonds, flush=True)
    rng = np.random.default_rng(cells + bonds)
    size = (420, 400)
    thin = cells * 3 // 4
    pos = [rng.uniform(0, 1, (thin, 2)) * size]
    for x, y, w, h, n in ((100, 100, 90, 70, cells - thin - 300), (0, 50, 2, 60, 150), (418, 55, 2, 60, 150)):
        pos.append(np.array([x, y]) + rng.uniform(0, 1, (n, 2)) * [w, h])
    c = H.cells(cells)
    c["connections"]["cellIndex"] = 0
    c["pos"] = np.minimum(np.concatenate(pos).astype(np.float32), np.nextafter(np.float32(size), np.float32(0)))
    c["vel"] = rng.normal(0, 0.2, (cells, 2))
    c["maxConnections"] = rng.integers(0, 6, cells) if bonds else 0
    parts = H.particles(0)
    worlds.assign_ids(c, parts)
    w = worlds.World("span", size, H.params(MOTION_FLUID, smoothingLength=0.8), c, parts, 5, 3)
    sim, ref = engine.Simulation.from_world(w), from_world(w, precision=32, threads=8)
    for steps in (1, 2):
        sim.step(steps)
        ref.step(steps)
        assert_identical(sim.get_data(), ref.get_data(), f"{cells} bonds={bonds} after {steps} more steps")
    sim.close()
