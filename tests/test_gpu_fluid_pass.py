"""The fluid neighbour pass where it splits its work: grids of three bins and of more, the torus' edge
columns and rows, bins of three units, more cells than an edge wave, a stage or a window of pairs takes,
against the oracle; without bond work (a variant of its own) and with it."""
import numpy as np
import pytest

from alien_amd import engine, worlds
from alien_amd.abi import MOTION_FLUID
from oracle.pyoracle import from_world

from . import helpers as H
from .test_gpu_parity import assert_identical

pytestmark = pytest.mark.gpu

# name: size, cells, smoothing length, crowds (x, y, w, h, cells)
CASES = {
    "three bins": ((6, 7), 25, 0.65, ()),
    "one wave high": ((300, 6), 400, 0.8, ()),
    "three bins wide": ((7, 240), 400, 0.65, ()),
    "small": ((64, 64), 1200, 0.65, ()),
    "three-unit bins": ((131, 97), 3500, 1.2, ()),
    "crowded edge column": ((120, 100), 900, 0.65, ((0, 30, 2, 2, 30), (118, 30, 2, 2, 9), (0, 60, 1, 2, 7), (119, 57, 1, 2, 70))),
    "crowded edge rows": ((120, 100), 900, 0.65, ((30, 0, 20, 2, 200), (50, 98, 20, 2, 200))),
    "more than the stage": ((160, 100), 600, 0.65, ((40, 40, 24, 24, 900), (90, 20, 2, 2, 60))),
    "more than a window": ((96, 96), 300, 0.8, ((20, 20, 30, 6, 500),)),
    "sparse": ((700, 500), 150, 0.65, ()),
}


def world(name, bonds):
    size, n, h, crowds = CASES[name]
    rng = np.random.default_rng(len(name) + 31 * n)
    pos = [rng.uniform(0, 1, (n, 2)) * np.array(size)]
    for x, y, w, k, cnt in crowds:
        pos.append(np.array([x, y]) + rng.uniform(0, 1, (cnt, 2)) * np.array([w, k]))
    pos = np.concatenate(pos)
    cells = H.cells(len(pos))
    cells["connections"]["cellIndex"] = 0
    cells["pos"] = pos.astype(np.float32)
    cells["vel"] = rng.normal(0, 0.3, pos.shape)
    # on the far edges, and just inside of them on the way out
    cells["pos"][:3] = [[np.nextafter(np.float32(size[0]), np.float32(0)), 1.5], [2.5, np.nextafter(np.float32(size[1]), np.float32(0))],
                        [0.0, 0.0]]
    cells["color"] = rng.integers(0, 7, len(pos))
    cells["maxConnections"] = 0
    if bonds:
        cells["maxConnections"] = rng.integers(0, 7, len(pos))
        cells["barrier"][rng.choice(len(pos), len(pos) // 20, replace=False)] = 1
    parts = H.particles(0)
    worlds.assign_ids(cells, parts)
    return worlds.World(name, size, H.params(MOTION_FLUID, smoothingLength=h, cellFusionVelocity=0.4), cells, parts, 5, 3)


@pytest.mark.parametrize("bonds", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_fluid_pass(name, bonds):
    print("fluid pass", name, bonds, flush=True)
    w = world(name, bonds)
    sim, ref = engine.Simulation.from_world(w), from_world(w, precision=32, threads=8)
    for steps in (1, 1, 4):
        sim.step(steps)
        ref.step(steps)
        assert_identical(sim.get_data(), ref.get_data(), f"{name} bonds={bonds}")
    sim.close()
