"""The neighbour passes' edge columns: more cells in a row's edge bins than waves for them, more candidates
than lanes, worlds so tall that groups of rows share their waves, several worlds in one set; no cell of an
edge column is left to a lane of its own; against the oracle."""
import numpy as np
import pytest

from alien_amd import engine, worlds
from alien_amd.abi import MOTION_COLLISION, MOTION_FLUID
from oracle.pyoracle import from_world

from . import helpers as H
from .test_gpu_parity import assert_identical

pytestmark = pytest.mark.gpu

# name: size, cells, reach, cells of crowds on the edge columns (left and right, two units wide)
CASES = {
    "few": ((60, 64), 500, 1.3, (9, 12)),
    "more cells than waves": ((80, 120), 900, 1.3, (30, 50)),
    "more candidates than lanes": ((80, 64), 300, 1.3, (70, 140)),
    "wide bins": ((121, 131), 2500, 6.0, (40, 25)),
    "two rows to a group": ((20, 1300), 2500, 1.3, (20, 40)),
    "eight rows to a group": ((14, 4600), 5000, 1.3, (25, 17)),
    "three bins wide and tall": ((6, 4500), 2500, 1.3, (12, 6)),
}


def world(name, motion, bonds):
    size, n, reach, crowds = CASES[name]
    rng = np.random.default_rng(n + motion)
    pos = [rng.uniform(0, 1, (n, 2)) * np.array(size)]
    for x, cnt, y in ((0, crowds[0], size[1] / 3), (size[0] - 2, crowds[1], size[1] / 3 + 1), (0, crowds[1], 0),
                      (size[0] - 2, crowds[0], size[1] - 2)):
        pos.append(np.array([x, y]) + rng.uniform(0, 2, (cnt, 2)))
    pos = np.concatenate(pos)
    cells = H.cells(len(pos))
    cells["connections"]["cellIndex"] = 0
    cells["pos"] = np.minimum(pos.astype(np.float32), np.nextafter(np.float32(size), np.float32(0)))
    cells["vel"] = rng.normal(0, 0.2, pos.shape)
    cells["maxConnections"] = 0
    if bonds:
        cells["maxConnections"][rng.choice(len(pos), len(pos) // 20, replace=False)] = 3
        cells["barrier"][rng.choice(len(pos), len(pos) // 30, replace=False)] = 1
    parts = H.particles(0)
    worlds.assign_ids(cells, parts)
    return worlds.World(name, size, H.params(motion, smoothingLength=reach / 2, cellMaxCollisionDistance=reach), cells, parts,
                        5, 3)


@pytest.mark.parametrize("motion,bonds", [(MOTION_FLUID, False), (MOTION_FLUID, True), (MOTION_COLLISION, True)])
@pytest.mark.parametrize("name", list(CASES))
def test_edge_columns(name, motion, bonds):
    print("edge columns", name, motion, bonds, flush=True)
    w = world(name, motion, bonds)
    sim, ref = engine.Simulation.from_world(w), from_world(w, precision=32, threads=8)
    sim.step(1)
    ref.step(1)
    assert_identical(sim.get_data(), ref.get_data(), name)
    if CASES[name][2] < 2.0:  # (with wide bins the cells next to the columns have long lists)
        assert sim.path_counts() == (0, 0)
    sim.step(3)
    ref.step(3)
    assert_identical(sim.get_data(), ref.get_data(), f"{name} after 3 more steps")
    sim.close()


def test_edge_columns_of_several_worlds():
    print("edge columns of several worlds", flush=True)
    several = [world(n, (MOTION_FLUID, MOTION_COLLISION)[k % 2], True) for k, n in enumerate(CASES)]
    batch = engine.Batch()
    for w in several:
        batch.add(w)
    refs = [from_world(w, precision=32, threads=8) for w in several]
    batch.step(3)
    for k, ref in enumerate(refs):
        ref.step(3)
        assert_identical(batch.get_data(k), ref.get_data(), several[k].name)
    batch.close()
