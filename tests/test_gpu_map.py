"""The map of the cells where it splits its work: worlds narrower and wider than a group of 256 bins, more
groups than one sum of groups, bins of more than a round of 64 cells, more movers into a group than its
list takes, movers further than a bin and across the torus' edges, and the steps after introspection,
against the oracle."""
import numpy as np
import pytest

from alien_amd import engine, worlds
from alien_amd.abi import MOTION_COLLISION, MOTION_FLUID
from oracle.pyoracle import from_world

from . import helpers as H
from .test_gpu_parity import assert_identical

pytestmark = pytest.mark.gpu

# name: size, cells, speed, crowds (x, y, width, height, cells)
CASES = {
    "three bins": ((6, 6), 30, 0.5, ()),
    "narrow": ((6, 4000), 6000, 0.6, ()),
    "low": ((4000, 6), 6000, 0.6, ()),
    "one row a group": ((512, 70), 9000, 0.4, ()),
    "ragged": ((701, 203), 30000, 0.3, ()),
    "several sums of groups": ((2000, 700), 20000, 0.5, ()),
    "fast": ((300, 200), 9000, 3.0, ()),
    "crowded bins": ((200, 150), 2000, 0.3, ((40, 40, 2, 2, 330), (60, 100, 4, 2, 300))),
    "more movers than the list": ((260, 100), 1000, 0.1, ((0, 40, 260, 8, 5000),)),
    "empty but for a corner": ((900, 900), 8, 0.5, ((0, 0, 9, 9, 60), (890, 890, 10, 10, 60))),
}


def world(name, motion):
    size, n, speed, crowds = CASES[name]
    rng = np.random.default_rng(len(name) + 7 * n + motion)
    pos = [rng.uniform(0, 1, (n, 2)) * np.array(size)]
    for x, y, w, h, cnt in crowds:
        pos.append(np.array([x, y]) + rng.uniform(0, 1, (cnt, 2)) * np.array([w, h]))
    pos = np.concatenate(pos)
    cells = H.cells(len(pos))
    cells["connections"]["cellIndex"] = 0
    cells["pos"] = np.minimum(pos.astype(np.float32), np.nextafter(np.float32(size), np.float32(0)))
    cells["vel"] = rng.normal(0, speed, pos.shape)
    if name == "more movers than the list":
        cells["vel"][n:] = [0.0, 1.9]  # a row of bins and more moves on together
    cells["maxConnections"] = 0
    parts = H.particles(0)
    worlds.assign_ids(cells, parts)
    return worlds.World(name, size, H.params(motion, cellMaxVelocity=4.0), cells, parts, 5, 3)


@pytest.mark.parametrize("motion", [MOTION_FLUID, MOTION_COLLISION])
@pytest.mark.parametrize("name", list(CASES))
def test_map(name, motion):
    print("map", name, motion, flush=True)
    w = world(name, motion)
    sim, ref = engine.Simulation.from_world(w), from_world(w, precision=32, threads=8)
    for k, steps in enumerate((1, 1, 3, 2)):
        sim.step(steps)
        ref.step(steps)
        assert_identical(sim.get_data(), ref.get_data(), f"{name} after {steps} more steps")
        if k == 1:
            sim.get_map()  # (enters every cell anew)
    sim.close()


def test_map_of_several_worlds():
    print("map of several worlds", flush=True)
    names = ["three bins", "fast", "ragged", "narrow", "several sums of groups", "crowded bins"]
    several = [world(n, (MOTION_FLUID, MOTION_COLLISION)[k % 2]) for k, n in enumerate(names)]
    batch = engine.Batch()
    for w in several:
        batch.add(w)
    refs = [from_world(w, precision=32, threads=8) for w in several]
    for steps in (1, 4):
        batch.step(steps)
        for k, ref in enumerate(refs):
            ref.step(steps)
            assert_identical(batch.get_data(k), ref.get_data(), f"{names[k]} after {steps} more steps")
    batch.close()
