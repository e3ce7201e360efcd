"""The neighbour passes where a wave's candidates do not fit its stage, its lists are long, or its pairs go
through several rounds of records: dense worlds, wide reach, crowds next to empty space; with the counts of
the waves and cells that took the slower paths, against the oracle."""
import numpy as np
import pytest

from alien_amd import engine, worlds
from alien_amd.abi import MOTION_COLLISION, MOTION_FLUID
from oracle.pyoracle import from_world

from . import helpers as H
from .test_gpu_parity import assert_identical

pytestmark = pytest.mark.gpu

# name: size, free cells, reach (fluid: twice the smoothing length), crowds (x, y, width, height, cells),
# whether every wave fits, none does, some do, or either (small sets have short waves)
CASES = {
    "sparse": ((96, 80), 1200, 1.3, (), "all"),
    "pairs in several rounds": ((64, 64), 8000, 1.3, (), "any"),
    "long lists": ((64, 60), 3800, 4.0, (), "none"),
    "wide reach": ((101, 97), 1000, 16.0, (), "none"),
    "drops": ((160, 128), 900, 1.3, tuple((9 + 19 * k, 11 + 17 * (k * 5 % 7), 7, 7, 160) for k in range(7)), "some"),
    "a full row of bins": ((90, 84), 300, 1.3, ((20, 40, 2, 2, 400), (22, 42, 2, 2, 90)), "some"),
    "one crowd among few cells": ((2000, 40), 500, 1.3, ((1000, 20, 30, 6, 500),), "any"),
}


def world(name, motion, bonds):
    size, n, reach, crowds, _ = CASES[name]
    rng = np.random.default_rng(n + motion)
    pos = [rng.uniform(0, 1, (n, 2)) * np.array(size)]
    for x, y, w, h, cnt in crowds:
        pos.append(np.array([x, y]) + rng.uniform(0, 1, (cnt, 2)) * np.array([w, h]))
    pos = np.concatenate(pos)[rng.permutation(n + sum(c[4] for c in crowds))]
    cells = H.cells(len(pos))
    cells["connections"]["cellIndex"] = 0
    cells["pos"] = np.minimum(pos.astype(np.float32), np.nextafter(np.float32(size), np.float32(0)))
    cells["vel"] = rng.normal(0, 0.1, pos.shape)
    cells["color"] = rng.integers(0, 7, len(pos))
    cells["maxConnections"] = 0
    if bonds:  # (few cells can fuse: at most four candidate pairs a cell fit the list)
        cells["maxConnections"][rng.choice(len(pos), len(pos) // 20, replace=False)] = 3
        cells["barrier"][rng.choice(len(pos), len(pos) // 30, replace=False)] = 1
    parts = H.particles(0)
    worlds.assign_ids(cells, parts)
    return worlds.World(name, size, H.params(motion, smoothingLength=reach / 2, cellMaxCollisionDistance=reach), cells, parts,
                        5, 3)


@pytest.mark.parametrize("motion,bonds", [(MOTION_FLUID, False), (MOTION_FLUID, True), (MOTION_COLLISION, True)])
@pytest.mark.parametrize("name", list(CASES))
def test_crowded_waves(name, motion, bonds):
    print("crowded waves", name, motion, bonds, flush=True)
    w = world(name, motion, bonds)
    sim, ref = engine.Simulation.from_world(w), from_world(w, precision=32, threads=8)
    for steps in (1, 2):
        sim.step(steps)
        ref.step(steps)
        assert_identical(sim.get_data(), ref.get_data(), f"{name} after {steps} more steps")
    waves, cells = sim.path_counts()
    fits = CASES[name][4]
    if fits == "all":
        assert (waves, cells) == (0, 0)
    elif fits != "any":
        assert waves > 0 and cells > 0
        assert fits == "some" or cells > len(w.cells)  # (most, in three steps)
    assert cells <= 3 * len(w.cells)
    sim.close()
