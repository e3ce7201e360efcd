"""The map of cells that move further than a bin: all cells of a world, beside more near movers than a
group's list takes, and so many into one bin that waves of their own place them; against the oracle."""
import numpy as np
import pytest

from alien_amd import engine, worlds
from alien_amd.abi import MOTION_COLLISION, MOTION_FLUID
from oracle.pyoracle import from_world

from . import helpers as H
from .test_gpu_parity import assert_identical

pytestmark = pytest.mark.gpu

# name: size, cells, speed, crowds (x, y, side, cells, velocity); bins are two units wide
CASES = {
    "all far": ((300, 200), 9000, 9.0, ()),
    "far and many near": ((128, 128), 14000, 2.5, ()),
    "into one bin": ((150, 90), 3000, 1.5, ((20, 40, 2, 15, 10), (60, 40, 2, 40, 10), (100, 40, 2, 150, 10))),
    "across the edge": ((64, 70), 1500, 1.0, ((60, 20, 2, 30, 6), (62, 44, 2, 100, 6))),
}


@pytest.mark.parametrize("motion", [MOTION_FLUID, MOTION_COLLISION])
@pytest.mark.parametrize("name", list(CASES))
def test_far_movers(name, motion):
    print("far movers", name, motion, flush=True)
    size, n, speed, crowds = CASES[name]
    rng = np.random.default_rng(n + motion)
    pos, vel = [rng.uniform(0, 1, (n, 2)) * np.array(size)], [rng.normal(0, speed, (n, 2))]
    for x, y, side, cnt, v in crowds:
        pos.append(np.array([x, y]) + rng.uniform(0, side, (cnt, 2)))
        vel.append(np.tile([float(v), 0.0], (cnt, 1)))
        # and some where the crowd goes, which stay or come from the bins around
        pos.append((np.array([x + v, y]) + rng.uniform(-1, side + 1, (12, 2))) % np.array(size))
        vel.append(rng.normal(0, 0.4, (12, 2)))
    pos, vel = np.concatenate(pos), np.concatenate(vel)
    order = rng.permutation(len(pos))
    cells = H.cells(len(pos))
    cells["connections"]["cellIndex"] = 0
    cells["pos"] = np.minimum(pos[order].astype(np.float32), np.nextafter(np.float32(size), np.float32(0)))
    cells["vel"] = vel[order]
    cells["maxConnections"] = 0
    parts = H.particles(0)
    worlds.assign_ids(cells, parts)
    w = worlds.World(name, size, H.params(motion, cellMaxVelocity=20.0), cells, parts, 5, 3)
    sim, ref = engine.Simulation.from_world(w), from_world(w, precision=32, threads=8)
    for steps in (1, 1, 3):
        sim.step(steps)
        ref.step(steps)
        assert_identical(sim.get_data(), ref.get_data(), f"{name} after {steps} more steps")
    sim.close()


# worlds of many cells to a bin, whose map's waves take 64 and 16 bins: cells per bin, bin edge, speed
@pytest.mark.parametrize("motion", [MOTION_FLUID, MOTION_COLLISION])
@pytest.mark.parametrize("size,per_bin,edge,speed", [((70, 66), 4, 2, 0.5), ((70, 66), 4, 2, 6.0), ((64, 512), 5, 2, 1.0),
                                                     ((40, 42), 12, 2, 0.5), ((40, 42), 12, 2, 5.0), ((61, 57), 25, 3, 2.0),
                                                     ((9, 300), 9, 3, 3.0), ((300, 9), 9, 3, 3.0), ((33, 35), 70, 3, 4.0)])
def test_dense_maps(size, per_bin, edge, speed, motion):
    print("dense map", size, per_bin, edge, speed, motion, flush=True)
    n = per_bin * (size[0] // edge) * (size[1] // edge)
    rng = np.random.default_rng(n + motion)
    cells = H.cells(n)
    cells["connections"]["cellIndex"] = 0
    cells["pos"] = np.minimum((rng.uniform(0, 1, (n, 2)) * np.array(size)).astype(np.float32),
                              np.nextafter(np.float32(size), np.float32(0)))
    cells["vel"] = rng.normal(0, speed, (n, 2))
    cells["maxConnections"] = 0
    parts = H.particles(0)
    worlds.assign_ids(cells, parts)
    w = worlds.World("dense", size, H.params(motion, cellMaxVelocity=15.0, smoothingLength=edge / 2 - 0.1,
                                             cellMaxCollisionDistance=edge - 0.2), cells, parts, 5, 3)
    sim, ref = engine.Simulation.from_world(w), from_world(w, precision=32, threads=8)
    for steps in (1, 1, 2):
        sim.step(steps)
        ref.step(steps)
        assert_identical(sim.get_data(), ref.get_data(), f"{size} {per_bin} after {steps} more steps")
    sim.get_map()  # (enters every cell anew)
    sim.step(1)
    ref.step(1)
    assert_identical(sim.get_data(), ref.get_data(), f"{size} {per_bin} after introspection")
    sim.close()
