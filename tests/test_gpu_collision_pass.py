"""The collision neighbour pass where it splits its work: worlds of three bins a side and more, the torus'
edges (collisions do not reach across them), wide reaches, bodies with more pairs than a wave has records,
barriers among the bonded, crowds that walk alone, against the oracle."""
import numpy as np
import pytest

from alien_amd import engine, worlds
from alien_amd.abi import MOTION_COLLISION
from oracle.pyoracle import from_world

from . import helpers as H
from .test_gpu_parity import assert_identical

pytestmark = pytest.mark.gpu

# name: size, free cells, reach, bodies (x, y, columns, rows, spacing), crowds (x, y, width, height, cells)
CASES = {
    "three bins": ((7, 6), 40, 2.0, (), ()),
    "four bins": ((8, 9), 50, 1.9, (), ()),
    "three-unit bins": ((140, 101), 5000, 2.7, (), ()),
    "edges": ((90, 80), 400, 1.3, ((86.4, 20.0, 8, 20, 0.9), (30.0, 76.5, 20, 6, 0.9)), ()),
    "bodies": ((300, 200), 3000, 1.3, ((20.0, 20.0, 60, 40, 0.55), (120.0, 50.0, 100, 90, 0.9)), ()),
    "pushed together": ((120, 100), 200, 1.3, ((30.0, 30.0, 70, 60, 0.25),), ()),
    "crowds": ((160, 100), 500, 1.3, (), ((40, 40, 6, 6, 400), (0, 20, 2, 2, 90), (158, 20, 2, 2, 30))),
    "64 cells a wave": ((420, 400), 70000, 1.3, ((100.0, 100.0, 120, 100, 0.8),), ()),
    "32 cells a wave": ((420, 400), 20000, 1.3, ((100.0, 100.0, 100, 60, 0.8),), ()),
}


def world(name):
    size, free, reach, bodies, crowds = CASES[name]
    rng = np.random.default_rng(len(name) + free)
    pos = [rng.uniform(0, 1, (free, 2)) * size]
    for x, y, w, h, n in crowds:
        pos.append(np.array([x, y]) + rng.uniform(0, 1, (n, 2)) * [w, h])
    links = []
    for x, y, nx, ny, d in bodies:
        base = sum(len(p) for p in pos)
        gx, gy = np.meshgrid(np.arange(nx), np.arange(ny))
        pos.append(np.stack([x + d * gx, y + d * gy], -1).reshape(-1, 2) + rng.uniform(-0.02, 0.02, (nx * ny, 2)))
        index = base + np.arange(nx * ny).reshape(ny, nx)
        links += [(a, b, d) for a, b in zip(index[:, :-1].ravel(), index[:, 1:].ravel())]
    pos = np.concatenate(pos) % np.array(size)
    c = H.cells(len(pos))
    c["connections"]["cellIndex"] = 0
    c["pos"] = np.minimum(pos.astype(np.float32), np.nextafter(np.float32(size), np.float32(0)))
    c["vel"] = rng.normal(0, 0.3, pos.shape)
    # (a step takes four fusion candidates per cell at most: the densest body has no free bond slots)
    c["maxConnections"] = 2 if name == "pushed together" else rng.integers(2, 7, len(pos))
    for a, b, d in links:
        for s, t in ((a, b), (b, a)):
            k = c["numConnections"][s]
            c["connections"][s, k] = (t, d, 180.0)
            c["numConnections"][s] = k + 1
    ends = c["numConnections"] == 1
    c["connections"]["angleFromPrevious"][ends, 0] = 360.0
    c["barrier"][rng.choice(len(pos), len(pos) // 40, replace=False)] = 1
    parts = H.particles(0)
    worlds.assign_ids(c, parts)
    return worlds.World(name, size, H.params(MOTION_COLLISION, cellMaxCollisionDistance=reach, cellFusionVelocity=0.5), c, parts, 5, 3)


@pytest.mark.parametrize("name", list(CASES))
def test_collision_pass(name):
    print("collision pass", name, flush=True)
    w = world(name)
    sim, ref = engine.Simulation.from_world(w), from_world(w, precision=32, threads=8)
    for steps in (1, 1, 4):
        sim.step(steps)
        ref.step(steps)
        assert_identical(sim.get_data(), ref.get_data(), f"{name} after {steps} more steps")
    sim.close()
