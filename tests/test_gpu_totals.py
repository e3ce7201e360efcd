"""The totals of a world, read without its other state, beside the sums over what get_data gives: particles
killed in the last step, halves split off in it and emitted ones included, and worlds of one kind only."""
import numpy as np
import pytest

from alien_amd import abi, engine, worlds
from alien_amd.abi import MOTION_COLLISION, MOTION_FLUID

from . import helpers as H

pytestmark = pytest.mark.gpu


def sums(cells, parts):
    v = cells["vel"].astype(np.float64)
    return {"cellEnergy": cells["energy"].astype(np.float64).sum(), "particleEnergy": parts["energy"].astype(np.float64).sum(),
            "momentum": v.sum(0), "kinetic": 0.5 * (v * v).sum()}


@pytest.mark.parametrize("n,np_,motion", [(0, 3000, MOTION_FLUID), (5000, 0, MOTION_COLLISION), (9000, 4000, MOTION_FLUID),
                                          (300000, 70000, MOTION_FLUID), (1, 1, MOTION_COLLISION)])
def test_totals(n, np_, motion):
    print("totals", n, np_, motion, flush=True)
    rng = np.random.default_rng(n + np_)
    size = (900, 700) if n > 100000 else (160, 128)
    cells = worlds.free_cells(rng, size, n, vel_sigma=0.3)
    parts = worlds.particles(rng, size, np_, vel_sigma=0.3)
    cells["energy"] = rng.uniform(10, 200, n)
    worlds.assign_ids(cells, parts)
    params = H.params(motion)
    if motion == MOTION_FLUID:
        for c in range(abi.MAX_COLORS):
            params.particleSplitEnergy[c] = 1.5
            params.radiationCellAgeStrength[c] = 0.001
    sim = engine.Simulation.from_world(worlds.World("totals", size, params, cells, parts, 0, 9))
    for steps in (0, 1, 6):
        sim.step(steps)
        c, p = sim.get_data()
        t, want = sim.totals(), sums(c, p)
        assert (t["numCells"], t["numParticles"]) == (len(c), len(p))
        # (sums of n doubles in another order: n roundings of the sum of the magnitudes at most)
        bound = 2.0 ** -53 * max(1, len(c) + len(p))
        assert abs(t["cellEnergy"] - want["cellEnergy"]) <= bound * want["cellEnergy"]
        assert abs(t["particleEnergy"] - want["particleEnergy"]) <= bound * want["particleEnergy"]
        assert abs(t["kinetic"] - want["kinetic"]) <= 4 * bound * want["kinetic"]
        for k in range(2):
            assert abs(t["momentum"][k] - want["momentum"][k]) <= bound * np.abs(c["vel"][:, k].astype(np.float64)).sum()
    sim.close()
