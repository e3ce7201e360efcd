"""The server's admission estimate beside the device memory that a simulation of the same world takes, after
steps and a read-back: cells only, cell radiation with and without splitting, mostly particles."""
import ctypes

import numpy as np
import pytest

from alien_amd import abi, engine, worlds
from alien_amd.abi import MOTION_FLUID

from . import helpers as H

pytestmark = pytest.mark.gpu

# allocations come in steps of 2 MiB: a set has its two arenas, its tables and the read-back's scratch, and a
# radiating one's particle arrays are 20 of their own once they have grown; the rest is the runtime's
SLACK = 64 << 20


def used():
    engine.lib()
    hip = ctypes.CDLL("libamdhip64.so.7")  # (the runtime that the engine has loaded)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return total.value - free.value


@pytest.mark.parametrize("n,np_,size,radiation,splitting", [(2_000_000, 0, (2000, 2000), False, False),
                                                            (400_000, 1000, (1000, 1000), True, False),
                                                            (250_000, 1000, (1000, 1000), True, True),
                                                            (1000, 1_500_000, (2000, 2000), False, False)])
def test_estimate_covers_a_simulation(n, np_, size, radiation, splitting):
    print("estimate", n, np_, radiation, splitting, flush=True)
    rng = np.random.default_rng(n)
    cells = worlds.free_cells(rng, size, n, vel_sigma=0.1)
    parts = worlds.particles(rng, size, np_, vel_sigma=0.1)
    cells["energy"] = rng.uniform(100, 200, n)
    worlds.assign_ids(cells, parts)
    params = H.params(MOTION_FLUID)
    for c in range(abi.MAX_COLORS):
        params.radiationCellAgeStrength[c] = 0.001 if radiation else 0.0
        params.highRadiationFactor[c] = 0.0
        if splitting:
            params.particleSplitEnergy[c] = 1.5
    world = worlds.World("estimate", size, params, cells, parts, 0, 3)
    server = engine.Server(budget_bytes=1 << 40, chunk_steps=8)
    estimate = server.poll(server.submit(size, params, cells, parts, 0, seed=3)).deviceBytes
    server.close()

    def run():
        before = used()
        sim = engine.Simulation.from_world(world)
        sim.step(6)
        sim.get_data()
        took = used() - before
        sim.close()
        return took

    run()  # (what the first use of the kernels and graphs leaves with the runtime)
    took = run()
    print("took", took, "estimate", estimate, flush=True)
    assert took <= estimate + SLACK
    assert estimate <= 1.3 * took + SLACK


def test_admission_counts_the_staging_of_mixed_sets():
    """A world without radiation takes staging slots too beside one that radiates: two jobs that fit the budget by
    their own estimates, but not in one set, run one after the other."""
    rng = np.random.default_rng(5)
    size = (800, 800)

    def job(n, radiation):
        cells = worlds.free_cells(rng, size, n, vel_sigma=0.1)
        cells["energy"] = 150
        params = H.params(MOTION_FLUID)
        for c in range(abi.MAX_COLORS):
            params.radiationCellAgeStrength[c] = 0.001 if radiation else 0.0
        return params, cells, np.zeros(0, dtype=abi.PARTICLE_DTYPE)

    big, small = job(300_000, False), job(10_000, True)
    probe = engine.Server(budget_bytes=1 << 40, chunk_steps=8)
    need = [probe.poll(probe.submit(size, *j, 0)).deviceBytes for j in (big, small)]
    probe.close()
    print("need", need, flush=True)
    server = engine.Server(budget_bytes=sum(need) + (2 << 20), chunk_steps=50)
    # (the first job leaves no room until it is done; the other two are queued by then)
    first = server.submit(size, *big, 20000)
    later = [server.submit(size, *j, 100) for j in (big, small)]
    for j in [first] + later:
        server.wait(j, timeout=100)
    one, two = (server.poll(j) for j in later)
    assert one.startTime >= server.poll(first).finishTime  # (both were queued while the first ran)
    assert two.startTime >= one.finishTime
    server.close()
