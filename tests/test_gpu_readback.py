"""The read-back packed on the device: order by id (any 64-bit ids, equal ones by index), the
pass-through fields, counts around the workgroup, sort-tile and chunk sizes, against the oracle."""
import numpy as np
import pytest

from alien_amd import engine, worlds
from oracle.pyoracle import from_world

from . import helpers as H
from .test_gpu_parity import assert_identical

pytestmark = pytest.mark.gpu


def world(n, np_, ids, seed):
    """n free cells and np_ particles of any colour; ids 'wide' (random 64-bit), 'equal' (few values) or
    'plain' (ascending)."""
    rng = np.random.default_rng(seed)
    size = (128, 96)
    cells, parts = H.cells(n), H.particles(np_)
    cells["connections"]["cellIndex"] = 0
    for a, count in ((cells, n), (parts, np_)):
        a["pos"] = rng.uniform(0, 1, (count, 2)) * np.array(size)
        a["vel"] = rng.normal(0, 0.1, (count, 2))
        a["color"] = rng.integers(0, 7, count)
        a["selected"] = rng.integers(0, 2, count)
        if ids == "wide":
            a["id"] = rng.integers(0, 2**64, count, dtype=np.uint64)
        elif ids == "equal":
            a["id"] = rng.integers(5, 9, count)
    parts["energy"] = rng.uniform(0.5, 3.0, np_)
    cells["maxConnections"] = 0
    for f in ("creatureId", "mutationId", "age", "cellFunction", "ancestorMutationId"):
        cells[f] = rng.integers(0, 200, n)
    cells["genomeComplexity"] = rng.normal(0, 3, n)
    return worlds.World(f"readback_{n}_{np_}_{ids}", size, H.params(H.MOTION_FLUID, smoothingLength=0.65), cells, parts, 3,
                        seed)


@pytest.mark.parametrize("n,np_,ids", [(1, 1, "plain"), (255, 2048, "wide"), (256, 2049, "equal"), (257, 0, "equal"),
                                       (4096, 4097, "wide"), (4097, 300, "equal"), (0, 5000, "wide"), (20000, 9000, "plain"),
                                       (15421, 100, "wide")])
def test_order_and_fields(n, np_, ids):
    print("readback", n, np_, ids, flush=True)
    w = world(n, np_, ids, 11 + n + np_)
    sim, ref = engine.Simulation.from_world(w), from_world(w, precision=32)
    for steps in (0, 1, 2):  # before any step, then in two other internal orders
        sim.step(steps)
        ref.step(steps)
        assert_identical(sim.get_data(), ref.get_data(), f"{w.name} after {steps} more")
    assert sim.counts() == ref.counts()
    sim.close()
