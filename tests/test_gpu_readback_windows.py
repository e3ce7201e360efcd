"""The read-back beyond the windows its sums are carried over: more than 256 sort tiles (1,048,576 keys) and
1024 particle tiles (2,097,152 entries), in several pinned chunks, beside the input sorted by id (stable)."""
import numpy as np
import pytest

from alien_amd import engine

from .test_gpu_readback import world

pytestmark = pytest.mark.gpu

CELL_FIELDS = ("id", "pos", "vel", "energy", "color", "creatureId", "mutationId", "age", "cellFunction",
               "ancestorMutationId", "genomeComplexity", "selected")
PARTICLE_FIELDS = ("id", "pos", "vel", "energy", "color", "selected")


@pytest.mark.parametrize("n,np_,ids", [(1_200_000, 2_150_000, "wide"), (1_200_000, 1_300_000, "equal"),
                                       (1_048_577, 2_097_153, "wide")])
def test_order_beyond_the_windows(n, np_, ids):
    print("readback windows", n, np_, ids, flush=True)
    w = world(n, np_, ids, 5 + n + np_)
    sim = engine.Simulation.from_world(w)
    for got, given, fields in zip(sim.get_data(), (w.cells, w.particles), (CELL_FIELDS, PARTICLE_FIELDS)):
        want = given[np.argsort(given["id"], kind="stable")].copy()
        # (positions come back wrapped; the upper edge, which a draw may be rounded to, is 0)
        want["pos"][want["pos"] == np.array(w.size, dtype=np.float32)] = 0
        assert len(got) == len(want)
        for f in fields:
            assert np.array_equal(got[f], want[f]), f
    sim.close()
