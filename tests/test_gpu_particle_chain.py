"""The particles' chain of sets with bond work at either of its places in the step (a launch later without
readers of the energies that absorption changes), and worlds whose parameters move it, at every workgroup
size, against the oracle."""
import pytest

from alien_amd import engine
from alien_amd.abi import MOTION_COLLISION, MOTION_FLUID
from oracle.pyoracle import from_world

from . import helpers as H
from .test_gpu_bond_phase import world
from .test_gpu_parity import assert_identical

pytestmark = pytest.mark.gpu

LIMITS = (float("inf"), 101.0, float("inf"))


@pytest.mark.parametrize("motion", [MOTION_FLUID, MOTION_COLLISION])
def test_chain_moves_with_the_parameters(motion):
    print("particle chain", motion, flush=True)
    w = world(motion, 90 + motion)
    w.params.cellMaxBindingEnergy = LIMITS[0]
    sim, ref = engine.Simulation.from_world(w), from_world(w, precision=32)
    for k, limit in enumerate(LIMITS):
        if k:
            p = H.params(motion, smoothingLength=0.65, innerFriction=0.3, cellMaxBindingEnergy=limit)
            sim.set_params(p)
            ref.set_params(p)
        for steps in (1, 4):
            sim.step(steps)
            ref.step(steps)
            assert_identical(sim.get_data(), ref.get_data(), f"limit {limit} ({k}) after {steps} more steps")
    sim.close()


@pytest.mark.parametrize("threads", [64, 128, 192, 256])
def test_late_chain_in_a_batch(threads):
    print("late particle chain", threads, flush=True)
    ws = [world(MOTION_COLLISION, 60 + threads), world(MOTION_FLUID, 61 + threads), world(MOTION_FLUID, 62 + threads, bonds=False)]
    for w in ws:
        w.params.cellMaxBindingEnergy = float("inf")
    refs = [from_world(w, precision=32) for w in ws]
    batch = engine.Batch()
    batch.set_block_size(threads)
    for w in ws:
        batch.add(w)
    for steps in (1, 3, 5):
        batch.step(steps)
        for k, ref in enumerate(refs):
            ref.step(steps)
            assert_identical(batch.get_data(k), ref.get_data(), f"world {k} threads {threads} after {steps} more steps")
    batch.close()
