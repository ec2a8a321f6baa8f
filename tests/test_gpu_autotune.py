"""What the autotuner leaves behind: the state as a step left it, and a variant chosen for
a reason."""
import numpy as np
import pytest

from test_gpu_parity import assert_bits_equal

pytestmark = pytest.mark.gpu


def test_the_next_step_starts_as_before(hip):
    """The step after the autotuner needs no new hash of the positions (the step before it
    wrote the keys), and its grid phase sorts them as if nothing had been in between."""
    lib = hip._lib
    pos = hip.scenes.lattice(16, 16, 16, 0.4, jitter_h=0.01, seed=4)
    a = hip.HIPGridParticleSimulator(0.4, capacity=len(pos) + 77, flags=lib.FLAG_PROFILE)
    b = hip.HIPGridParticleSimulator(0.4, capacity=len(pos) + 77)
    for sim in (a, b):
        sim.upload(pos)
        sim.advance(3)
    lib.check(a._lib.sph_autotune(a._ctx, 2, None))
    a.stage_times(reset=True)
    for sim in (a, b):
        sim.updateGrid()
    assert a.stage_times()["hash"][1] == 0
    for kind in (lib.DEBUG_CELL_PRESORT, lib.DEBUG_PERM, lib.DEBUG_CELL, lib.DEBUG_CELL_START, lib.DEBUG_IDS):
        np.testing.assert_array_equal(a.debug(kind), b.debug(kind))
    for sim in (a, b):
        for phase in (sim.updateDensityPressure, sim.updateForces, sim.updateCollisions, sim.integrate):
            phase()
        sim.advance(4)
    assert_bits_equal(a.download()[0], b.download()[0], "positions after the autotuner")
    a.close()
    b.close()


@pytest.mark.parametrize("variant", [3, 12])
def test_one_shape_keeps_the_variant(hip, variant):
    """Up to 40,960 slots the mask mode has one kernel for all variants: one time stands
    for all, and where it wins the variant stays what it was."""
    lib = hip._lib
    pos = hip.scenes.lattice(12, 12, 12, 0.4, jitter_h=0.01, seed=4)
    with hip.SceneBatch([(0.4, len(pos))]) as b:
        b.upload(0, pos)
        b.set_variant(variant, lib.NEIGHBOURS_MASKS)
        b.step(2)
        times = b.autotune(steps=2)
        masks = [times[(v, lib.NEIGHBOURS_MASKS)] for v in range(lib.NUM_VARIANTS)]
        assert len(set(masks)) == 1
        chosen, mode = b.variant()
        if mode == lib.NEIGHBOURS_MASKS:
            assert chosen == variant
        else:
            assert times[(chosen, mode)] < masks[0]
