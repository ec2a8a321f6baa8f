"""sph_step_noalloc at the edges of its sizes against sph_step: one particle, a wave
and one more, and its largest particle count in its largest grid, one call after the
other on the same scratch array."""
import numpy as np
import pytest

from test_zz_no_alloc import CallerArrays, _hip_runtime, bits_equal, step_with_context, step_without_alloc

pytestmark = pytest.mark.gpu


def test_noalloc_sizes(hip):
    h = float(hip.scenes.H)
    arrays = CallerArrays(_hip_runtime(), hip._lib.NOALLOC_MAX_PARTICLES)
    rng = np.random.default_rng(3)
    try:
        # (n, cells an axis, steps): 64^3 cells are the most it takes
        for n, res, steps in ((65536, 64, 3), (65, 4, 4), (1, 1, 2), (64, 3, 1), (4097, 16, 5), (65536, 64, 2)):
            box = float(np.float32((res - 0.5) * h))
            pos = ((rng.random((n, 3)) - 0.5) * box).astype(np.float32)
            vel = rng.normal(0, 0.3, (n, 3)).astype(np.float32)
            ids = rng.permutation(n).astype(np.uint32)
            print("noalloc: %d particles, %d^3 cells, %d steps" % (n, res, steps), flush=True)
            ref = step_with_context(hip, box, pos, vel, ids, steps)
            got = step_without_alloc(hip, arrays, box, pos, vel, ids, steps)
            for a, b, what in zip(got, ref, ("positions", "velocities", "ids")):
                assert bits_equal(a, b), "%s differ" % what
    finally:
        arrays.free()
