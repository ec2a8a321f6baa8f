"""Crowded launches of up to 40,960 slots, which leave the passes that share a particle
between lanes: on both sides of the lines (a cell of more than 64 particles; cells of
800,000 slots together, counted for every particle), in both orders and in every grid
phase. Bit-exact against the oracle."""
import numpy as np
import pytest

from test_gpu_parity import assert_bits_equal
from test_zz_no_alloc import CallerArrays, _hip_runtime, bits_equal, step_with_context, step_without_alloc

pytestmark = pytest.mark.gpu


def filled_cells(h, res, sizes, box, rng):
    """sizes[c] particles in the middle of cell c of a res^3 grid, visited along x first."""
    c = np.repeat(np.arange(len(sizes)), sizes)
    cell = np.stack([c % res, c // res % res, c // (res * res)], 1)
    return ((cell + 0.5 + 0.4 * rng.uniform(-1, 1, (len(c), 3))) * h - box / 2).astype(np.float32)


def one_step(hip, orc, res, pos, reference, fused):
    h = float(hip.scenes.H)
    box = float(np.float32((res - 0.25) * h))
    rng = np.random.default_rng(len(pos))
    pos = np.ascontiguousarray(pos[rng.permutation(len(pos))])
    vel = rng.normal(0, 0.3, pos.shape).astype(np.float32)
    o = orc.OracleSim(box, len(pos))
    o.add_particles(pos, vel)
    o.set_order_mode(orc.ORDER_REFERENCE if reference else orc.ORDER_CANONICAL)
    o.step(1)
    want = o.state()
    assert np.isfinite(want["vel"]).all()
    flags = hip._lib.FLAG_REFERENCE_ORDER if reference else 0
    with hip.HIPGridParticleSimulator(box, capacity=len(pos) + 9, flags=flags, fused=fused) as sim:
        sim.upload(pos, vel)
        sim.step()
        p, v, _ = sim.download()
    assert_bits_equal(p, want["pos"], "positions")
    assert_bits_equal(v, want["vel"], "velocities")


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("reference", [False, True])
@pytest.mark.parametrize("sizes", [[64], [65], [30, 64, 20, 65, 1], [64] * 40, [300, 2], [20] * 2000, [20] * 1999 + [21]])
def test_one_step(hip, orc, sizes, reference, fused):
    res = 13
    print("%d cells of up to %d, reference order %s, fused %s" % (len(sizes), max(sizes), reference, fused), flush=True)
    box = float(np.float32((res - 0.25) * float(hip.scenes.H)))
    pos = filled_cells(float(hip.scenes.H), res, sizes, box, np.random.default_rng(len(sizes)))
    one_step(hip, orc, res, pos, reference, fused)


@pytest.mark.parametrize("most", [64, 65])
def test_sparse_grid(hip, orc, most):
    """Sorted by digits (8.6 million cells)."""
    res = 205
    box = float(np.float32((res - 0.25) * float(hip.scenes.H)))
    pos = filled_cells(float(hip.scenes.H), res, [10, most, 3], box, np.random.default_rng(most))
    one_step(hip, orc, res, pos, False, True)


def test_noalloc(hip):
    """sph_step_noalloc, with a scene that is crowded between two that are not."""
    h = float(hip.scenes.H)
    res, box = 13, float(np.float32(12.75 * h))
    rng = np.random.default_rng(8)
    arrays = CallerArrays(_hip_runtime(), hip._lib.NOALLOC_MAX_PARTICLES)
    try:
        for sizes in ([20] * 100, [200, 30, 70], [64, 64]):
            pos = filled_cells(h, res, sizes, box, rng)
            vel = rng.normal(0, 0.3, pos.shape).astype(np.float32)
            ids = rng.permutation(len(pos)).astype(np.uint32)
            ref = step_with_context(hip, box, pos, vel, ids, 3)
            got = step_without_alloc(hip, arrays, box, pos, vel, ids, 3)
            for a, b, what in zip(got, ref, ("positions", "velocities", "ids")):
                assert bits_equal(a, b), "%s differ" % what
    finally:
        arrays.free()


def test_a_crowded_scene_is_no_slower_than_a_wide_one(hip):
    """40,000 particles at spacing h/5 in a scene of as many slots, against a scene of more
    than 65,536, which has one lane a particle whatever is in it (2.4 times as long when the
    particles were shared all the same)."""
    h = float(hip.scenes.H)
    n, side = 40000, 35
    rng = np.random.default_rng(5)
    g = np.arange(side) * (h / 5)
    pos = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)[:n]
    pos = (pos - 0.3 + rng.uniform(-0.02 * h, 0.02 * h, pos.shape)).astype(np.float32)
    ms = []
    for capacity in (n, 70000):
        with hip.HIPGridParticleSimulator(0.7, capacity=capacity) as sim:
            t = []
            for _ in range(6):
                sim.upload(pos)
                t.append(sim.advance(1))
            ms.append(min(t[1:]))
    print("%d slots %.3f ms, 70,000 slots %.3f ms" % (n, *ms), flush=True)
    assert ms[0] < 1.25 * ms[1]
