"""The row masks' kernels, one lane a particle: a scene of more than 65,536 slots keeps
them, however few of its slots are in use. Bit-exact against the oracle."""
import numpy as np
import pytest

from test_gpu_parity import assert_bits_equal

pytestmark = pytest.mark.gpu

CAPACITY = 65_600   # slots: too many for passes that share a particle between lanes


def edge_clusters(h, sizes, rng):
    """Clusters of the given sizes in the four rows of cells around a cell edge along x, in the
    rows' order, all of their particles within h of each other."""
    edge = np.array([0.5, 1.0, 1.0]) * h
    side = [(-1, -1), (1, -1), (-1, 1), (1, 1)]   # (y, z)
    parts = []
    for n, (sy, sz) in zip(sizes, side):
        d = 0.001 + 0.01 * rng.random((n, 3))     # (diagonal of the four: 0.038)
        parts.append(edge + d * np.array([1.0, sy, sz]))
    return np.concatenate(parts).astype(np.float32)


@pytest.mark.parametrize("sizes", [(512, 512, 0, 40), (512, 512, 64, 3), (512, 511, 0, 64), (500, 512, 512, 30),
                                   (512, 513, 20, 0)])
def test_full_rows(hip, orc, sizes):
    """Rows of 512 accepted candidates one after the other: as many pairs as a queue of 32
    words can hold, seen from particles of a third row in waves of their own."""
    box = 0.4
    rng = np.random.default_rng(list(sizes))
    corner = -np.float32(box) / 2
    pos = (edge_clusters(float(hip.scenes.H), sizes, rng) + corner).astype(np.float32)
    vel = rng.normal(0, 0.5, pos.shape).astype(np.float32)
    o = orc.OracleSim(box, len(pos))
    o.add_particles(pos, vel)
    o.set_order_mode(orc.ORDER_CANONICAL)
    o.step(1)
    want = o.state()
    assert np.isfinite(want["vel"]).all()
    for v in range(hip._lib.NUM_VARIANTS):
        print("rows of %s, variant %d" % (sizes, v), flush=True)
        with hip.SceneBatch([(box, CAPACITY)]) as b:
            b.upload(0, pos, vel)
            b.set_variant(v, hip._lib.NEIGHBOURS_MASKS)
            b.step(1)
            p, w, _ = b.download(0)
        assert_bits_equal(p, want["pos"], "variant %d positions" % v)
        assert_bits_equal(w, want["vel"], "variant %d velocities" % v)


def lattice_block(h, side, spacing, rng):
    """side^3 sites `spacing` apart, jittered by 0.01 h, from the corner of a 0.4 m box."""
    g = np.arange(side) * spacing - 0.15
    pos = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    return (pos + rng.uniform(-0.01 * h, 0.01 * h, pos.shape)).astype(np.float32)


@pytest.mark.parametrize("reference", [False, True])
@pytest.mark.parametrize("scene,steps", [("loose", 8), ("six words a row", 3), ("twelve words a row", 2),
                                         ("rows too long", 2)])
def test_variants_on_the_masks(hip, orc, scene, steps, reference):
    """Every variant where the queues drain once, several times and not at all (rows of more
    than 512 candidates are walked); the phases and the accelerations with the default one.
    The reference order is compiled in one shape."""
    lib = hip._lib
    h = float(hip.scenes.H)
    rng = np.random.default_rng(31)
    if scene == "loose":
        pos = hip.scenes.lattice(15, 16, 17, 0.4, jitter_h=0.01, seed=3)
    elif scene == "rows too long":
        pos = (rng.random((3000, 3)) * 0.09 - 0.2).astype(np.float32)
    else:
        pos = lattice_block(h, 16 if scene == "six words a row" else 15, h / (4 if scene == "six words a row" else 5), rng)
    vel = rng.normal(0, 0.3, pos.shape).astype(np.float32)
    flags = lib.FLAG_REFERENCE_ORDER if reference else 0
    o = orc.OracleSim(0.4, len(pos))
    o.add_particles(pos, vel)
    o.set_order_mode(orc.ORDER_REFERENCE if reference else orc.ORDER_CANONICAL)
    o.step(steps)
    want = o.state()
    assert np.isfinite(want["vel"]).all()
    for v in [12] if reference else range(lib.NUM_VARIANTS):
        print("%s, reference order %s, variant %d" % (scene, reference, v), flush=True)
        with hip.HIPGridParticleSimulator(0.4, capacity=CAPACITY, flags=flags) as sim:
            sim.upload(pos, vel)
            lib.check(sim._lib.sph_set_variant(sim._ctx, v, lib.NEIGHBOURS_MASKS))
            sim.advance(steps)
            p, w, _ = sim.download()
        assert_bits_equal(p, want["pos"], "variant %d positions" % v)
        assert_bits_equal(w, want["vel"], "variant %d velocities" % v)
    for fused in (True, False):
        with hip.HIPGridParticleSimulator(0.4, capacity=CAPACITY, flags=flags | lib.FLAG_DIAGNOSTICS, fused=fused) as sim:
            sim.upload(pos, vel)
            for _ in range(steps):
                sim.step()
            p, w, _ = sim.download()
            ids = sim.debug(lib.DEBUG_IDS)
            assert_bits_equal(sim.debug(lib.DEBUG_DENSITY), want["density"][ids], "density, fused %s" % fused)
            if fused:   # the phases' acceleration is the forces' alone until the walls' are added
                assert_bits_equal(sim.debug(lib.DEBUG_ACCEL), want["acc"][ids], "acceleration")
        assert_bits_equal(p, want["pos"], "positions, fused %s" % fused)
        assert_bits_equal(w, want["vel"], "velocities, fused %s" % fused)
