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
