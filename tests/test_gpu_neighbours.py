"""The neighbour passes where their parts change: launches on both sides of the rule
that shares particles between lanes (40,960 slots), sizes around a wave's 16 or 64
particles, and clusters of particles that all see each other, at the edges of what
the passes hand to each other (288 entries; 512 candidates of a row) and of the
lists in LDS. Bit-exact against the oracle, one step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SPLIT = 40960   # slots


def cluster(n, rng):
    """n particles within a cube whose diagonal is shorter than h."""
    return (0.02 * rng.random((n, 3))).astype(np.float32)


@pytest.mark.parametrize("reference", [False, True])
@pytest.mark.parametrize("capacity,crowd,sparse", [
    (1, 1, 0), (2, 2, 0), (15, 3, 12), (16, 8, 8), (17, 1, 16), (63, 33, 30), (65, 32, 33), (SPLIT, 25, 3000),
    (289, 289, 0), (290, 290, 0), (1400, 700, 700),
    (SPLIT + 1, 25, 3000), (SPLIT + 64, 510, 1), (SPLIT + 64, 512, 67), (SPLIT + 64, 514, 63),
])
def test_one_step(hip, orc, capacity, crowd, sparse, reference):
    box = 0.4
    rng = np.random.default_rng([capacity, crowd, sparse])
    loose = (box * (rng.random((sparse, 3)) - 0.5)).astype(np.float32)
    pos = np.concatenate([cluster(crowd, rng), loose])
    pos = np.ascontiguousarray(pos[rng.permutation(len(pos))])
    vel = rng.normal(0, 0.5, pos.shape).astype(np.float32)
    print("capacity %d, %d crowded, %d loose, reference order %s" % (capacity, crowd, sparse, reference), flush=True)
    o = orc.OracleSim(box, len(pos))
    o.add_particles(pos, vel)
    o.set_order_mode(orc.ORDER_REFERENCE if reference else orc.ORDER_CANONICAL)
    sim = hip.HIPGridParticleSimulator(box, flags=hip._lib.FLAG_REFERENCE_ORDER if reference else 0,
                                       capacity=capacity)
    sim.upload(pos, vel)
    sim.advance(1)
    o.step(1)
    st = o.state()
    p, v, _ = sim.download(by_id=True)
    assert np.isfinite(st["vel"]).all()
    assert np.array_equal(p.view(np.uint32), np.asarray(st["pos"], np.float32).view(np.uint32))
    assert np.array_equal(v.view(np.uint32), np.asarray(st["vel"], np.float32).view(np.uint32))
    sim.close()
