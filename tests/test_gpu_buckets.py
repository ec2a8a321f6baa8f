"""The reference order's buckets where their scan changes: buckets of up to 64 entries
(one wave) and more (one workgroup, 1,024 entries at a time), with stayers, movers and
early arrivals in all of them. Against the oracle's buckets after every grid phase."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box,n", [(0.04, 70), (0.08, 63), (0.08, 64), (0.08, 65), (0.08, 520), (0.08, 9000),
                                   (0.13, 1700), (0.13, 12000), (0.4, 1023), (0.4, 1024), (0.4, 1025), (0.4, 8200)])
def test_buckets_over_grid_phases(hip, orc, box, n):
    rng = np.random.default_rng([n, int(box * 100)])
    pos = (box * (rng.random((n, 3)) - 0.5)).astype(np.float32)
    vel = rng.normal(0, 4, (n, 3)).astype(np.float32)
    print("box %g, %d particles" % (box, n), flush=True)
    sim = hip.HIPGridParticleSimulator(box, flags=hip._lib.FLAG_REFERENCE_ORDER, capacity=n + 100)
    sim.upload(pos, vel)
    o = orc.OracleSim(box, n)
    o.add_particles(pos, vel)
    o.set_order_mode(orc.ORDER_REFERENCE)
    for step in range(4):
        sim.updateGrid()
        o.update_grid()
        rx, ry, rz = o.grid_dims
        start, ids = o.buckets()
        cells = np.arange(rx * ry * rz).reshape(rz, ry, rx).transpose(2, 1, 0).ravel()   # x outer, z inner
        want = np.concatenate([ids[start[c]:start[c + 1]] for c in cells])
        np.testing.assert_array_equal(sim.debug(hip._lib.DEBUG_IDS), want, err_msg="grid phase %d" % step)
        sim.updateDensityPressure()
        sim.updateForces()
        sim.updateCollisions()
        sim.integrate()
        o.update_density_pressure()
        o.update_forces()
        o.integrate()
        assert np.isfinite(o.state()["pos"]).all()
    sim.close()
