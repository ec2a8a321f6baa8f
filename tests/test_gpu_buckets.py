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


@pytest.mark.parametrize("res,part,n", [
    (28, 1.0, 3000), (28, 0.25, 9000), (28, 0.18, 9000),    # up to 32 entries a cell, about 32, and over 64
    (28, 0.05, 33), (29, 0.001, 16), (101, 0.2, 70000),
    (407, 0.02, 5000),                                      # 67 million cells: more than 2^32 / 64
])
def test_buckets_of_large_grids(hip, orc, res, part, n):
    """Grids where a lane takes a bucket of up to 32 entries; the particles fill `part` of each
    edge of the box, around its middle."""
    h = float(hip.scenes.H)
    box = float(np.float32((res - 0.5) * h))
    rng = np.random.default_rng([res, n])
    pos = (part * box * (rng.random((n, 3)) - 0.5)).astype(np.float32)
    vel = rng.normal(0, 3, (n, 3)).astype(np.float32)
    print("%d^3 cells, %d particles over %g of the box" % (res, n, part), flush=True)
    sim = hip.HIPGridParticleSimulator(box, flags=hip._lib.FLAG_REFERENCE_ORDER, capacity=n + 100)
    sim.upload(pos, vel)
    assert sim.grid_dims()[0] == (res, res, res)
    o = orc.OracleSim(box, n)
    o.add_particles(pos, vel)
    o.set_order_mode(orc.ORDER_REFERENCE)
    for step in range(3):
        sim.updateGrid()
        o.update_grid()
        start, ids = o.buckets()
        c = np.flatnonzero(np.diff(start))
        visit = np.argsort(c % res * res * res + c // res % res * res + c // (res * res))   # x outer, z inner
        want = np.concatenate([ids[start[k]:start[k + 1]] for k in c[visit]])
        np.testing.assert_array_equal(sim.debug(hip._lib.DEBUG_IDS), want, err_msg="grid phase %d" % step)
        if step == 2:
            break
        for phase in (sim.updateDensityPressure, sim.updateForces, sim.updateCollisions, sim.integrate):
            phase()
        o.update_density_pressure()
        o.update_forces()
        o.integrate()
        assert np.isfinite(o.state()["pos"]).all()
    sim.close()
