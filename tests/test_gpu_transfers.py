"""Particles in and out at the edges of the transfers' parts: 256 particles a
workgroup, four words a piece, 16,384 particles an upload's part; at rest or moving,
with the ids that upload gives or shuffled ones, appended behind others."""
import ctypes as C

import numpy as np
import pytest

from test_zz_no_alloc import _hip_runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 5, 255, 256, 257, 1023, 16383, 16384, 16385, 32768, 32769, 70001])
@pytest.mark.parametrize("moving,shuffled", [(False, False), (True, False), (True, True)])
def test_upload_append_readback(hip, n, moving, shuffled):
    rng = np.random.default_rng([n, moving, shuffled])
    more = max(1, n // 3)
    pos = rng.normal(0, 1, (n + more, 3)).astype(np.float32)
    vel = rng.normal(0, 1, (n + more, 3)).astype(np.float32)
    ids = rng.permutation(n + more).astype(np.uint32) if shuffled else np.arange(n + more, dtype=np.uint32)
    print("%d particles, moving %s, shuffled %s" % (n, moving, shuffled), flush=True)
    with hip.HIPGridParticleSimulator(4.0, capacity=n + more + 7) as sim:
        for part, put in ((slice(0, n), sim.upload), (slice(n, n + more), sim.append)):
            put(pos[part], vel[part] if moving else None, ids[part] if shuffled else None)
        if not moving:
            vel[:] = 0
        p, v, got = sim.download(by_id=False)
        assert np.array_equal(got, ids)
        assert np.array_equal(p.view(np.uint32), pos.view(np.uint32))
        assert np.array_equal(v.view(np.uint32), vel.view(np.uint32))
        order = np.argsort(ids)
        p, v = sim.readback()
        assert np.array_equal(p.view(np.uint32), pos[order].view(np.uint32))
        assert np.array_equal(v.view(np.uint32), vel[order].view(np.uint32))
        p, v = sim.readback(with_velocity=False)
        assert np.array_equal(p.view(np.uint32), pos[order].view(np.uint32)) and v is None
        sim.upload(pos[:n], vel[:n], np.minimum(ids[:n], n))   # an id that readback refuses, unless all are below n
        if ids[:n].max() >= n:
            with pytest.raises(Exception, match="ids are not 0..count-1"):
                sim.readback()


def test_readback_takes_no_device_memory(hip):
    """The slots by id lie in a buffer that the context has: the first readback of 4 million
    particles (16 MB of them) leaves the device's free memory as it was."""
    free, total = C.c_size_t(), C.c_size_t()
    rt = _hip_runtime()

    def free_bytes():
        assert rt.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    n = 4_000_000
    rng = np.random.default_rng(11)
    pos = (9.0 * (rng.random((n, 3)) - 0.5)).astype(np.float32)
    ids = rng.permutation(n).astype(np.uint32)
    with hip.HIPGridParticleSimulator(10.0, capacity=n) as sim:
        sim.upload(pos, None, ids)
        sim.sync()
        before = free_bytes()
        p, _ = sim.readback()
        after = free_bytes()
        assert np.array_equal(p[ids].view(np.uint32), pos.view(np.uint32))
        assert before - after < 4 * n
        # between phases: the grid phase's results stay as they are
        sim.updateGrid()
        p, _ = sim.readback(with_velocity=False)
        assert np.array_equal(p[ids].view(np.uint32), pos.view(np.uint32))
        for phase in (sim.updateDensityPressure, sim.updateForces, sim.updateCollisions, sim.integrate):
            phase()
            assert np.isfinite(sim.readback()[0]).all()
