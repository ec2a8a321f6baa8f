"""The grid phase's stable sort by cell, where its parts change: cell counts at the
edges of the scan's tiles (4,096 entries), slot counts at the edges of the
workgroups (256), crowded cells, particles outside the box, and keys counted by the
hash as well as by the step before. Against numpy's stable argsort of the cells."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def positions(layout, n, box, rng):
    pos = (rng.random((n, 3)) - 0.5) * box
    if layout == "one cell":
        pos[:] = 0.001 * rng.random((n, 3))
    elif layout == "two cells":
        pos[:] = 0.001 * rng.random((n, 3))
        pos[::2, 0] += 0.0914
    elif layout == "outside":
        pos[::3] *= 1e3
        pos[1::7] = np.nan
    return pos.astype(np.float32)


def check_sorted(sim, lib, ncells):
    pre = sim.debug(lib.DEBUG_CELL_PRESORT)
    want = np.argsort(pre, kind="stable").astype(np.uint32)
    np.testing.assert_array_equal(sim.debug(lib.DEBUG_PERM), want)
    np.testing.assert_array_equal(sim.debug(lib.DEBUG_CELL), pre[want])
    np.testing.assert_array_equal(sim.debug(lib.DEBUG_CELL_START),
                                  np.searchsorted(pre[want], np.arange(ncells + 1), side="left").astype(np.uint32))
    return pre, want


@pytest.mark.parametrize("res,n,layout", [
    ((1, 1, 1), 1, "uniform"), ((3, 5, 7), 255, "uniform"), ((3, 5, 7), 256, "uniform"), ((3, 5, 7), 257, "uniform"),
    ((2, 23, 89), 5000, "uniform"),      # 4,094 cells: 4,096 scanned entries, one tile
    ((3, 5, 273), 5000, "uniform"),      # 4,095: one entry of a second tile
    ((16, 16, 16), 5000, "uniform"), ((65, 64, 63), 70000, "uniform"),   # 64 tiles; 1 more than a look-back reads
    ((9, 9, 9), 3000, "one cell"), ((9, 9, 9), 4097, "two cells"), ((9, 8, 7), 3000, "outside"),
    ((210, 200, 204), 3000, "uniform"),  # more cells than are worth counting: sorted by digits
])
def test_stable_sort_and_cell_table(hip, res, n, layout):
    lib = hip._lib
    h = float(hip.scenes.H)
    box = np.array([(r - 0.5) * h for r in res], np.float32)
    rng = np.random.default_rng([n, *res])
    pos = positions(layout, n, box, rng)
    vel = rng.normal(0, 0.5, (n, 3)).astype(np.float32)
    print("grid %s, %d particles, %s" % (res, n, layout), flush=True)
    sim = hip.HIPGridParticleSimulator(box, capacity=n + 300)   # unused slots after the particles
    sim.upload(pos, vel)
    dims, ncells = sim.grid_dims()
    assert dims == res
    sim.updateGrid()
    pre, want = check_sorted(sim, lib, ncells)
    p, v, ids = sim.download(by_id=False)
    assert np.array_equal(ids, want)
    assert np.array_equal(p.view(np.uint32), pos[want].view(np.uint32))
    assert np.array_equal(v.view(np.uint32), vel[want].view(np.uint32))
    # the next sort starts from the keys that the integration wrote
    sim.updateDensityPressure()
    sim.updateForces()
    sim.updateCollisions()
    sim.integrate()
    sim.updateGrid()
    check_sorted(sim, lib, ncells)
    for phase in (sim.updateDensityPressure, sim.updateForces, sim.updateCollisions, sim.integrate):
        phase()
    # and from those that the fused step wrote
    sim.advance(2)
    sim.updateGrid()
    check_sorted(sim, lib, ncells)
    sim.close()


def test_sort_with_uneven_scenes_and_an_emitter(hip):
    """Scenes with unused slots, an empty one and one that grows on the device: in
    every scene the cell table counts exactly the live particles, step after step,
    eagerly and from graphs."""
    lib = hip._lib
    for graphs in (False, True):
        b = hip.SceneBatch([(0.4, 700), (0.3, 600), (0.5, 2000)])
        rng = np.random.default_rng(7)
        b.upload(0, ((rng.random((650, 3)) - 0.5) * 0.4).astype(np.float32))
        b.upload(2, ((rng.random((900, 3)) - 0.5) * 0.5).astype(np.float32))
        b.set_emitter(2, rate=150, limit=1900, radius=0.1, seed=5)
        b.set_graphs(graphs)
        for step in range(6):
            b.phase(lib.PHASE_GRID)
            for i, n in ((0, 650), (1, 0), (2, min(1900, 900 + 150 * (3 * step + 1)))):
                assert b.count(i) == n
                cells = b.debug(i, lib.DEBUG_CELL)
                start = b.debug(i, lib.DEBUG_CELL_START)
                want = np.searchsorted(cells, np.arange(len(start)), side="left").astype(np.uint32)
                assert np.all(np.diff(cells.astype(np.int64)) >= 0) and np.array_equal(start, want)
                assert np.array_equal(np.sort(b.download(i, by_id=False)[2]), np.arange(n))
            for phase in (lib.PHASE_DENSITY, lib.PHASE_FORCES, lib.PHASE_COLLISIONS, lib.PHASE_INTEGRATE):
                b.phase(phase)
            b.step(2)
        b.close()


@pytest.mark.parametrize("n,run", [(256, 1), (258, 1), (2000, 1), (2000, 3), (2000, 7), (40000, 64), (5001, 1000)])
def test_crowded_cells(hip, n, run):
    """Two cells of n / 2 particles, as many as a lane goes through by itself (128), one more,
    and many, with runs of 1 to 1,000 consecutive slots."""
    lib = hip._lib
    h = float(hip.scenes.H)
    rng = np.random.default_rng([n, run])
    pos = (0.01 * h * rng.random((n, 3)) + 0.3 * h).astype(np.float32)
    pos[(np.arange(n) // run) % 2 == 1, 0] += np.float32(h)
    print("%d particles, runs of %d" % (n, run), flush=True)
    sim = hip.HIPGridParticleSimulator((4 * h, 3 * h, 3 * h), capacity=n + 3)
    sim.upload(pos, rng.normal(0, 0.2, (n, 3)).astype(np.float32))
    for step in range(2):
        sim.updateGrid()
        check_sorted(sim, lib, sim.grid_dims()[1])
        for phase in (sim.updateDensityPressure, sim.updateForces, sim.updateCollisions, sim.integrate):
            phase()
    sim.close()


def test_a_crowded_cell_does_not_hold_up_the_sort(hip):
    """40,000 particles in one cell against as many in 8,000 cells: the sort's time grew with
    the square of a cell's particles (14 times as long), and may be some times as long."""
    h = float(hip.scenes.H)
    n, box = 40000, 19.5 * h
    rng = np.random.default_rng(1)
    at = rng.random((n, 3))
    ms = []
    for pos in ((box * (at - 0.5)), 0.9 * h * at):
        with hip.HIPGridParticleSimulator(box, capacity=n) as sim:
            t = []
            for _ in range(6):
                sim.upload(pos.astype(np.float32))
                t.append(sim.updateGrid())
                for phase in (sim.updateDensityPressure, sim.updateForces, sim.updateCollisions, sim.integrate):
                    phase()
            ms.append(min(t[1:]))
    print("spread %.3f ms, crowded %.3f ms" % tuple(ms), flush=True)
    assert ms[1] < 6.0 * ms[0]


@pytest.mark.parametrize("res,n,more", [(30, 200_000, 220), (102, 200_000, 220), (102, 1_200_000, 260),
                                        (257, 200_000, 0), (385, 8_000_000, 0)])
def test_digit_sort_across_key_widths(hip, res, n, more):
    """The stable sort by digits: two 8-bit passes (30^3 cells), three (102^3) and three of 10
    bits (257^3, 385^3; with 8,000,000 particles the histograms fill 489 scan tiles). An
    empty scene of more^3 cells beside the first makes the cells too many to count."""
    lib = hip._lib
    h = float(hip.scenes.H)
    boxes = [float(np.float32((r - 0.5) * h)) for r in (res, more) if r]
    assert sum(r ** 3 for r in (res, more)) > (8 << 20) + 6 * n
    rng = np.random.default_rng([res, n])
    pos = ((rng.random((n, 3)) - 0.5) * boxes[0]).astype(np.float32)
    print("%d^3 cells, %d particles" % (res, n), flush=True)
    with hip.SceneBatch([(boxes[0], n)] + [(b, 256) for b in boxes[1:]]) as b:
        b.upload(0, pos)
        assert b.grid(0)[0] == (res, res, res)
        b.phase(lib.PHASE_GRID)
        pre = b.debug(0, lib.DEBUG_CELL_PRESORT)
        want = np.argsort(pre, kind="stable").astype(np.uint32)
        np.testing.assert_array_equal(b.debug(0, lib.DEBUG_PERM), want)
        np.testing.assert_array_equal(b.debug(0, lib.DEBUG_CELL), pre[want])
        np.testing.assert_array_equal(b.debug(0, lib.DEBUG_CELL_START),
                                      np.searchsorted(pre[want], np.arange(res ** 3 + 1), side="left").astype(np.uint32))
        np.testing.assert_array_equal(b.download(0, by_id=False)[2], want)
