"""The kernel forms for few particles (deep passes, four-lane search) and the
staged search where they can go wrong: particle counts around the waves' and
the blocks' edges, lists at and past their cap and past the slots kept in LDS,
periodic boxes that the cells fill exactly and ones they do not, and counts on
both sides of the forms' limits, one step against the oracle from a
synchronised state.  Lists are compared bit for bit, fields within the
per-step tolerance (the sums are the oracle's in its order)."""
import numpy as np
import pytest

from alluvion_amd import scenes
from gpu_sync import compare_fields, oracle_for, sync

pytestmark = pytest.mark.gpu


def cloud(n, cells, seed, wrap=None, kmax=64, margin=0, density=1.0):
    """n random particles in a box of cells[a] cells (h = 0.01), optionally
    periodic on the axes of `wrap`, with `margin` cells of grid around it."""
    rng = np.random.default_rng(seed)
    length = np.array(cells) * 0.01
    x = ((rng.random((n, 3)) - 0.5) * length * 0.999999).astype(np.float32)
    v = rng.uniform(-0.5, 0.5, (n, 3)).astype(np.float32)
    w = tuple(float(length[a]) if wrap and wrap[a] else 0.0 for a in range(3))
    return scenes.Scene(
        name="cloud", x=x, v=v, gravity=(0.0, -9.81, 0.0), wrap_length=w, max_num_neighbors=kmax,
        max_num_particles_per_cell=512,
        grid_offset=tuple(-(c // 2) - margin for c in cells),
        grid_res=tuple(c + 2 * margin for c in cells), boundaries=[],
        max_divergence_solve=3, max_density_solve=4)


def step_matches(sc, kind="df", tiles=False):
    dp, pile, solver, _, _ = scenes.build_solver(sc, kind)
    solver.set_tiles(tiles)
    orc = oracle_for(sc, dp, [], kind=kind)
    solver.update_particle_neighbors()
    orc.update_particle_neighbors()
    ids, cnt = solver.get_neighbors()
    oids, ocnt = orc.neighbors()
    np.testing.assert_array_equal(cnt[:sc.n], ocnt[:sc.n])
    mask = np.arange(sc.max_num_neighbors)[None, :] < ocnt[:sc.n, None]
    np.testing.assert_array_equal(np.where(mask, ids[:sc.n], 0), np.where(mask, oids[:sc.n], 0))
    sync(dp, solver, pile, orc, kind=kind)
    solver.step()
    orc.step()
    assert solver.num_density_solve == orc.report()["num_density_solve"]
    compare_fields(dp, solver, orc, kind=kind, tag=str((sc.n, kind)))


@pytest.mark.parametrize("n", [1, 15, 17, 63, 65, 255, 257, 1000])
def test_counts_around_waves_and_blocks(n):
    step_matches(cloud(n, (4, 4, 4), n))


@pytest.mark.parametrize("kmax", [7, 30, 40, 64, 90])
def test_list_caps(kmax):
    # mean list length about 60: caps below, at and above the slots in LDS
    step_matches(cloud(900, (4, 4, 4), 3, kmax=kmax))


@pytest.mark.parametrize("cells,wrap,margin", [
    ((6, 8, 5), (True, True, True), 0),
    ((6, 4, 6), (True, True, True), 0),  # an axis of four cells: the general wrap
    ((6, 8, 6), (True, False, True), 0),
    ((8, 6, 6), (False, True, False), 0),
    ((6, 6, 8), (True, True, True), 1),  # the grid is larger than the box
])
@pytest.mark.parametrize("kind", ["df", "ii", "i"])
def test_periodic_boxes(cells, wrap, margin, kind):
    n = int(8 * np.prod(cells)) - 3
    step_matches(cloud(n, cells, 5, wrap=wrap, margin=margin), kind)


@pytest.mark.parametrize("wrap", [None, (True, True, True)])
@pytest.mark.parametrize("n", [81920, 81921, 98304, 98305])
def test_both_sides_of_the_limits(n, wrap):
    step_matches(cloud(n, (22, 24, 20), 7, wrap=wrap))


@pytest.mark.parametrize("kind", ["ii", "i"])
@pytest.mark.parametrize("n,cells,kmax", [(17, (4, 4, 4), 64), (900, (4, 4, 4), 7),
                                          (900, (4, 4, 4), 41), (900, (4, 4, 4), 90),
                                          (98305, (22, 24, 20), 64),
                                          (131072, (24, 26, 24), 64),
                                          (131073, (24, 26, 24), 64)])
def test_pressure_solvers(n, cells, kmax, kind):
    # a wave's last particles, lists of one and of several rounds, the other form
    step_matches(cloud(n, cells, 9, kmax=kmax), kind)


@pytest.mark.parametrize("ns", [1, 15, 65, 300])
@pytest.mark.parametrize("kmax,wrap", [(7, None), (64, None), (40, (True, True, True)),
                                       (64, (True, False, True))])
def test_sample_lists(ns, kmax, wrap):
    sc = cloud(900, (6, 5 if wrap is None else 6, 6), 9, wrap=wrap, kmax=kmax)
    dp, pile, solver, _, _ = scenes.build_solver(sc)
    solver.update_particle_neighbors()
    orc = oracle_for(sc, dp, [])
    orc.update_particle_neighbors()
    rng = np.random.default_rng(ns)
    pts = ((rng.random((ns, 3)) - 0.5) * 0.07).astype(np.float32)  # some outside the grid
    pts[:ns // 3] = sc.x[:ns // 3]  # the particle of the sample's own index is left out
    sx = dp.create_coated((ns,), 3)
    sx.set(pts)
    nbr, cnt = dp.create((ns, kmax), 4), dp.create((ns,), 1, np.uint32)
    runner = dp.Runner()
    runner.launch_make_neighbor_list(sx, solver.pid, solver.pid_length, nbr, cnt, solver.grid_anomaly,
                                     ns)
    ids, xixj, counts = orc.sample_neighbors(pts)
    np.testing.assert_array_equal(dp.coat(cnt).get(), counts)
    got = dp.coat(nbr).get().reshape(ns, kmax, 4)
    for k in range(ns):
        c = counts[k]
        np.testing.assert_array_equal(got[k, :c, 3].view(np.uint32), ids[k, :c])
        np.testing.assert_array_equal(got[k, :c, :3], xixj[k, :c].astype(np.float32))
    out = dp.create((ns,), 1)
    runner.launch_sample_fluid_density(nbr, cnt, out, ns)
    want = orc.sample_density(xixj, counts)
    assert np.abs(dp.coat(out).get() - want).max() <= 1e-5 * max(np.abs(want).max(), 1e-30)
