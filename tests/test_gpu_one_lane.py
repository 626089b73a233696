"""The forms for many particles where they can go wrong.  A solver with LDS
tiles switched on takes neither the deep passes nor the four-lane search, so
small scenes reach the one-lane passes of IISPH, ISPH and pellets: lists below,
at and past their cap, counts around the waves' edges, periodic boxes, bodies
moved by the fluid and pellets that push back, one step at a time against the
oracle from a synchronised state.  Past 81,920 particles (or with tiles, in a
periodic box) the search stages its rows, and falls back to global memory where
it cannot: those lists, bit for bit."""
import time

import numpy as np
import pytest

import alluvion_amd._alluvion as al
from alluvion_amd import scenes
from gpu_sync import oracle_for, rel_err
from test_gpu_edges import free_body_matches
from test_gpu_few_particles import cloud, step_matches
from test_gpu_pellets import isph_steps_match

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["ii", "i"])
@pytest.mark.parametrize("n,kmax", [(1, 64), (63, 64), (257, 64), (900, 7), (900, 41), (900, 90)])
def test_pressure_solvers(n, kmax, kind):
    step_matches(cloud(n, (4, 4, 4), 9, kmax=kmax), kind, tiles=True)


@pytest.mark.parametrize("cells,wrap,margin", [
    ((6, 8, 5), (True, True, True), 0), ((6, 8, 6), (True, False, True), 0),
    ((6, 4, 6), (True, True, True), 0), ((6, 6, 8), (True, True, True), 1)])
@pytest.mark.parametrize("kind", ["df", "ii", "i"])
def test_periodic_boxes(cells, wrap, margin, kind):
    n = int(8 * cells[0] * cells[1] * cells[2]) - 3
    step_matches(cloud(n, cells, 5, wrap=wrap, margin=margin), kind, tiles=True)


@pytest.mark.parametrize("kind", ["ii", "i"])
def test_free_body(kind):
    free_body_matches(kind, tiles=True)


def test_pellets():
    isph_steps_match(tiles=True)


def lists_match(sc, tiles=False):
    """Lists bit for bit, their density, and the flag of a list past its cap."""
    dp, pile, solver, _, _ = scenes.build_solver(sc)
    solver.set_tiles(tiles)
    orc = oracle_for(sc, dp, [])
    solver.update_particle_neighbors()
    orc.update_particle_neighbors()
    ids, cnt = solver.get_neighbors()
    oids, ocnt = orc.neighbors()
    n, K = sc.n, sc.max_num_neighbors
    np.testing.assert_array_equal(cnt[:n], ocnt[:n])
    mask = np.arange(K)[None, :] < ocnt[:n, None]
    np.testing.assert_array_equal(np.where(mask, ids[:n], 0), np.where(mask, oids[:n], 0))
    assert rel_err(dp.coat(solver.particle_density).get()[:n], orc.get("density")[:n]) < 1e-6
    flags = dp.coat(solver.grid_anomaly).get()
    assert bool(flags[2]) == bool((ocnt[:n] == K).any())
    return ocnt[:n]


def stretched(sc, factor):
    sc.x = (sc.x * np.float32(factor)).astype(np.float32)
    return sc


@pytest.mark.parametrize("name", ["short lists", "past LDS", "sparse", "dense", "outside",
                                  "wider than the box", "four cells high"])
def test_staged_search(name):
    n = 82001
    sc = {
        "short lists": lambda: cloud(n, (22, 24, 20), 1, kmax=24),  # below the mean of 33
        "past LDS": lambda: cloud(n, (18, 20, 18), 1, kmax=70),
        "sparse": lambda: cloud(n, (48, 50, 48), 1),  # more runs of cells per wave than staged
        "dense": lambda: cloud(n, (10, 12, 10), 1, kmax=40),  # 205 candidates in a row
        "outside": lambda: stretched(cloud(n, (22, 24, 20), 1), 1.08),
        "wider than the box": lambda: cloud(n, (22, 24, 20), 1, wrap=(True, True, True), margin=1),
        "four cells high": lambda: cloud(n, (50, 52, 4), 1, wrap=(True, False, True)),
    }[name]()
    cnt = lists_match(sc)
    if name in ("short lists", "dense"):
        assert (cnt == sc.max_num_neighbors).any()


@pytest.mark.parametrize("n,cells,kmax,wrap,margin", [
    (900, (6, 5, 6), 7, (True, True, True), 0), (2500, (6, 5, 6), 40, (True, False, True), 0),
    (2500, (6, 5, 6), 90, (True, True, True), 0),
    (9000, (6, 5, 5), 40, (True, True, True), 0),  # a row of 180 candidates
    (400, (12, 12, 12), 64, (True, True, True), 0),  # a particle per run
    (900, (6, 5, 6), 7, (True, True, False), 1), (900, (6, 5, 6), 41, (False, False, True), 1),
    (900, (6, 3, 4), 200, (True, True, True), 0), (900, (3, 6, 3), 200, (True, False, True), 0)])
def test_periodic_search(n, cells, kmax, wrap, margin):
    lists_match(cloud(n, cells, 3, kmax=kmax, wrap=wrap, margin=margin), tiles=True)


@pytest.mark.parametrize("name,most", [("wider than the box", 1.25), ("tiles", 1.6)])
def test_general_loop_keeps_a_wave_together(name, most):
    """The search of 300,000 particles where rows are not staged, over the one
    where they are: 1.05 and 1.34, and 1.48 and 1.83 with a wave's lanes scanning
    their spans one after another."""
    cells = (34, 34, 34)
    wrap = (True, True, True) if name != "tiles" else None
    margin = 1 if name != "tiles" else 0
    solvers = []
    for m, tiles in ((0, False), (margin, name == "tiles")):
        built = scenes.build_solver(cloud(300000, cells, 1, wrap=wrap, margin=m))
        built[2].set_tiles(tiles)
        solvers.append(built)
    best = [1e30, 1e30]
    for _ in range(12):
        for k, built in enumerate(solvers):
            al.device_synchronize()
            t0 = time.perf_counter()
            built[2].update_particle_neighbors()
            al.device_synchronize()
            best[k] = min(best[k], time.perf_counter() - t0)
    print(name, "%.3f" % (best[1] / best[0]), flush=True)
    assert best[1] < most * best[0], best
