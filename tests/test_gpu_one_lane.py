"""The forms for many particles where they can go wrong.  A solver with LDS
tiles switched on takes neither the deep passes nor the four-lane search, so
small scenes reach the one-lane passes of IISPH, ISPH and pellets: lists below,
at and past their cap, counts around the waves' edges, periodic boxes, bodies
moved by the fluid and pellets that push back, one step at a time against the
oracle from a synchronised state."""
import pytest

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
