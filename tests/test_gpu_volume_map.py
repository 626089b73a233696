"""Volume maps over the classes of their nodes (outside, inside, near) and the
kernels that sum the near ones: every shape and sign at odd resolutions
against the oracle, and maps large enough for the one-wave kernel against the
few-node kernel bit for bit at the nodes both have."""
import numpy as np
import pytest

import oracle_ffi as of
from alluvion_amd import scenes

pytestmark = pytest.mark.gpu


def one_boundary(kind, params, sign, res, sampled=False):
    sc = scenes.dam_break_small()
    sc.boundaries = [scenes.BoundarySpec(kind, params, sign, res, sampled=sampled)]
    return sc


def gpu_map(sc):
    dp, pile, _, _, _ = scenes.build_solver(sc)
    dist = dp.coat(pile.distance_grids[0]).get() if sc.boundaries[0].sampled else None
    return dp.coat(pile.volume_grids[0]).get(), dist


@pytest.mark.parametrize("kind,params,sign,res", [
    ("box", (0.1, 0.06, 0.08, 0.0), -1.0, (7, 5, 6)),
    ("box", (0.05, 0.04, 0.03, 0.002), 1.0, (9, 4, 1)),
    ("box_shell", (0.06, 0.05, 0.04, 0.015, 0.001), 1.0, (8, 3, 6)),
    ("sphere", (0.03,), 1.0, (6, 7, 9)),
    ("sphere", (0.004,), 1.0, (4, 4, 4)),  # smaller than the kernel: no node is inside
    ("sphere", (0.05,), -1.0, (3, 8, 2)),
])
@pytest.mark.parametrize("sampled", [False, True])
def test_every_class_matches_oracle(kind, params, sign, res, sampled):
    sc = one_boundary(kind, params, sign, res, sampled)
    got, dist = gpu_map(sc)
    orc = of.Oracle(sc, precision=4)
    if sampled:
        orc.set_distance_map(0, dist)
    orc.build_volume_map(0)
    ref = orc.volume_map(0)
    scale = 4 * np.pi / 3 * sc.kernel_radius ** 3
    # 27,000 single-precision terms: the sum's rounding is below 1e-5 of it
    assert np.abs(got.astype(np.float64) - ref).max() <= 1e-5 * scale
    np.testing.assert_array_equal(got == 0.0, ref == 0.0)


@pytest.mark.parametrize("kind,params,sign", [
    ("sphere", (0.05,), 1.0), ("box", (0.2, 0.2, 0.2, 0.0), -1.0),
    ("box_shell", (0.1, 0.1, 0.1, 0.02, 0.0), 1.0)])
def test_both_kernels_give_the_same_sums(kind, params, sign):
    # corner nodes of the coarse grid are corner nodes of the fine one: their
    # coordinates are the same numbers (cell sizes in the ratio 4)
    coarse, _ = gpu_map(one_boundary(kind, params, sign, (24,) * 3))
    fine, _ = gpu_map(one_boundary(kind, params, sign, (96,) * 3))
    c = coarse[:25 ** 3].reshape(25, 25, 25)
    f = fine[:97 ** 3].reshape(97, 97, 97)[::4, ::4, ::4]
    assert (c > 0).any()
    np.testing.assert_array_equal(c, f)


def test_large_sampled_map_matches_oracle():
    """A sampled map with more nodes near the surface than run as teams (every
    node whose volume lies between none and the whole ball is one)."""
    sc = one_boundary("box", (0.04, 0.05, 0.045, 0.0), 1.0, (48, 50, 52), sampled=True)
    got, dist = gpu_map(sc)
    ball = 4 * np.pi / 3 * sc.kernel_radius ** 3
    near = np.flatnonzero((got > 1e-3 * ball) & (got < 0.99 * ball))
    assert near.size > 1 << 19
    dmin, dmax, res, cs = of.Oracle(sc, precision=4).grid_info(0)
    picked = np.random.default_rng(3).choice(near, 40, replace=False)
    picked = np.concatenate([picked, [0, got.size - 1], np.flatnonzero(got == 0.0)[:10],
                             np.argsort(got)[-10:]])
    for node in picked:
        ref = of.volume_from_distance_map(4, sc.kernel_radius, dmin, dmax, res, cs, 1.0, dist,
                                          int(node), int(node) + 1)[0]
        assert abs(float(got[node]) - ref) <= 1e-5 * ball, node
