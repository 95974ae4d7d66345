"""The plain FP64 body's edges: polygons whose edges follow the aperture frame's axes (their slopes
take the reference's clamps, diff_mod.f90:379-382, so the phase after the edge is not the next
vertex's and is looked up by itself) mixed with triangles and oblique polygons of 4 to 9 vertices,
and the same sets as the whole beam list or behind other beams in it.  Tolerance 1e-9 per bin of the
oracle, the plain kernel's parity bound everywhere."""
import numpy as np
import pytest

from abt_amd import lib
from abt_amd.beams import BeamSet, concat
from abt_amd.workloads import grid, random_triangles
from tests.gpu_util import ampl_rel_err, summary

pytestmark = pytest.mark.gpu
LAM = 0.532


def _polygon(verts, rng, tilt):
    prop = np.array([[np.sin(tilt), 0.0, -np.cos(tilt)]])
    return BeamSet(rng.normal(size=(1, 8)), [(0.0, 1.0, 0.0)], prop, [1.0], [0, len(verts)], verts)


def _aligned(rng):
    """Rectangles and an L-free octagon in the xy plane, edges along x and y, propagating in the x-z plane."""
    sets = []
    for _ in range(3):
        a, b = rng.uniform(2, 6, 2)
        v = np.array([[0, 0, 0], [a, 0, 0], [a, b, 0], [0, b, 0.0]]) + rng.uniform(-3, 3, 3)
        sets.append(_polygon(v, rng, rng.uniform(0.2, 1.0)))
    c = rng.uniform(0.4, 0.9)
    o = np.array([[c, 0], [3 - c, 0], [3, c], [3, 2 - c], [3 - c, 2], [c, 2], [0, 2 - c], [0, c]])
    sets.append(_polygon(np.column_stack([o, np.zeros(8)]) + rng.uniform(-3, 3, 3), rng, 0.6))
    return sets


def _oblique(rng, nv):
    t = 2 * np.pi * (np.arange(nv) + rng.uniform(-0.3, 0.3, nv)) / nv
    v = np.column_stack([3 * np.cos(t), 2 * np.sin(t), 0.7 * np.cos(t) - 0.4 * np.sin(t)])
    return _polygon(v + rng.uniform(-3, 3, 3), rng, rng.uniform(0.2, 1.0))


@pytest.mark.parametrize("seed", [0, 1])
def test_plain_body_polygon_edges(orc, seed):
    th, ph = grid((0, 5, 180), (0, 10, 350))
    rng = np.random.default_rng(seed)
    sets = _aligned(rng) + [_oblique(rng, nv) for nv in (4, 5, 6, 9)]
    for bs in (concat(sets), concat([random_triangles(9, seed=seed, box=8.0)] + sets)):
        ref, _ = orc.diff_main(th, ph, LAM, bs, BeamSet.empty(), nthreads=4)
        got, _ = lib.diff_main(th, ph, LAM, bs, BeamSet.empty(), precision="fp64")
        err = ampl_rel_err(got, ref)
        assert err.max() <= 1e-9, summary(err)
