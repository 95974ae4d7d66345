"""Bins that a caller of abt_diffraction places nearer than make_far_field_bins does (1e6 um), or at mixed distances: the
restructured body's far geometry is used within a limit of the aperture's distance from the origin that follows from
the nearest bin, the full geometry beyond.  Apertures on either side of that limit agree with the plain body.  Its phase
k |x - c| carries at most 12 roundings of 2^-53 (the offset 1, its rotation 5.2, the root 2.5, the products with k 3);
1e-10 is left for the cancellation in its edge sums."""
import numpy as np
import pytest

from abt_amd import lib
from abt_amd.workloads import grid, random_triangles

pytestmark = pytest.mark.gpu
LAM = 0.532


def _far_limit(rmin):
    krev = 2.0 * float(np.float32(3.14159265358979)) / LAM / (2 * np.pi)
    return min((2e-13 / (krev * rmin)) ** 0.2, 1.4e-4) * rmin


@pytest.mark.parametrize("rmin,spread", [(1e3, 1.0), (3e3, 1.0), (1e4, 1.0), (1e5, 1.0), (2e3, 400.0)])
@pytest.mark.parametrize("at", [0.0, 0.5, 0.98, 1.02, 30.0, 900.0])
def test_far_limit_of_near_bins(rmin, spread, at):
    th, ph = grid((0, 6, 180), (0, 17, 340))
    x, y, z = lib.make_far_field_bins(th, ph)
    rng = np.random.default_rng(int(rmin + 10 * at))
    f = rmin / 1e6 * spread ** rng.uniform(size=x.size)
    f[rng.integers(x.size)] = rmin / 1e6
    b = random_triangles(1, seed=3, box=1e-9)
    u = rng.normal(size=3)
    b.verts += at * _far_limit(rmin) * u / np.linalg.norm(u)
    want = lib.diffraction(th, ph, x * f, y * f, z * f, LAM, b, 0, precision="fp64")
    got = lib.diffraction(th, ph, x * f, y * f, z * f, LAM, b, 0, precision="fp64_fast")
    tol = 1e-10 + 12 * 2 * np.pi * (rmin * spread / LAM) * 2.0 ** -53
    assert np.abs(got - want).max() <= tol * np.abs(want).max()
