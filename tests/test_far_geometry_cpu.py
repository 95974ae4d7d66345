"""The restructured FP64 body's geometry on both sides of its far limit (|com| against the bins'
distance), at its smallest and largest wavelengths and for bins nearer than usual, on the CPU emulator of
the kernel bodies against the frame-free FP64 model: centres just inside, on and beyond the limit, where
the distances take over from the series.  Tolerance 1e-9 of the floored amplitude: the model's phase
k (|x - c| - |x|) <= 6e4 rad is rounded to 4e-12 rad, its polarisation to ~1e-12 at these bins."""
import numpy as np
import pytest

from abt_amd import lib
from abt_amd.beams import BeamSet
from abt_amd.workloads import grid, random_triangles
from tests import emu
from tests.gpu_util import ampl_rel_err, summary


def _centred_at(n, dist, seed):
    """n seeded triangles with centres at distance `dist` from the origin."""
    b = random_triangles(n, seed=seed, box=2.0)
    v = b.verts.reshape(n, 3, 3)
    c = v.mean(1)
    d = np.random.default_rng(seed + 1).normal(size=(n, 3))
    d *= dist / np.linalg.norm(d, axis=1)[:, None]
    return BeamSet(b.ampl, b.vk7, b.prop, b.fov, b.vert_off, (v - c[:, None] + d[:, None]).reshape(-1, 3))


@pytest.mark.parametrize("lam", [0.2, 0.532, 1.5])
@pytest.mark.parametrize("dist", [0.0, 1e-3, 10.0, 100.0, 139.0, 141.0, 1000.0])
def test_far_and_near_geometry(lam, dist):
    th, ph = grid((0, 7, 175), (0, 23, 345))
    b = _centred_at(12, dist, seed=int(dist) + 3)
    recs, vr = lib.prepare_beams_host(b, lam)
    got = emu.far_field(4, th, ph, lam, recs, b.n, vr)
    want = emu.far_field(3, th, ph, lam, recs, b.n, vr)
    err = ampl_rel_err(got, want)
    assert err.max() <= 1e-9, summary(err)
