"""abt_diff_main's two ways back: results that fit one slot (1 MiB, 8192 bins) in one copy, larger ones each on their own,
with a second stream from 8 external beams on.  Trees of every length on either side, empty ones among them,
bit-identical to the device interface on the same records."""
import numpy as np
import pytest

from abt_amd import lib
from abt_amd.beams import BeamSet
from abt_amd.workloads import random_triangles
from tests.test_gpu_host_staging import LAM, _angles, _device, _polygons

pytestmark = pytest.mark.gpu
EXT_FOV = np.float64(np.float32(3.14159265358979)) / 2


@pytest.mark.parametrize("nth,nph", [(3, 3), (2730, 3), (64, 128), (2731, 3), (91, 91)])
@pytest.mark.parametrize("nb,ne", [(1, 1), (3, 7), (3, 8), (700, 40), (0, 9), (5, 0)])
def test_both_trees(nth, nph, nb, ne):
    th, ph = _angles(nth, nph)
    b = random_triangles(nb, seed=nb, box=20.0) if nb else BeamSet.empty()
    e = _polygons(ne, ne) if ne else BeamSet.empty()
    print(f"both trees {nth} x {nph}, {nb} + {ne}", flush=True)
    got_b, got_e = lib.diff_main(th, ph, LAM, b, e, raw=True)
    np.testing.assert_array_equal(got_b, _device(th, ph, b) if nb else np.zeros(8 * nth * nph))
    np.testing.assert_array_equal(got_e, _device(th, ph, e, EXT_FOV) if ne else np.zeros(8 * nth * nph))
