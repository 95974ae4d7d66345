"""A device grid's arrays: the exponential table, which kernels read in 16-byte pairs, is aligned to them on grids of every
size (the other arrays' lengths add up to an odd number of doubles on half of all grids)."""
import ctypes

import pytest

from abt_amd import lib
from abt_amd.workloads import grid

pytestmark = pytest.mark.gpu


class DevGrid(ctypes.Structure):   # abt::DevGrid, the first member of the handle
    _fields_ = [("sizes", ctypes.c_int32 * 4), ("scales", ctypes.c_double * 4), ("f32", ctypes.c_float * 2),
                ("more", ctypes.c_double * 3)] + [(k, ctypes.c_void_p) for k in (
                    "x", "y", "z", "cphi", "sphi", "rad", "kr_rev", "theta", "phi", "etab", "wphi", "wth")]


@pytest.mark.parametrize("nth,nph", [(3, 3), (4, 3), (3, 4), (4, 4), (181, 90), (37, 35)])
def test_table_is_aligned(nth, nph):
    g = lib.DeviceGrid(*grid((0, 180.0 / (nth - 1), 180.0), (0, 360.0 / nph, 360.0 - 360.0 / nph)), 0.532)
    d = ctypes.cast(g.handle, ctypes.POINTER(DevGrid))[0]
    assert list(d.sizes[:3]) == [nph, nth, nph * nth] and d.scales[0] == 0.532
    assert all(getattr(d, k) for k in ("x", "etab", "wth")) and d.y == d.x + 8 * g.nbins
    assert d.etab % 16 == 0
