"""Facet midpoints that are not finite.  The reference's edge checks of such a midpoint are comparisons with NaN or an
infinity, which are false or decided by sign: a NaN midpoint is outside no edge, so every triangle of its box in
front of it blocks it, whichever side it is seen from.  Bit-identical to the oracle, as everywhere."""
import numpy as np
import pytest

import oracle as O
from abt_amd import visibility as V
from abt_amd.workloads import vis_workload
from tests.test_gpu_vis import _batch, _geom, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["int", "ext", "inc"])
@pytest.mark.parametrize("x,y", [(np.nan, None), (None, np.nan), (np.nan, np.nan), (np.inf, None), (None, -np.inf),
                                 (np.inf, np.nan)])
def test_midpoints_not_finite(mode, x, y):
    nbeam = 5
    topo, v, mid, nz, apn, ino, fin, bmz = vis_workload(nbeam, mode, seed=13)
    for b in range(1, nbeam):   # beam 0 as it is; 1, 3, 9 and 27 facets of the others
        for k in np.linspace(0, topo.nf - 1, 3 ** (b - 1)).astype(int):
            if x is not None:
                mid[b, k, 0] = x
            if y is not None:
                mid[b, k, 1] = y
    args = topo, v, mid, nz, apn, ino, fin, bmz
    print(f"vis not finite {mode} {x} {y}", flush=True)
    ref, _ = O.find_vis_batch(mode, *args)
    r, _ = _batch(mode, *args, counts=False)
    _same(r, ref, mode)
    f = fin[ino[4]:ino[5]] if mode != "inc" else None
    _same(V.find_vis(mode, _geom(topo, v, mid, nz, apn, 4), f, bmz[4]), {k: ref[k][4] for k in ref}, f"{mode} one beam")
