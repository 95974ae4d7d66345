"""Polygons whose vertex records lie 2^31 and more records into the set's (a set of that many vertices
fits the card): the same bits as near the start.  Only the polygons' own records are there; the
record pointer is moved back by what their offsets are moved on, so every address that is read is the same."""
import ctypes

import numpy as np
import pytest

from abt_amd import lib
from abt_amd.beams import BeamSet, concat
from abt_amd.workloads import grid, random_triangles
from tests import emu

LAM = 0.532
R_NV, R_VOFF, VREC = 30, 31, 12
SHIFTS = [0, 1, 2**31 - 8, 2**31, 2**31 + 9, 5 * 2**31 - 3]


def _case():
    rng = np.random.default_rng(2)
    sets = [random_triangles(3, seed=4, box=8.0)]
    for nv in (4, 5, 7):
        t = 2 * np.pi * (np.arange(nv) + rng.uniform(-0.3, 0.3, nv)) / nv
        v = np.column_stack([3 * np.cos(t), 2 * np.sin(t), 0.7 * np.cos(t) - 0.4 * np.sin(t)])
        prop = [[np.sin(0.6), 0.0, -np.cos(0.6)]]
        sets.append(BeamSet(rng.normal(size=(1, 8)), [(0.0, 1.0, 0.0)], prop, [1.0], [0, nv], v))
    bs = concat(sets)
    recs, vrecs = lib.prepare_beams_host(bs, LAM)
    assert vrecs.size == VREC * len(bs.verts)
    return bs.n, np.array(recs), np.array(vrecs)


def _moved(recs, shift):
    r = recs.copy()
    assert (r[:, R_NV] > 3).sum() == 3
    r[:, R_VOFF] += shift
    return r


@pytest.mark.parametrize("prec", [0, 1, 4])
@pytest.mark.parametrize("shift", SHIFTS)
def test_emu_vertex_offset(prec, shift):
    import oracle
    n, recs, vrecs = _case()
    th, ph = grid((0, 15, 180), (0, 30, 330))
    want = emu.far_field(prec, th, ph, LAM, recs, n, vrecs)
    x, y, z = oracle.make_far_field_bins(th, ph)
    cp, sp = np.cos(ph), np.sin(ph)
    r = _moved(recs, shift)
    out = np.empty(8 * len(th) * len(ph))
    P = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    ti = int(np.argmax(th > oracle.PI_R4 / 180))
    emu.lib().emu_far_field(ctypes.c_int(prec), ctypes.c_int(len(ph)), ctypes.c_int(len(th)), ctypes.c_int(ti),
                            ctypes.c_double(LAM), P(x), P(y), P(z), P(cp), P(sp), P(r),
                            ctypes.c_void_p(vrecs.ctypes.data - 8 * VREC * shift), ctypes.c_int64(n),
                            ctypes.c_int(0), P(out))
    np.testing.assert_array_equal(lib.raw_to_complex(out, len(ph), len(th)), want)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp64_fast", "mixed"])
def test_gpu_vertex_offset(precision):
    import torch
    n, recs, vrecs = _case()
    g = lib.DeviceGrid(*grid((0, 15, 180), (0, 30, 330)), LAM)
    v = torch.from_numpy(vrecs.reshape(-1)).cuda()
    outs = []
    for shift in SHIFTS:
        r = torch.from_numpy(_moved(recs, shift).reshape(-1)).cuda()
        out = torch.full((8 * g.nbins,), np.nan, dtype=torch.float64, device="cuda")
        lib._check(lib.load().abt_far_field_dev(g.handle, ctypes.c_void_p(r.data_ptr()),
                                                ctypes.c_void_p(v.data_ptr() - 8 * VREC * shift), n,
                                                lib.PRECISIONS[precision], 0, ctypes.c_void_p(out.data_ptr()),
                                                None, 0, None))
        torch.cuda.synchronize()
        outs.append(out.cpu().numpy())
    assert np.isfinite(outs[0]).all()
    for o in outs[1:]:
        np.testing.assert_array_equal(o, outs[0])
