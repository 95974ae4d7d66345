"""The host entry points' staging at the edges of its slots: results around the size that goes in one copy (64 KiB), a
slot (1 MiB) and the ring of four; record sets around the threads' share and beyond the pinned memory; polygons; several
threads at once.  Bit-identical to the device interface on the same records."""
import threading

import numpy as np
import pytest

from abt_amd import lib
from abt_amd.beams import BeamSet
from abt_amd.workloads import random_triangles

pytestmark = pytest.mark.gpu
LAM = 0.532


def _angles(nth, nph):
    return np.linspace(0.0, 3.1, nth), np.linspace(0.0, 6.2, nph)


def _device(th, ph, b, fov_value=None):
    import torch
    g = lib.DeviceGrid(th, ph, LAM)
    recs, vrecs = lib.prepare_beams_host(b, LAM, fov_value)
    out = torch.empty(8 * g.nbins, dtype=torch.float64, device="cuda")
    lib.far_field_dev(g, torch.from_numpy(recs).cuda(), b.n, out, vrecs=torch.from_numpy(vrecs).cuda(), precision="fp64")
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _polygons(n, seed):
    rng = np.random.default_rng(seed)
    tri = random_triangles(n, seed=seed, box=20.0)
    nv = rng.integers(3, 8, n)
    off = np.r_[0, np.cumsum(nv)]
    verts = []
    for i in range(n):
        v = tri.verts[3 * i:3 * i + 3]
        e1, e2 = v[1] - v[0], v[2] - v[0]
        a = 2 * np.pi * np.arange(nv[i]) / nv[i]
        verts.append(v.mean(0) + 0.3 * (np.cos(a)[:, None] * e1 + np.sin(a)[:, None] * e2))
    return BeamSet(tri.ampl, tri.vk7, tri.prop, tri.fov, off, np.concatenate(verts))


@pytest.mark.parametrize("nth,nph", [(31, 33), (32, 32), (41, 25), (127, 129), (128, 128), (145, 113), (256, 256),
                                     (257, 255), (300, 290)])
def test_results_around_slot_sizes(nth, nph):
    th, ph = _angles(nth, nph)
    b, e = random_triangles(7, seed=nth, box=20.0), _polygons(5, nph)
    print(f"staging {nth} x {nph}", flush=True)
    got_b, got_e = lib.diff_main(th, ph, LAM, b, e, raw=True)
    np.testing.assert_array_equal(got_b, _device(th, ph, b))
    np.testing.assert_array_equal(got_e, _device(th, ph, e, np.float64(np.float32(3.14159265358979)) / 2))
    only_e = lib.diff_main(th, ph, LAM, b, e, raw=True, trees=("ext",))[1]
    np.testing.assert_array_equal(only_e, got_e)


@pytest.mark.parametrize("n", [1, 511, 1023, 1024, 1025, 5000])
def test_records_over_threads_match_one_by_one(n):
    b = _polygons(n, n)
    recs, vrecs = lib.prepare_beams_host(b, LAM)
    for i in range(0, n, max(1, n // 40)):
        one, v1 = lib.prepare_beams_host(b.subset(np.array([i])), LAM)
        a, c = recs[i].copy(), one[0].copy()
        a[31] = c[31] = 0.0                       # the first vertex record
        np.testing.assert_array_equal(a, c)
        np.testing.assert_array_equal(vrecs[b.vert_off[i]:b.vert_off[i + 1]], v1)


def test_more_records_than_pinned_memory():
    th, ph = _angles(5, 4)
    b = random_triangles(80000, seed=3, box=20.0)
    got = lib.diff_main(th, ph, LAM, b, BeamSet.empty(), raw=True)[0]
    np.testing.assert_array_equal(got, _device(th, ph, b))


def test_threads_at_once():
    th, ph = _angles(150, 140)
    b = random_triangles(8, seed=9, box=20.0)
    x, y, z = lib.make_far_field_bins(th, ph)
    want = [lib.diffraction(th, ph, x, y, z, LAM, b, i) for i in range(8)]
    bad = []

    def work(i):
        for _ in range(5):
            if not np.array_equal(lib.diffraction(th, ph, x, y, z, LAM, b, i), want[i]):
                bad.append(i)
    ts = [threading.Thread(target=work, args=(i,)) for i in range(8)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
