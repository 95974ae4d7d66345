"""Beam lists cut into segments: the far field of one orientation with a workspace, without one and
inside a graph capture, and the batched plan, at list lengths around the segment and LDS-tile
boundaries.  The cut only regroups a bin's beam sum, so every form agrees with the longest
segments to the rounding of a reordered sum: n 2^-53 of the sum of magnitudes, bounded here by
1e-12 of the largest amplitude (n <= 2100, sums that cancel by less than 10)."""
import numpy as np
import pytest

from abt_amd import lib
from abt_amd.beams import concat
from abt_amd.workloads import grid, random_triangles

pytestmark = pytest.mark.gpu
LAM = 0.532


def _close(a, b):
    assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max(), np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("precision", ["fp64", "fp64_fast", "mixed"])
@pytest.mark.parametrize("n", [1, 31, 33, 64, 95, 1023, 1025, 2100])
def test_far_field_cut(n, precision):
    import torch
    th, ph = grid((0, 9, 180), (0, 17, 340))          # 21 x 21 bins: a partly filled tile
    g = lib.DeviceGrid(th, ph, LAM)
    recs = torch.from_numpy(lib.prepare_beams_host(random_triangles(n, seed=n, box=20.0), LAM)[0]).cuda()
    out = [torch.full((8 * g.nbins,), np.nan, dtype=torch.float64, device="cuda") for _ in range(4)]
    ws = lib.far_field_workspace(g, n, precision)
    assert ws <= 2048 * g.nbins
    work = torch.empty(ws // 8 + 1, dtype=torch.float64, device="cuda")
    lib.far_field_dev(g, recs, n, out[0], precision=precision, work=work if ws else None)
    lib.far_field_dev(g, recs, n, out[1], precision=precision)
    torch.cuda.synchronize()
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(3):                                # one thread, two streams, the library's buffer
        lib.far_field_dev(g, recs, n, out[2], precision=precision, stream=s1)
        lib.far_field_dev(g, recs, n, out[3], precision=precision, stream=s2)
    torch.cuda.synchronize()
    a = [o.cpu().numpy() for o in out]
    assert np.isfinite(a[0]).all()
    for x in a[1:]:
        np.testing.assert_array_equal(x, a[0])
    if n < 1024:                                      # captured without a workspace: nothing is allocated
        out[2].fill_(np.nan)
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            lib.far_field_dev(g, recs, n, out[2], precision=precision)
        for _ in range(3):
            out[2].fill_(np.nan)
            graph.replay()
            torch.cuda.synchronize()
            _close(out[2].cpu().numpy(), a[0])


@pytest.mark.parametrize("precision", ["fp64", "fp64_fast", "mixed", "fp64_accurate"])
def test_batch_cut_matches_single_orientations(precision):
    """The plan's per-orientation amplitudes and Mueller sum against single orientations summed in one
    segment each by a one-beam-tree plan of the same body."""
    import torch
    th, ph = grid((0, 9, 180), (0, 17, 340))
    g = lib.DeviceGrid(th, ph, LAM)
    nb, ne = [32, 0, 65, 130], [33, 96, 0, 1]
    f64 = dict(dtype=torch.float64, device="cuda")
    bl = [random_triangles(max(k, 1), seed=50 + i, box=20.0).subset(np.arange(k)) for i, k in enumerate(nb)]
    el = [random_triangles(max(k, 1), seed=70 + i, box=20.0).subset(np.arange(k)) for i, k in enumerate(ne)]
    rb, re = (torch.from_numpy(lib.prepare_beams_host(concat(x), LAM)[0]).cuda() for x in (bl, el))
    bo, eo = np.concatenate([[0], np.cumsum(nb)]), np.concatenate([[0], np.cumsum(ne)])

    def run(bo, eo, rb, re):
        p = lib.BatchPlan(g, bo, eo, precision)
        n = len(bo) - 1
        m, i, x = torch.empty(16 * g.nbins, **f64), torch.empty(6 * n, **f64), torch.empty(8 * g.nbins * n, **f64)
        p.run(rb, re, m, i, ampl=x)
        torch.cuda.synchronize()
        return m.cpu().numpy(), i.cpu().numpy(), x.cpu().numpy().reshape(n, -1)

    M, I, X = run(bo, eo, rb, re)
    single = [run([0, nb[o]], [0, ne[o]], rb[bo[o]:bo[o + 1]].contiguous(), re[eo[o]:eo[o + 1]].contiguous())
              for o in range(4)]
    for o, (m, i, x) in enumerate(single):
        _close(X[o], x[0])
        np.testing.assert_allclose(I[6 * o:6 * o + 6], i, rtol=0, atol=1e-12 * np.abs(i).max())
    _close(M, sum(s[0] for s in single))
