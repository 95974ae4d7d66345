"""An eager call without a workspace on one stream while another stream is being captured: the thread's buffer it takes
may have to be allocated or grown there, which must neither fail nor invalidate the capture."""
import numpy as np
import pytest

from abt_amd import lib
from abt_amd.workloads import grid, random_triangles

pytestmark = pytest.mark.gpu
LAM = 0.532


@pytest.mark.parametrize("precision", ["fp64", "fp64_fast", "mixed"])
def test_eager_call_beside_a_capture(precision):
    import torch
    n = 500
    recs = torch.from_numpy(lib.prepare_beams_host(random_triangles(n, seed=1, box=20.0), LAM)[0]).cuda()
    grids = [lib.DeviceGrid(*grid((0, 9, 180), (0, 17, 340)), LAM), lib.DeviceGrid(*grid((0, 2, 180), (0, 7, 350)), LAM)]
    want, got = ([torch.full((8 * g.nbins,), np.nan, dtype=torch.float64, device="cuda") for g in grids] for _ in "ab")
    for g, o in zip(grids, want):
        lib.far_field_dev(g, recs, n, o, precision=precision)
    x, side, graph = torch.zeros(4, device="cuda"), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    lib.load().abt_finalize()            # the thread's buffers are gone: the calls below allocate and grow one
    with torch.cuda.graph(graph):
        x.add_(1)
        for g, o in zip(grids, got):
            lib.far_field_dev(g, recs, n, o, precision=precision, stream=side)
    for _ in range(3):
        graph.replay()
    torch.cuda.synchronize()
    assert x.tolist() == [3.0] * 4
    for a, b in zip(got, want):
        assert torch.equal(a, b)
