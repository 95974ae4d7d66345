"""abt_far_field_dev without a workspace inside a graph capture, for lists long enough that an eager call cuts
them into segments: the graph holds no buffer of the calling thread, so eager calls after the capture, on a larger grid
(whose segment sums make the thread's buffer grow) and on another stream while the graph replays, change nothing in
its result.  The eager and the captured form differ by the order of a bin's sum only, bounded as in test_gpu_cut by 1e-12 of
the largest amplitude."""
import numpy as np
import pytest

from abt_amd import lib
from abt_amd.workloads import grid, random_triangles

pytestmark = pytest.mark.gpu
LAM = 0.532


@pytest.mark.parametrize("precision", ["fp64", "fp64_fast", "mixed"])
@pytest.mark.parametrize("n", [16, 1023, 1024, 2100])
def test_captured_call_takes_no_thread_buffer(n, precision):
    import torch
    g = lib.DeviceGrid(*grid((0, 9, 180), (0, 17, 340)), LAM)
    big = lib.DeviceGrid(*grid((0, 1, 180), (0, 4, 356)), LAM)
    recs = torch.from_numpy(lib.prepare_beams_host(random_triangles(n, seed=n, box=20.0), LAM)[0]).cuda()
    other = torch.from_numpy(lib.prepare_beams_host(random_triangles(700, seed=1, box=20.0), LAM)[0]).cuda()
    new = lambda q: torch.full((8 * q.nbins,), np.nan, dtype=torch.float64, device="cuda")
    want, out, far = new(g), new(g), new(big)
    lib.far_field_dev(g, recs, n, want, precision=precision)      # warm-up: the thread's buffer exists
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        lib.far_field_dev(g, recs, n, out, precision=precision)
    want = want.cpu().numpy()
    side = torch.cuda.Stream()
    for _ in range(3):
        out.fill_(np.nan)
        torch.cuda.synchronize()
        graph.replay()
        lib.far_field_dev(big, other, 700, far, precision=precision, stream=side)
        torch.cuda.synchronize()
        a = out.cpu().numpy()
        assert np.abs(a - want).max() <= 1e-12 * np.abs(want).max()
