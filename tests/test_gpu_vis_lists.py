"""The visibility set-up and scan where their lists and launches change shape: lists without the triangles that
face away (uncounted runs), few and many beams, set-up and scan on their own, and vertex counts around what a workgroup
keeps in LDS.  Bit-identical to the oracle, as everywhere."""
import numpy as np
import pytest

import oracle as O
from abt_amd import visibility as V
from abt_amd.workloads import hex_column_apertures, random_rotations, vis_workload
from tests.test_gpu_vis import _batch, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["int", "ext", "inc"])
@pytest.mark.parametrize("nbeam", [3, 600])
def test_uncounted_scan_and_its_phases_match_oracle(mode, nbeam):
    """Without counters the lists leave out triangles that face away; frames turned about the particle's own
    axes see many facets exactly or almost edge on.  A set-up and a scan of their own agree with the whole."""
    import torch
    topo, v, mid, nz, apn, ino, fin, bmz = vis_workload(nbeam, mode, seed=21)
    for b in range(0, nbeam, 2):   # edge-on frames: quarter turns, some off by a rounding or a little more
        ang = np.pi / 2 * (b % 4) + (0.0, 1e-16, 1e-15, 1e-9)[b // 2 % 4]
        g = topo.rotated([[np.cos(ang), 0, np.sin(ang)], [0, 1, 0], [-np.sin(ang), 0, np.cos(ang)]])
        v[b], mid[b], nz[b], apn[b] = g.v.T, g.mid, g.nz, g.ap_nz
    args = topo, v, mid, nz, apn, ino, fin, bmz
    print(f"vis uncounted {mode} {nbeam}", flush=True)
    ref, _ = O.find_vis_batch(mode, *args)
    r, _ = _batch(mode, *args, counts=False)
    _same(r, ref, mode)
    dev = torch.device("cuda:0")
    t = lambda a, dt=torch.float64: torch.from_numpy(np.ascontiguousarray(a)).to(dev, dt)  # noqa: E731
    B = V.VisBatch(mode, topo, t(v), t(mid), t(nz), t(apn), t(ino, torch.int64),
                   t(fin if len(fin) else np.zeros(1, np.int64), torch.int64), t(bmz))
    B.run(phases=1)
    B.run(phases=2)
    torch.cuda.synchronize()
    _same({k: x.cpu().numpy() for k, x in B.results().items()}, ref, f"{mode} in phases")
    B.run(phases=2, counts=True)   # after a set-up that left facets out
    in_phase = B.counts.clone()
    B.counts.zero_()
    B.run(counts=True)
    torch.cuda.synchronize()
    assert torch.equal(in_phase, B.counts) and int(B.counts[0]) > 0
    _same({k: x.cpu().numpy() for k, x in B.results().items()}, ref, f"{mode} counted")


@pytest.mark.parametrize("shape,lo,hi", [((14, 28), 3300, 3584), ((20, 40), 3585, 10000)])
def test_vertices_up_to_and_beyond_the_staged_count(shape, lo, hi):
    """Nearly as many vertices as a workgroup keeps in LDS (3584), and more, which are read from memory."""
    v, f, ap, apn = hex_column_apertures(10.0, 20.0, *shape)
    g = V.VisGeometry.from_mesh(v, f, ap, apn)
    assert lo <= g.nv <= hi, g.nv
    for s, mode in enumerate(("int", "ext", "inc")):
        r = g.rotated(random_rotations(1, 40 + s)[0])
        want = r.ap_nz > 0.01 if mode == "int" else r.ap_nz < -0.01
        fi = None if mode == "inc" else np.nonzero(r.ap == np.nonzero(want)[0][0] + 1)[0] + 1
        bz = r.v[:, 2].max() + 1.0
        print(f"vis {r.nv} vertices {mode}", flush=True)
        _same(V.find_vis(mode, r, fi, bz), O.find_vis(mode, r, fi, bz), mode)
