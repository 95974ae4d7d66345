"""What the library keeps for a host thread (stream, device buffers, pinned memory) goes to the next thread when that one
ends: calls from threads one after another hold the memory of one."""
import threading

import numpy as np
import pytest

from abt_amd import lib
from abt_amd import visibility as V
from abt_amd.workloads import hex_column_apertures, random_triangles
from tests.test_gpu_host_staging import LAM, _angles

pytestmark = pytest.mark.gpu


def test_threads_one_after_another():
    import torch
    th, ph = _angles(361, 180)          # 4 MiB of results, and as much pinned
    b = random_triangles(3, seed=5, box=20.0)
    xyz = lib.make_far_field_bins(th, ph)
    v, f, ap, apn = hex_column_apertures(10.0, 20.0, 2, 3)
    g = V.VisGeometry.from_mesh(v, f, ap, apn)
    want = lib.diffraction(th, ph, *xyz, LAM, b, 1)
    seen = V.find_vis("inc", g, None, 30.0)["is_vis"]
    bad, free = [], []

    def work(i):
        if not np.array_equal(lib.diffraction(th, ph, *xyz, LAM, b, 1), want):
            bad.append(i)
        if not np.array_equal(V.find_vis("inc", g, None, 30.0)["is_vis"], seen):
            bad.append(i)

    for i in range(32):
        t = threading.Thread(target=work, args=(i,))
        t.start()
        t.join()
        free.append(torch.cuda.mem_get_info()[0])
    assert not bad, bad
    assert free[1] - free[-1] < 16 << 20, (free[1], free[-1])   # one state's: 4.2 MB and up a thread before
