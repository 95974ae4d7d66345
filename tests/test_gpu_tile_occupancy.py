"""The batched plan's tile shapes keep the waves that their registers were laid out for: four workgroups on a CU (one
wave of each on a SIMD) with one bin a lane, three with two; two for the accurate body."""
import pytest

from abt_amd import lib
from abt_amd.workloads import grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tb,bpt,waves", [
    ("fp64_fast", 8, 1, 4), ("fp64_fast", 16, 1, 4), ("fp64_fast", 32, 1, 4), ("fp64_fast", 8, 2, 3),
    ("fp64_fast", 16, 2, 3), ("fp64", 16, 1, 4), ("fp64", 16, 2, 3), ("mixed", 32, 1, 4), ("mixed", 8, 2, 3),
    ("mixed_gated", 16, 1, 4), ("fp64_accurate", 16, 1, 2)])
def test_workgroups_a_cu(precision, tb, bpt, waves):
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    g = lib.DeviceGrid(*grid((0, 30, 180), (0, 60, 300)), 0.532)
    p = lib.BatchPlan(g, [0, 8], [0, 8], precision)
    p.set_tiles(tb, bpt)
    assert p.tiles()["workgroups"] >= waves * cus
    p.close()
