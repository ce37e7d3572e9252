"""The plans of W4A16 experts on blocks of 64 slots (csrc/w4a16_tile.hip), which need no GPU."""
from ctypes import byref, c_int

import pytest

from vllm_gcu_amd import _lib


def plan(numel, E, K, N, group, zeros, dtype, scratch):
    rows, ranges = c_int(), c_int()
    _lib.call("mi355q_moe_w4a16_plan_scratch", numel, E, K, N, group, zeros, dtype, scratch, byref(rows), byref(ranges))
    return "rows" if rows.value else ranges.value


# us without a workspace, tiles in one range / kernel with copying wavefronts
@pytest.mark.parametrize("E,K,N,rows,dtype", [(1, 11776, 12544, 43, _lib.F16),      # 99.0 / 41.1
                                              (4, 7168, 4096, 40, _lib.F16),        # 62.9 / 26.9
                                              (4, 8704, 13184, 47, _lib.BF16),      # 131.8 / 94.4 (not staged)
                                              (1, 13312, 10368, 83, _lib.F16)])     # 109.9 / 55.1
def test_ranges_without_room_are_no_reason_for_tiles(E, K, N, rows, dtype):
    with_room = plan(E * rows, E, K, N, 128, _lib.ZP_NONE, dtype, 1)
    assert with_room != "rows" and with_room > 1
    assert plan(E * rows, E, K, N, 128, _lib.ZP_NONE, dtype, 0) == "rows"


@pytest.mark.parametrize("group,zeros", [(128, _lib.ZP_PACKED), (64, _lib.ZP_PACKED), (32, _lib.ZP_NONE), (128, _lib.ZP_PRESCALED)])
def test_nothing_is_cut_without_a_workspace(group, zeros):
    for E in (1, 8, 60):
        for rows in (29, 64, 250):
            for K, N in ((1024, 1024), (4096, 28672), (14336, 4096), (12800, 1152)):
                for dtype in (_lib.F16, _lib.BF16):
                    assert plan(E * rows, E, K, N, group, zeros, dtype, 0) in ((1,) if group == 32 else (1, "rows"))
