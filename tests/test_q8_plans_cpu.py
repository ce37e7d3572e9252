"""The plans of the 8-bit kernel for a few dozen to some hundred rows (csrc/q8_mid.hip), which need no GPU."""
from ctypes import byref, c_int

import pytest
import torch

from vllm_gcu_amd import _lib

LAYERS = [(7168, 4096), (8192, 8192), (4096, 6144), (4096, 28672), (8192, 10240), (2048, 7168), (3584, 4608), (5120, 13824), (14336, 4096),
          (18944, 3584), (11008, 4096), (28672, 8192), (6144, 2048), (1024, 1024), (1536, 6656), (1024, 5120)]       # (K, N)


def tile(kind, M, N, K):
    out = [c_int() for _ in range(3)]
    _lib.call("mi355q_q8_mid_tile", kind, M, N, K, *(byref(v) for v in out))
    return tuple(v.value for v in out)


@pytest.mark.parametrize("kind", [0, 1, 2])
def test_every_tile_is_taken_somewhere(kind):
    """What is built is also chosen: fp8 with block scales (which alone has 144 and 160 rows), fp8 and int8 with scales outside the K sum."""
    rows = {tile(kind, M, N, K)[0] for K, N in LAYERS for M in range(17, 1537)}
    assert rows == {0, 32, 48, 64, 80, 96, 112, 128} | ({144, 160} if kind == 0 else set())


def int8_plan(M, N, K, kslab=True):
    """(kernel, K ranges): 0 = csrc/q8_mid.hip, 1 = the tiles of csrc/fp8_block_tile.hip, 2 = the tiles of csrc/w8a8_int8.hip"""
    kernel, ranges = c_int(), c_int()
    _lib.call("mi355q_w8a8_int8_plan", M, N, K, kslab, byref(kernel), byref(ranges))
    return kernel.value, ranges.value


def tile_plan(kind, M, N, K):
    """(rows of a tile, K ranges) of the kernel for more rows, csrc/fp8_block_tile.hip"""
    rows, ranges = c_int(), c_int()
    _lib.call("mi355q_q8_tile_plan", kind, M, N, K, byref(rows), byref(ranges))
    return rows.value, ranges.value


@pytest.mark.parametrize("kind", [0, 1, 2])
def test_every_height_is_taken_somewhere(kind):
    heights = {tile_plan(kind, M, N, K)[0] for K, N in LAYERS for M in range(65, 2049, 9) if tile(kind, M, N, K)[0] == 0}
    assert heights == {128, 160, 192, 224, 256}


def test_the_int8_kernel_is_the_one_that_the_others_were_compared_with():
    """Where the prices of the two tile kernels are close, the 8-bit kernel for some hundred rows gives way to the one that is launched: the
    128-column tiles here (us, 8-bit kernel / 128-column tiles / 256 rows: K 3456 x N 20096 at 362 rows 49.6 / 42.1 / 44.9)."""
    assert int8_plan(335, 19968, 3712) == (1, 1)
    assert int8_plan(362, 20096, 3456) == (1, 1)
    assert int8_plan(594, 26112, 1408) == (1, 1)


def test_no_plan_outside_the_range():
    for M, N, K in ((16, 4096, 4096), (1537, 4096, 4096), (64, 4096 + 32, 4096)):
        assert tile(1, M, N, K) == (0, 0, 0)
    with pytest.raises(RuntimeError, match="bad shape"):
        tile(3, 64, 4096, 4096)


def way(kind, M, N, K, scratch=1):
    """(tile, K ranges, added in the kernel)"""
    out = [c_int() for _ in range(3)]
    _lib.call("mi355q_q8_mid_way", kind, M, N, K, scratch, *(byref(v) for v in out))
    return out[0].value, out[1].value, bool(out[2].value)


NO_ROOM = [(0, 49, 128, 1792), (0, 64, 256, 1792), (0, 100, 128, 1792), (0, 128, 128, 1792), (2, 49, 256, 2688), (2, 52, 256, 2688), (2, 76, 128, 2688)]


# us without a workspace, tiles of 256 rows / here: 9.6 / 5.4, 9.9 / 5.6, 10.7 / 5.5, 11.1 / 5.5, 13.1 / 6.3, 13.2 / 6.3, 13.6 / 6.2
@pytest.mark.parametrize("kind,M,N,K", NO_ROOM)
def test_ranges_without_room_do_not_lose_the_kernel(kind, M, N, K):
    tile_, ranges, _ = way(kind, M, N, K)
    assert tile_ in (0, 1) and ranges > 1
    assert way(kind, M, N, K, 0) == (3, 1, False)


def test_what_needs_no_room_is_the_same_without():
    for kind in range(3):
        for K, N in LAYERS:
            for M in range(1, 1600, 7):
                w = way(kind, M, N, K)
                without = way(kind, M, N, K, 0)
                assert without == w if w[1] <= 1 else without[1] <= 1


# rows that the kernel for few rows takes, and what runs of the same layer where it does not
FEW = [(0, 33, 1408, 3712), (0, 31, 128, 2048), (0, 48, 4096, 2048), (1, 23, 4096, 4096), (1, 32, 1024, 2048), (2, 28, 4096, 4096), (2, 40, 4096, 1408), (2, 64, 8192, 1024)]


@pytest.mark.parametrize("kind,M,N,K", FEW)
def test_the_plans_state_the_kernel_for_few_rows(kind, M, N, K):
    assert way(kind, M, N, K) == way(kind, M, N, K, 0) == (12, 1, False)
    rows, columns, ranges = tile(kind, M, N, K)
    assert rows == (M + 15) // 16 * 16 and columns % 16 == 0 and -(-N // columns) <= 256 and ranges == 1
    assert kind != 2 or int8_plan(M, N, K) == (0, 1)
    assert way(kind, 65, N, K)[0] not in (-1, 12)


@pytest.mark.parametrize("kind,M,N,K", [(0, 36, 8192, 3200), (0, 40, 5248, 3200), (2, 24, 8320, 3584), (2, 32, 9216, 2176), (2, 17, 9216, 3072)])
def test_rows_that_the_tiles_are_ahead_on(kind, M, N, K):
    """us, the kernel for few rows / the tiles, the weights in the cache: 8.6 / 7.9, 7.9 / 7.9, 8.6 / 7.7, 6.8 / 6.6, 7.8 / 7.5."""
    assert way(kind, M, N, K)[0] in range(12)


def _launches(shapes):
    for kind, M, N, K in shapes:
        t, ranges, in_kernel = way(kind, M, N, K)
        if t >= 0:
            yield kind, t, "whole" if ranges == 1 else "added in the kernel" if in_kernel else "second launch"


def test_every_launch_of_the_plans_is_among_the_shapes_that_are_run():
    """(kind, tile, how its K ranges are added): what the plans of a wide range of layers take against what the GPU tests run."""
    import test_q8_mid_gpu as gpu
    wide = LAYERS + [(K, N) for N in (64, 128, 192, 256, 384, 640, 1024, 1152, 1408, 2176, 2432, 3072, 4096)
                     for K in (384, 1024, 1408, 2048, 3072, 3968, 5120, 6400, 8192, 9088, 10240, 10880, 14336)]
    rows = [*range(17, 130), *range(130, 1537, 11)]
    planned = set(_launches((kind, M, N, K) for kind in range(3) for K, N in wide if kind or N % 128 == 0 for M in rows))
    run = set(_launches([(kind, *s) for kind in range(3) for s in gpu.SHAPES if kind == gpu.INT8 or s[1] % 128 == 0] +
                        [s[:4] for s in gpu.RANGES] + gpu.MORE))
    assert len(planned) > 50 and planned <= run, sorted(planned - run)


@pytest.mark.skipif(torch.cuda.device_count() > 0, reason="launches on addresses that are none")
@pytest.mark.parametrize("kind", [0, 1, 2])
def test_the_kernel_for_few_rows_is_built_for_every_call_it_is_chosen_for(kind):
    """Every launch that the rules ask for, codes in both weight layouts and rows quantised in the launch: without a GPU each ends at the device, not at a launch that
    is not there."""
    lib = _lib.load()
    columns = [64, 320, 4096, 4224, 6144, 8192, 8320, 11008, 12288, 12544, 14336, 16384, 16512, 20480, 28672, 32768]
    seen = set()

    def ends_at_the_device(rc):
        error = lib.mi355q_last_error().decode()
        assert rc != 0 and "device" in error, error
        seen.add("few" if "q8_decode" in error else "other")
    for N in columns:
        for K in [*range(128, 8192, 128), 10240, 16384, 20480, 28672, 65536]:
            if N * K >= 1 << 31:
                continue
            for M in (1, 2, 3, 5, 8, 9, 16, 17, 20, 24, 25, 32, 33, 36, 40, 41, 48, 49, 56, 64):
                for kslab in (0, 1) if M <= 16 else (1,):
                    if kind == 1:
                        ends_at_the_device(lib.mi355q_fp8_scaled_gemm(4096, 4096, 4096, 4096, 1, 4096, 1, None, M, N, K, K, 0 if kslab else K, N, _lib.BF16, None))
                    else:
                        ends_at_the_device(lib.mi355q_kcontig_gemm(4096, 4096, 4096, 4096, 4096, None, 1 + kind // 2, 128, M, K, N, _lib.F16, _lib.BF16, kslab, None))
                for quant in (1, 2):
                    if lib.mi355q_q8_quant_gemm_takes(kind, quant, M, N, K):
                        ends_at_the_device(lib.mi355q_q8_quant_gemm(4096, 4096, 4096, 4096, 4096, 1, None, kind, quant, M, N, K, _lib.BF16, None))
    assert seen == {"few", "other"}
