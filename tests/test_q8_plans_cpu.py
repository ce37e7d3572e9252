"""The plans of the 8-bit kernel for a few dozen to some hundred rows (csrc/q8_mid.hip), which need no GPU."""
from ctypes import byref, c_int

import pytest

from vllm_gcu_amd import _lib

LAYERS = [(7168, 4096), (8192, 8192), (4096, 6144), (4096, 28672), (8192, 10240), (2048, 7168), (3584, 4608), (5120, 13824), (14336, 4096),
          (18944, 3584), (11008, 4096), (28672, 8192), (6144, 2048), (1024, 1024), (1536, 6656), (1024, 5120)]       # (K, N)


def tile(kind, M, N, K):
    out = [c_int() for _ in range(3)]
    _lib.call("mi355q_q8_mid_tile", kind, M, N, K, *(byref(v) for v in out))
    return tuple(v.value for v in out)


@pytest.mark.parametrize("kind", [0, 1, 2])
def test_every_tile_is_taken_somewhere(kind):
    """What is built is also chosen: fp8 with block scales, fp8 and int8 with scales outside the K sum."""
    rows = {tile(kind, M, N, K)[0] for K, N in LAYERS for M in range(17, 1537)}
    assert rows == {0, 32, 48, 64, 80, 96, 112, 128, 144, 160}


def test_no_plan_outside_the_range():
    for M, N, K in ((16, 4096, 4096), (1537, 4096, 4096), (64, 4096 + 32, 4096)):
        assert tile(1, M, N, K) == (0, 0, 0)
    with pytest.raises(RuntimeError, match="bad shape"):
        tile(3, 64, 4096, 4096)
