"""The entry points of csrc/w4a16_decode.hip where they need no GPU: plans and refused arguments."""
import os
import subprocess
import sys
from ctypes import byref, c_int

import pytest

from vllm_gcu_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_the_fused_sum_refuses_k_below_a_block():
    """K of less than one block is an error (in a process of its own: it was a division by zero)."""
    code = """
from vllm_gcu_amd import _lib
lib = _lib.load()
for K, N, g in ((64, 128, 64), (192, 128, 64), (128, 192, 128), (128, 128, 64), (127, 128, 127)):
    rc = lib.mi355q_moe_w4a16_unsorted_sum(1, 1, 1, 1, None, _lib.ZP_NONE, g, 1, 1, 0, 4, 2, 8, K, N, _lib.F16, 1, 1 << 30, None)
    assert rc != 0 and b"multiples of 128" in lib.mi355q_last_error(), (K, N, g, rc, lib.mi355q_last_error())
print("refused")
"""
    p = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True)
    assert p.returncode == 0 and p.stdout.strip() == "refused", (p.returncode, p.stdout, p.stderr[-500:])


def plan(M, K, N):
    """(column tiles of a workgroup, its wavefronts, K blocks of a wavefront), zeros for the streaming kernel"""
    out = [c_int() for _ in range(3)]
    _lib.call("mi355q_w4a16_decode_plan", M, K, N, *(byref(v) for v in out))
    return tuple(v.value for v in out)


NOT = (0, 0, 0)


@pytest.mark.parametrize("K,N,to_4,to_8", [(8320, 2048, (1, 16, 5), NOT), (10240, 3072, (1, 16, 5), (1, 16, 5)), (10368, 4096, (1, 16, 6), NOT),
                                           (12288, 2048, (1, 16, 6), NOT), (12416, 2048, NOT, NOT), (12416, 3072, (1, 16, 7), NOT),
                                           (14336, 4096, (1, 16, 7), NOT), (14464, 4096, NOT, NOT), (10240, 4352, (2, 16, 5), NOT),
                                           (10368, 4352, NOT, NOT), (8448, 8192, (2, 16, 5), (2, 16, 5)), (8320, 8320, NOT, NOT), (8320, 1920, NOT, NOT)])
def test_deep_k(K, N, to_4, to_8):
    """On 256 CUs, either side of every line: K blocks and column tiles, up to four rows, up to eight, and none above."""
    assert [plan(M, K, N) for M in (1, 4, 5, 8, 9, 16)] == [to_4, to_4, to_8, to_8, NOT, NOT]


def test_every_plan_is_among_the_shapes_that_are_run():
    """(plan, rows that a load covers) of any layer against what the GPU tests of this kernel run."""
    import test_w4a16_decode_gpu as gpu
    rows = (1, 4, 5, 8, 9, 16)

    def launches(shapes):
        return {(plan(M, K, N), 4 if M <= 4 else 8 if M <= 8 else 16) for K, N in shapes for M in rows} - {(NOT, 4), (NOT, 8), (NOT, 16)}
    planned = launches((K, N) for K in range(128, 16000, 128) for N in range(128, 17000, 256))
    assert len(planned) > 40 and planned <= launches((K, N) for K, N, _ in gpu.SHAPES + gpu.DEEP)
