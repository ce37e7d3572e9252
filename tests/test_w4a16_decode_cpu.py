"""The entry points of csrc/w4a16_decode.hip where they need no GPU: refused arguments."""
import os
import subprocess
import sys

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
