"""The align block size that an expert layer takes: W4A16 experts whose kernel takes blocks by their live row tiles (groups other
than 32) leave the blocks of 16 slots above 12 rows per expert, every other kind above 16."""
import pytest

from vllm_gcu_amd.kernels.fused_moe import get_default_config
from vllm_gcu_amd.kernels.modular_experts import TritonExpertsPad

KINDS = [(dict(use_int4_w4a16=True, block_shape=[0, 128]), 12), (dict(use_int4_w4a16=True, block_shape=[0, 64]), 12),
         (dict(use_int4_w4a16=True, block_shape=[0, -1]), 12), (dict(use_int4_w4a16=True, block_shape=[0, 32]), 16),
         (dict(use_int8_w8a16=True, block_shape=[0, 128]), 16), (dict(use_int8_w8a16=True, block_shape=[0, -1]), 16),
         (dict(use_fp8_w8a8=True, block_shape=[128, 128]), 16), (dict(use_int8_w8a8=True), 16)]


@pytest.mark.parametrize("kind,rows", KINDS)
def test_rows_per_expert_that_leave_blocks_of_16(kind, rows):
    experts = TritonExpertsPad(**kind)

    def block(per_expert):
        return get_default_config(M=4 * per_expert, E=8, N=28672, K=4096, topk=2, dtype=experts.config_dtype, is_marlin=False,
                                  block_shape=experts.block_shape)["BLOCK_SIZE_M"]
    assert [block(r) for r in (1, rows, rows + 1, 28)] == [16, 16, 32, 32]
