"""The grouped form of the W4A16 kernel with copying wavefronts (csrc/w4a16_rows.hip): blocks of 32 and 64 slots that hold
one to four row tiles and their edges, experts with no rows and with several blocks, experts of other ranks, odd numbers
of K blocks, groups of 64 to K, every kind of zero-points, both forms of the expert GEMM."""
import numpy as np
import pytest
import torch

from oracle import moe as om
from oracle import w4 as ow4
from vllm_gcu_amd.kernels import _custom_ops as ops
from vllm_gcu_amd.kernels import fused_moe as fmoe
from vllm_gcu_amd.kernels.quantization import rearrange

pytestmark = pytest.mark.gpu
ROWS = {32: [0, 1, 15, 16, 17, 31, 32, 33], 64: [0, 1, 16, 17, 32, 33, 47, 48, 49, 64, 66]}     # rows of each expert


@pytest.mark.parametrize("zeros", ["packed", "prescaled", None])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("block,K,N,g", [(32, 128, 128, 128), (32, 640, 256, 64), (32, 1024, 384, 1024), (64, 4096, 256, 256), (64, 4224, 128, 64)])
def test_blocks_of_every_fill(block, K, N, g, dtype, zeros, monkeypatch):
    print(f"case w4a16 rows grouped block={block} K={K} N={N} g={g} {dtype} zeros={zeros}", flush=True)
    monkeypatch.setattr(ops, "_RECOVER_INTEGER_ZEROS", False)
    rng = np.random.default_rng(block + K)
    rows, T = ROWS[block] + [5], 2                     # the last expert is another rank's
    E = len(rows) - 1
    ids = rng.permutation(np.repeat(np.arange(E + 1, dtype=np.int32), rows))
    ids = np.append(ids, [E] * (ids.size % T)).astype(np.int32).reshape(-1, T)
    M = len(ids)
    tw = rng.uniform(0.1, 1.0, ids.shape).astype(np.float32)
    q = rng.integers(0, 16, size=(E, K, N), dtype=np.uint8)
    z = rng.integers(0, 16, size=(E, K // g, N), dtype=np.uint8) if zeros else None
    s = torch.from_numpy(rng.uniform(0.001, 0.01, size=(E, K // g, N)).astype(np.float32)).to(dtype)
    sf = s.float().numpy()
    w, zp = rearrange.rearrange_uint4_int32_gptq(torch.from_numpy(np.stack([ow4.gptq_pack_weight(e) for e in q])).cuda(),
                                                 torch.from_numpy(np.stack([ow4.gptq_pack_zeros(e) for e in z])).cuda() if zeros else None)
    if zeros == "prescaled":
        zp = (torch.from_numpy(z.astype(np.float32)) * s.float()).to(dtype).cuda()
    dense = [ow4.dequantize(q[e], z[e] if zeros else None, sf[e], g) for e in range(E)] + [np.zeros((K, N), np.float32)]
    emap = torch.tensor(list(range(E)) + [-1], dtype=torch.int32)
    dev_ids = torch.from_numpy(ids).cuda()
    sid, eid, npp = fmoe.moe_align_block_size(dev_ids, block, E + 1, emap.cuda(), None)
    for topk, weighted in ((T, False), (1, True)):     # rows shared by a token's slots; a row per slot and its routing weight
        x = torch.from_numpy(rng.standard_normal((M * T // topk, K)).astype(np.float32)).to(dtype)
        out = torch.full((M, T, N), float("nan"), dtype=dtype, device="cuda")
        fmoe.invoke_fused_moe_kernel(x.cuda(), w, out, None, s.cuda(), zp, torch.from_numpy(tw).cuda(), dev_ids, sid, eid, npp, weighted,
                                     topk, {"BLOCK_SIZE_M": block}, use_fp8_w8a8=False, use_int8_w8a8=False, use_int8_w8a16=False,
                                     use_int4_w4a16=True, block_shape=[0, g])
        want = om.fused_moe_gemm(x.float().numpy(), lambda e: dense[e], ids, topk, tw if weighted else None, weighted)
        np.testing.assert_allclose(out.view(-1, N).float().cpu().numpy(), want, rtol=1e-2, atol=1e-2)
