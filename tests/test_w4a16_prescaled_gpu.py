"""Pre-scaled zero-points that are no integer times the scale are taken as given, w = q * s - zeros, by every kernel that the
library picks -- dense from one row to prefill, grouped at every block size, groups of 128, 64 and 32 -- and a scale of 0 gives
weights of -zeros (0 where they are 0), not NaN."""
import numpy as np
import pytest
import torch

from oracle import moe as om
from oracle import w4 as ow4
from vllm_gcu_amd.kernels import _custom_ops as ops
from vllm_gcu_amd.kernels import fused_moe as fmoe
from vllm_gcu_amd.kernels.quantization import rearrange

pytestmark = pytest.mark.gpu


def _weights(rng, K, N, g, dtype):
    q = rng.integers(0, 16, size=(K, N), dtype=np.uint8)
    s = rng.uniform(0.001, 0.01, size=(K // g, N)).astype(np.float32)
    s[:, ::7] = 0.0                                     # a scale of 0 with zero-points of 0 and (below) of something else
    z = rng.uniform(0.0, 15.0, size=(K // g, N))        # not integers
    z[:, 1::5] = rng.integers(0, 16, size=z[:, 1::5].shape)          # integers beside them, of exact products
    s[:, 1::5] = 2.0 ** -rng.integers(7, 10, size=s[:, 1::5].shape)
    z[:, 2::11] = rng.uniform(-4.0, 24.0, size=z[:, 2::11].shape)    # out of the range of int4
    s = torch.from_numpy(s).to(dtype)
    zs = (torch.from_numpy(z.astype(np.float32)) * s.float()).to(dtype)
    zs[:, ::21] = 0.01
    return q, s, zs


# Weights are read exactly or (ring kernels) rounded to 16 bits, sums are fp32, the result is rounded once to 16 bits: 2^-8 of the
# value at most, and 2^-11 of weights up to 0.24 over sqrt(K) terms near zero (0.004 at K = 1024).  A zero-point that is bit for
# bit an integer times the scale, rounded -- some fractions round to one, too -- may be read as that integer: `slack` is the
# rounding times the sum of the group's activations.  An integer read in the place of any other fraction is 0.25 s off on average:
# 0.04 rms.
def _slack(s, zs, x, g):
    sf, zf = s.float(), zs.float()
    z = torch.nan_to_num(torch.round(zf / sf), 0.0, 15.0, 0.0).clamp(0, 15)
    near = torch.where((z * sf).to(zs.dtype) == zs, (z * sf - zf).abs(), torch.zeros(()))
    return (x.float().view(x.shape[0], -1, g).sum(-1).abs() @ near).numpy()


def _close(got, want, slack):
    got = got.float().cpu().numpy()
    assert (np.abs(got - want) <= 1e-2 + 1e-2 * np.abs(want) + slack).all(), np.abs(got - want).max()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N,g", [(3, 1024, 512, 128), (40, 1024, 512, 128), (100, 1024, 512, 128), (100, 1024, 512, 64), (100, 1024, 512, 32),
                                     (128, 1024, 384, 1024), (300, 1024, 512, 128), (300, 512, 2048, 32), (700, 1024, 4096, 128),
                                     (2100, 512, 2048, 128), (2100, 512, 2048, 64)])
def test_dense(M, K, N, g, dtype):
    print(f"case w4a16 prescaled M={M} K={K} N={N} g={g} {dtype}", flush=True)
    rng = np.random.default_rng(M + g)
    q, s, zs = _weights(rng, K, N, g, dtype)
    w, _ = rearrange.rearrange_uint4_int32_gptq(torch.from_numpy(ow4.gptq_pack_weight(q)).cuda(), None)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(dtype)
    want = x.float().numpy() @ ow4.dequantize_prescaled_zeros(q, zs.float().numpy(), s.float().numpy(), g)
    _close(ops.w4a16_gemm(x.cuda(), w, s.cuda(), zs.cuda(), None, g), want, _slack(s, zs, x, g))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("block,K,N,g", [(16, 512, 256, 128), (16, 512, 256, 64), (32, 512, 256, 128), (32, 512, 256, 64), (32, 512, 256, 32),
                                         (64, 512, 256, 128), (64, 4096, 128, 128), (64, 512, 256, 64), (128, 512, 256, 128), (128, 512, 256, 32)])
def test_grouped(block, K, N, g, dtype):
    print(f"case w4a16 prescaled grouped block={block} K={K} N={N} g={g} {dtype}", flush=True)
    rng = np.random.default_rng(block + K + g)
    M, E, T = 60, 3, 2
    parts = [_weights(rng, K, N, g, dtype) for _ in range(E)]
    w, _ = rearrange.rearrange_uint4_int32_gptq(torch.from_numpy(np.stack([ow4.gptq_pack_weight(p[0]) for p in parts])).cuda(), None)
    s, zs = torch.stack([p[1] for p in parts]).cuda(), torch.stack([p[2] for p in parts]).cuda()
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(dtype)
    tw, ids, _ = om.topk_softmax(rng.standard_normal((M, E)).astype(np.float32), T, True)
    dev_ids = torch.from_numpy(np.ascontiguousarray(ids, dtype=np.int32)).cuda()
    sid, eid, npp = fmoe.moe_align_block_size(dev_ids, block, E, None, None)
    out = torch.empty((M, T, N), dtype=dtype, device="cuda")
    fmoe.invoke_fused_moe_kernel(x.cuda(), w, out, None, s, zs, torch.from_numpy(tw).cuda(), dev_ids, sid, eid, npp, False, T,
                                 {"BLOCK_SIZE_M": block}, use_fp8_w8a8=False, use_int8_w8a8=False, use_int8_w8a16=False,
                                 use_int4_w4a16=True, block_shape=[0, g])
    want = om.fused_moe_gemm(x.float().numpy(), lambda e: ow4.dequantize_prescaled_zeros(parts[e][0], parts[e][2].float().numpy(),
                                                                                         parts[e][1].float().numpy(), g), ids, T)
    slack = np.stack([_slack(p[1], p[2], x, g) for p in parts])
    _close(out.view(-1, N), want, np.stack([slack[e, i // T] for i, e in enumerate(ids.reshape(-1))]))
