"""A row that holds infinities (and so an infinite group scale) reaches its own outputs only: every other row's output is, bit
for bit, that of the same problem with finite values in that row.  The problems have more output tiles than CUs, so that
workgroups go from one row tile to another, and the row lies where a wavefront's running products outlast its tile."""
import pytest
import torch

from vllm_gcu_amd.kernels import _custom_ops as ops
from vllm_gcu_amd.kernels import _runtime as rt
from vllm_gcu_amd.kernels import fused_moe as fmoe

pytestmark = pytest.mark.gpu
BAD = 117            # in the last two 16-row tiles of a wavefront's share, for tiles of 256 rows and of 128


def _fp8(gen, *shape):
    return (torch.randn(*shape, device="cuda", generator=gen) * 50).to(torch.float8_e4m3fn)


def _others_equal(got, want, bad):
    keep = torch.ones(got.shape[0], dtype=torch.bool, device=got.device)
    keep[bad] = False
    assert torch.isfinite(want).all()
    assert torch.equal(got[keep], want[keep])


# rows and columns for: tiles of 128 rows with the column tiles dealt out over the XCDs, of 256 with and without, of 128 without
@pytest.mark.parametrize("M,N,K", [(1537, 7168, 256), (2304, 7168, 256), (768, 21760, 256), (700, 12800, 384)])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_fp8_block_scales(M, N, K, value):
    print(f"case rows apart fp8 block M={M} N={N} K={K} {value}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(M)
    x, w = _fp8(gen, M, K), _fp8(gen, N, K)
    xs, ws = torch.rand(M, K // 128, device="cuda", generator=gen), torch.rand(N // 128, K // 128, device="cuda", generator=gen) * 1e-4
    outs = []
    for v in (value, 1.0):
        xs[BAD, -1] = v
        out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
        torch.ops._C.linear_quant(out, x, w, None, xs, ws)      # (row-major weights: the tile kernel)
        outs.append(out)
    _others_equal(outs[0], outs[1], BAD)
    assert not torch.isfinite(outs[0][BAD]).any()


@pytest.mark.parametrize("block", [256, 128])
@pytest.mark.parametrize("bad", [BAD, -1])           # (pads read the last token's row)
def test_fp8_block_scales_grouped(block, bad):
    print(f"case rows apart fp8 grouped block={block} bad={bad}", flush=True)
    N, K, rows = 7168, 256, [256, 300, 512, 270]
    E, M = len(rows), sum(rows)
    gen = torch.Generator(device="cuda").manual_seed(block)
    x, w = _fp8(gen, M, K), _fp8(gen, E, N, K)
    xs = torch.rand(M, K // 128, device="cuda", generator=gen)
    ws = torch.rand(E, N // 128, K // 128, device="cuda", generator=gen) * 1e-4
    ids = torch.repeat_interleave(torch.arange(E, device="cuda", dtype=torch.int32), torch.tensor(rows, device="cuda"))[:, None].contiguous()
    sid, eid, npp = fmoe.moe_align_block_size(ids, block, E, None, None)
    outs = []
    for v in (float("inf"), 1.0):
        xs[bad, -1] = v
        out = torch.zeros(M, 1, N, dtype=torch.bfloat16, device="cuda")
        fmoe.invoke_fused_moe_kernel(x, w, out, xs, ws, None, torch.ones(M, 1, device="cuda"), ids, sid, eid, npp, False, 1,
                                     {"BLOCK_SIZE_M": block}, use_fp8_w8a8=True, use_int8_w8a8=False, use_int8_w8a16=False,
                                     use_int4_w4a16=False, block_shape=[128, 128])
        outs.append(out.view(M, N))
    _others_equal(outs[0], outs[1], bad)
