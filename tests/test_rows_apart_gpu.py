"""A row that holds infinities or NaN (and so an infinite group scale) reaches its own outputs only: every other row's output is,
bit for bit, that of the same problem with finite values in that row.  The problems of the 256-row tile kernel have more output
tiles than CUs, so that workgroups go from one row tile to another, and the row lies where a wavefront's running products outlast
its tile."""
import pytest
import torch

from vllm_gcu_amd.kernels import _custom_ops as ops
from vllm_gcu_amd.kernels import _runtime as rt
from vllm_gcu_amd.kernels import fused_moe as fmoe
from vllm_gcu_amd.kernels.quantization import rearrange

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


# (rows, columns, K) that the 8-bit kernel for some hundred rows takes with its tiles of 32 to 128 rows, whole K and in ranges
@pytest.mark.parametrize("M,N,K", [(31, 256, 128), (48, 1024, 7168), (65, 1024, 1024), (200, 2048, 1408), (512, 8192, 2048), (1024, 4096, 4096)])
@pytest.mark.parametrize("block", [True, False])
def test_fp8_some_hundred_rows(M, N, K, block):
    print(f"case rows apart fp8 mid M={M} N={N} K={K} block={block}", flush=True)
    assert rt.host.q8_mid_plan(0 if block else 1, M, N, K) >= 0
    gen = torch.Generator(device="cuda").manual_seed(M)
    x, w = _fp8(gen, M, K), rearrange.to_kslab(_fp8(gen, N, K))
    xs, ws = torch.rand(M, K // 128, device="cuda", generator=gen), torch.rand(N // 128, K // 128, device="cuda", generator=gen) * 1e-4
    bad, code = M // 2, x[M // 2, 3].clone()
    outs = []
    for v, c in ((float("inf"), torch.tensor(float("nan"), device="cuda").to(x.dtype)), (1.0, code)):
        xs[bad, -1], x[bad, 3] = v, c
        out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
        if block:
            torch.ops._C.linear_quant(out, x, w, None, xs, ws)
        else:
            torch.ops._C.cutlass_scaled_mm(out, x, w.t(), xs[:, -1:].contiguous(), ws[:1, :1], None)
        outs.append(out)
    _others_equal(outs[0], outs[1], bad)


def _int4(gen, *lead, K, N, g):
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (*lead, K // 8, N), device="cuda", generator=gen, dtype=torch.int32)
    z = torch.randint(-2 ** 31, 2 ** 31 - 1, (*lead, K // g, N // 8), device="cuda", generator=gen, dtype=torch.int32)
    return w, z, torch.rand(*lead, K // g, N, device="cuda", generator=gen) * 0.01


@pytest.mark.parametrize("mt,nt", [(2, 1), (3, 1), (4, 1), (2, 2), (3, 2), (4, 2), (5, 2), (6, 2)])
@pytest.mark.parametrize("kind", ["packed", "fractions"])
def test_int4_some_hundred_rows(mt, nt, kind):
    M, N, K, g = 40 * mt, 256, 640, 64
    print(f"case rows apart w4a16 rows {16 * mt}x{64 * nt} {kind}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(mt)
    w, z, s = _int4(gen, K=K, N=N, g=g)
    for dtype in (torch.float16, torch.bfloat16):
        x, sd = torch.randn(M, K, device="cuda", generator=gen).to(dtype), s.to(dtype)
        zeros = z if kind == "packed" else (sd.float() * 7.4).to(dtype)
        outs = []
        for v in (float("inf"), 1.0):
            x[M // 2, K - 3] = v
            outs.append(ops.w4a16_gemm(x, w, sd, zeros, None, g, family=4, split_k=1 | mt << 8 | nt << 16))
        _others_equal(outs[0], outs[1], M // 2)


@pytest.mark.parametrize("block", [32, 64])
def test_int4_some_hundred_rows_grouped(block):
    print(f"case rows apart w4a16 rows grouped block={block}", flush=True)
    E, T, M, K, N, g = 4, 2, 60, 4096, 256, 128
    gen = torch.Generator(device="cuda").manual_seed(block)
    w, z, s = _int4(gen, E, K=K, N=N, g=g)
    s = s.half()
    x = torch.randn(M, K, device="cuda", generator=gen).half()
    ids = torch.stack([torch.randperm(E, device="cuda", generator=gen)[:T] for _ in range(M)]).int().contiguous()
    sid, eid, npp = fmoe.moe_align_block_size(ids, block, E, None, None)
    for bad in (M // 2, M - 1):                      # (pads read the last token's row)
        outs, keep = [], x[bad, 9].clone()
        for v in (float("inf"), keep):
            x[bad, 9] = v
            out = torch.empty(M, T, N, dtype=torch.float16, device="cuda")
            fmoe.invoke_fused_moe_kernel(x, w, out, None, s, z, torch.ones(M, T, device="cuda"), ids, sid, eid, npp, False, T,
                                         {"BLOCK_SIZE_M": block}, use_fp8_w8a8=False, use_int8_w8a8=False, use_int8_w8a16=False,
                                         use_int4_w4a16=True, block_shape=[0, g])
            outs.append(out)
        _others_equal(outs[0], outs[1], bad)
