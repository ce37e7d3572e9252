"""The W4A16 ring kernel with 80, 96 and 112 rows to a workgroup (csrc/w4a16_mid.hip), fp16 and bf16 rows staged as fp16, 256 and 512
columns, with and without K splits, and the order in which workgroups take the output tiles: one tile to more row tiles than fit a group,
column tiles that are and are not a multiple of eight, rows and columns that end inside a tile.  Sums that fp32 holds exactly and scales that
are powers of two: bit for bit the oracle's, every element written."""
import numpy as np
import pytest
import torch

from oracle import w4 as ow4
from vllm_gcu_amd.kernels import _custom_ops as ops
from vllm_gcu_amd.kernels.quantization import rearrange

pytestmark = pytest.mark.gpu
CASES = [(1024, 384, 128), (512, 2304, 256), (1152, 128, 1152), (640, 4224, 128), (2048, 1024, 128)]


def _data(K, N, g, M, dtype):
    rng = np.random.default_rng(K + N)
    q = rng.integers(0, 16, size=(K, N), dtype=np.uint8)
    z = rng.integers(0, 16, size=(K // g, N), dtype=np.uint8)
    s = (2.0 ** -rng.integers(4, 8, size=(K // g, N))).astype(np.float32)
    x = rng.integers(-4, 5, size=(M, K)).astype(np.float32)
    w, zp = rearrange.rearrange_uint4_int32_gptq(torch.from_numpy(ow4.gptq_pack_weight(q)).cuda(), torch.from_numpy(ow4.gptq_pack_zeros(z)).cuda())
    bias = rng.integers(-8, 9, size=N).astype(np.float32)
    want = torch.from_numpy(x @ ow4.dequantize(q, z, s, g) + bias).to(dtype)
    return w, zp, torch.from_numpy(s).to(dtype).cuda(), torch.from_numpy(x).to(dtype).cuda(), torch.from_numpy(bias).to(dtype).cuda(), want


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,N,g", CASES)
def test_heights(K, N, g, dtype):
    w, zp, s, x, bias, want = _data(K, N, g, 1300, dtype)
    for mt in (5, 6, 7, 8):
        for M in (65, 16 * mt - 1, 16 * mt, 16 * mt + 1, 333, 1300):
            for tw in (2, 4):
                for split in (1, 2, 3) if dtype == torch.float16 else (1,):
                    print(f"case w4a16 ring rows={16 * mt} tw={tw} split={split} M={M} K={K} N={N} {dtype}", flush=True)
                    out = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
                    ops.w4a16_gemm(x[:M], w, s, zp, bias, g, family=3, split_k=split | tw << 8 | mt << 16, out=out)
                    assert torch.equal(out.cpu(), want[:M])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,N,g", CASES)
def test_two_heights(K, N, g, dtype):
    """Workgroups of 128 rows first and of 112 after them: one of either, rows that end inside the last one, K splits; a number of them that does not
    come out (9 for 1300 rows: all of 128)."""
    w, zp, s, x, bias, want = _data(K, N, g, 1300, dtype)
    for M, rows in ((225, 2), (239, 2), (240, 2), (352, 3), (368, 3), (1237, 11), (1300, 11), (1300, 9)):
        for split in (1, 3) if dtype == torch.float16 else (1,):
            print(f"case w4a16 ring two heights rows={rows} split={split} M={M} K={K} N={N} {dtype}", flush=True)
            out = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
            ops.w4a16_gemm(x[:M], w, s, zp, bias, g, family=3, split_k=split | 4 << 8 | 8 << 16 | rows << 24, out=out)
            assert torch.equal(out.cpu(), want[:M])


@pytest.mark.parametrize("dtype,kind", [(torch.float16, "none"), (torch.bfloat16, "none"), (torch.float16, "pre-scaled")])
def test_heights_and_zero_points(dtype, kind, monkeypatch):
    """No zero-points, and z * s in the activation type read as they are (fp16; bf16 rows with those are not staged)."""
    monkeypatch.setattr(ops, "_RECOVER_INTEGER_ZEROS", False)
    K, N, g = 768, 1408, 128
    w, _, s, x, bias, _ = _data(K, N, g, 333, dtype)
    q = rearrange.unpack_slab(w).cpu().numpy()
    z = np.full((K // g, N), 8, dtype=np.uint8) if kind == "none" else np.random.default_rng(1).integers(0, 16, size=(K // g, N), dtype=np.uint8)
    zs = None if kind == "none" else (torch.from_numpy(z).cuda() * s.float()).to(dtype)
    want = torch.from_numpy(x.float().cpu().numpy() @ ow4.dequantize(q, z, s.float().cpu().numpy(), g) + bias.float().cpu().numpy()).to(dtype)
    for mt in (5, 6, 7, 8):
        for M in (16 * mt + 1, 333):
            for tw in (2, 4):
                print(f"case w4a16 ring {kind} rows={16 * mt} tw={tw} M={M} {dtype}", flush=True)
                out = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
                ops.w4a16_gemm(x[:M], w, s, zs, bias, g, family=3, split_k=1 | tw << 8 | mt << 16, out=out)
                assert torch.equal(out.cpu(), want[:M])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,N,g", CASES)
def test_chosen(K, N, g, dtype):
    """The library's choice, and the 64-row tiles, around the rows where their tiles end."""
    w, zp, s, x, bias, want = _data(K, N, g, 2100, dtype)
    for M in (129, 144, 160, 161, 222, 256, 257, 400, 513, 1025, 2100):
        print(f"case w4a16 chosen M={M} K={K} N={N} {dtype}", flush=True)
        for family in (0, 2):
            out = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
            assert torch.equal(ops.w4a16_gemm(x[:M], w, s, zp, bias, g, family=family, out=out).cpu(), want[:M])


@pytest.mark.parametrize("M,K,N", [(130, 18944, 3584), (333, 28672, 5120), (600, 11008, 5120), (800, 14336, 8192)])
def test_fixed_scratch(M, K, N):
    """Layers that a call with the fixed scratch of 32 MiB has always taken, where K splits that fill the chip would need more: taken, with
    the result of the call that brings a workspace, which a much smaller workspace changes in nothing but the order of additions."""
    from vllm_gcu_amd import _lib
    lib = _lib.load()
    print(f"case w4a16 fixed scratch M={M} K={K} N={N}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(M)
    qw = torch.randint(-2 ** 31, 2 ** 31 - 1, (K * N // 8,), dtype=torch.int32, device="cuda", generator=gen)
    s = torch.rand(K // 128, N, device="cuda", generator=gen).mul_(0.009).add_(0.001).half()
    x = torch.randn(M, K, device="cuda", generator=gen).half()
    st = torch.cuda.current_stream().cuda_stream
    outs = [torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda") for _ in range(3)]
    need = lib.mi355q_w4a16_workspace_bytes(M, K, N)
    for out, size in zip(outs, (need, 3 << 20)):
        ws = torch.zeros(size, dtype=torch.uint8, device="cuda")
        _lib.check(lib.mi355q_w4a16_gemm(out.data_ptr(), x.data_ptr(), qw.data_ptr(), s.data_ptr(), None, _lib.ZP_NONE, None, M, K, N, 128, _lib.F16,
                                         ws.data_ptr(), size, st), "w4a16_gemm")
    _lib.check(lib.mi355q_w4a16_gemm_noalloc(outs[2].data_ptr(), x.data_ptr(), qw.data_ptr(), s.data_ptr(), None, _lib.ZP_NONE, None, M, K, N, 128,
                                             _lib.F16, st), "w4a16_gemm_noalloc")
    assert torch.equal(outs[0], outs[2])
    # (two roundings to fp16 of outputs below 64, and the weights' own, K of them of 2^-12 relative each, averaged)
    torch.testing.assert_close(outs[1].float(), outs[0].float(), rtol=2e-3, atol=3e-2)
