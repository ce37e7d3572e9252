"""The 8-bit GEMMs on tiles of 128 .. 256 rows (csrc/fp8_block_tile.hip): row counts on both sides of every tile height, odd and
even numbers of K blocks, row-major weights (for int8 csrc/w8a8_int8.hip takes a few of them, for fp8 nothing else does at these rows); kslab
weights, which csrc/q8_mid.hip takes at many of those shapes, at shapes that it leaves to every height, with one and with several K ranges.
int8 is exact; fp8 is compared with a float64 product."""
import pytest
import torch

from test_q8_plans_cpu import int8_plan, tile, tile_plan
from vllm_gcu_amd import _lib
from vllm_gcu_amd.kernels.quantization import rearrange

pytestmark = pytest.mark.gpu
# (M, N, K).  256 column tiles: one round holds one row tile, so the height is the smallest multiple of 32 that holds M
SHAPES = [(m, 32768, k) for m, k in ((96, 128), (128, 256), (129, 384), (160, 128), (161, 256), (192, 384), (193, 128), (224, 640), (225, 256),
                                     (256, 384), (257, 128))]
SHAPES += [(320, 16384, 256), (448, 16384, 384), (1537, 4096, 896), (700, 14336, 256), (130, 2048, 4096), (333, 1024, 6144), (1600, 128, 128)]
# kslab weights: (rows of a tile, K ranges) -> shape
SERVED = {(128, 1): (1800, 1024, 640), (160, 1): (1543, 2560, 640), (192, 1): (337, 11008, 640), (224, 1): (197, 16512, 640),
          (256, 1): (455, 11008, 640), (128, 2): (1598, 128, 2048), (160, 5): (1540, 512, 5120), (192, 3): (1604, 1024, 3072),
          (224, 4): (1923, 768, 4096), (256, 6): (1805, 640, 6144)}
SHAPES += SERVED.values()
F16, BF16, F32 = 0, 1, 2


@pytest.mark.parametrize("kind", [0, 1, 2])
def test_kslab_weights_at_every_height(kind):
    assert {h for h, _ in SERVED} == {128, 160, 192, 224, 256} == {h for h, ranges in SERVED if ranges > 1}
    for plan, s in SERVED.items():
        assert tile(kind, *s) == (0, 0, 0) and tile_plan(kind, *s) == plan
        assert kind != 2 or int8_plan(*s) == (1, plan[1])


def _common(M, N, K):
    print(f"case q8 tiles M={M} N={N} K={K}", flush=True)
    torch.manual_seed(M + N + K)
    return torch.zeros(80 << 20, dtype=torch.uint8, device="cuda"), torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int8(M, N, K):
    ws, st = _common(M, N, K)
    x = torch.randint(-128, 128, (M, K), dtype=torch.int8, device="cuda")
    w = torch.randint(-128, 128, (N, K), dtype=torch.int8, device="cuda")
    xs, wsc = torch.rand(M, device="cuda") * 0.1, torch.rand(N, device="cuda") * 0.01
    bias = torch.randn(N, device="cuda")
    acc = (x.double() @ w.double().t()).float()              # exact: K * 2^14 is below 2^24 up to K = 1024, and rounds once above
    for wt, ldw in ((w, K), (rearrange.to_kslab(w), 0)):
        for dt, code, b in ((torch.float16, F16, None), (torch.float32, F32, bias), (torch.bfloat16, BF16, bias)):
            out = torch.full((M, N), float("nan"), device="cuda", dtype=dt)
            _lib.call("mi355q_w8a8_int8_gemm_ws", out.data_ptr(), None, x.data_ptr(), wt.data_ptr(), xs.data_ptr(), 1, wsc.data_ptr(), 1,
                      None if b is None else b.data_ptr(), 1, M, N, K, K, ldw, N, code, ws.data_ptr(), ws.numel(), st)
            want = acc * xs.view(-1, 1) * wsc.view(1, -1)
            assert torch.equal(out, (want if b is None else want + b).to(dt))
    # one scale for all, and none at all
    out = torch.full((M, N), float("nan"), device="cuda")
    _lib.call("mi355q_w8a8_int8_gemm_ws", out.data_ptr(), None, x.data_ptr(), w.data_ptr(), xs.data_ptr(), 0, None, 1, None, 0, M, N, K, K, K,
              N, F32, ws.data_ptr(), ws.numel(), st)
    assert torch.equal(out, acc * xs[0])


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_fp8(M, N, K):
    ws, st = _common(M, N, K)
    x = (torch.randn(M, K, device="cuda") * 40).to(torch.float8_e4m3fn)
    w = (torch.randn(N, K, device="cuda") * 40).to(torch.float8_e4m3fn)
    bias = torch.randn(N, device="cuda").bfloat16()
    xb, wb = torch.rand(M, K // 128, device="cuda") * 0.01 + 0.001, torch.rand(N // 128, K // 128, device="cuda") * 0.01 + 0.001
    xs, wsc = torch.rand(M, device="cuda") * 0.01, torch.rand(N, device="cuda") * 0.01
    xd = (x.double().view(M, K // 128, 128) * xb.double()[..., None]).view(M, K)
    wd = (w.double().view(N // 128, 128, K // 128, 128) * wb.double()[:, None, :, None]).view(N, K)
    blocks = xd @ wd.t() + bias.double()
    scaled = (x.double() @ w.double().t()) * xs.double().view(-1, 1) * wsc.double().view(1, -1) + bias.double()
    for wt, ldw in ((w, K), (rearrange.to_kslab(w), 0)):
        out = torch.full((M, N), float("nan"), device="cuda").bfloat16()
        _lib.call("mi355q_fp8_block_gemm_ws", out.data_ptr(), x.data_ptr(), wt.data_ptr(), xb.data_ptr(), wb.data_ptr(), bias.data_ptr(), M, N, K,
                  K, ldw, N, BF16, ws.data_ptr(), ws.numel(), st)
        assert float((out.double() - blocks).norm() / blocks.norm()) < 3e-3       # one rounding to bf16
        out.fill_(float("nan"))
        _lib.call("mi355q_fp8_scaled_gemm_ws", out.data_ptr(), x.data_ptr(), wt.data_ptr(), xs.data_ptr(), 1, wsc.data_ptr(), 1, bias.data_ptr(),
                  M, N, K, K, ldw, N, BF16, ws.data_ptr(), ws.numel(), st)
        assert float((out.double() - scaled).norm() / scaled.norm()) < 3e-3


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_fp8_to_fp16(M, N, K):
    """The same sums, stored as fp16: within one rounding of the float64 product."""
    ws, st = _common(M, N, K)
    x, w = ((torch.randn(r, K, device="cuda") * 40).to(torch.float8_e4m3fn) for r in (M, N))
    xb, wb = torch.rand(M, K // 128, device="cuda") * 1e-4 + 1e-5, torch.rand(N // 128, K // 128, device="cuda") + 0.1
    xs, wsc = torch.rand(M, device="cuda") * 1e-4, torch.rand(N, device="cuda")
    xd = (x.double().view(M, K // 128, 128) * xb.double()[..., None]).view(M, K)
    wd = (w.double().view(N // 128, 128, K // 128, 128) * wb.double()[:, None, :, None]).view(N, K)
    want = xd @ wd.t(), (x.double() @ w.double().t()) * xs.double().view(-1, 1) * wsc.double().view(1, -1)
    for wt, ldw in ((w, K), (rearrange.to_kslab(w), 0)):
        outs = [torch.full((M, N), float("nan"), device="cuda").half() for _ in range(2)]
        _lib.call("mi355q_fp8_block_gemm_ws", outs[0].data_ptr(), x.data_ptr(), wt.data_ptr(), xb.data_ptr(), wb.data_ptr(), None, M, N, K,
                  K, ldw, N, F16, ws.data_ptr(), ws.numel(), st)
        _lib.call("mi355q_fp8_scaled_gemm_ws", outs[1].data_ptr(), x.data_ptr(), wt.data_ptr(), xs.data_ptr(), 1, wsc.data_ptr(), 1, None,
                  M, N, K, K, ldw, N, F16, ws.data_ptr(), ws.numel(), st)
        for out, ref in zip(outs, want):
            assert float((out.double() - ref).norm() / ref.norm()) < 1e-3
