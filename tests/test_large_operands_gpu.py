"""Operands past the 32-bit index ranges of a single launch: only the rows that are looked at are written and checked, the rest of
the memory is whatever the allocator hands out."""
import pytest
import torch

from vllm_gcu_amd.kernels import _custom_ops as ops

pytestmark = pytest.mark.gpu
GIB = 1 << 30


@pytest.fixture(autouse=True)
def _give_back():
    torch.cuda.empty_cache()
    yield
    torch.cuda.empty_cache()


def _need(gib):
    free = torch.cuda.mem_get_info()[0]
    if free < (gib + 4) * GIB:
        pytest.skip(f"needs {gib} GiB of GPU memory, {free / GIB:.0f} are free")


def test_fp8_block_scales_of_four_gib(monkeypatch):
    """2^23 rows of 128 block scales are 4 GiB: the rows behind them have their own scales, not those 2^32 bytes before."""
    print("case large fp8 block scales", flush=True)
    _need(140)
    monkeypatch.setattr(ops, "_FP8_STAGE_SCALES", False)      # (the scales are read as they are)
    K, N, tail = 16384, 128, 300
    M = (1 << 23) + tail
    gen = torch.Generator(device="cuda").manual_seed(1)
    x, xs = torch.empty(M, K, dtype=torch.float8_e4m3fn, device="cuda"), torch.empty(M, K // 128, device="cuda")
    w = (torch.randn(N, K, device="cuda", generator=gen) * 50).to(torch.float8_e4m3fn)
    ws = torch.rand(1, K // 128, device="cuda", generator=gen) * 1e-4
    out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    parts = [slice(0, tail), slice(M - tail - 20, M)]
    for p in parts:
        n = p.stop - p.start
        x[p] = (torch.randn(n, K, device="cuda", generator=gen) * 50).to(torch.float8_e4m3fn)
        xs[p] = torch.rand(n, K // 128, device="cuda", generator=gen)
    torch.ops._C.linear_quant(out, x, w, None, xs, ws)
    wf = w.float() * ws.repeat_interleave(128, 1)
    for p in parts:
        want = (x[p].float() * xs[p].repeat_interleave(128, 1)) @ wf.t()
        torch.testing.assert_close(out[p].float(), want, rtol=1e-2, atol=1e-2 * want.std().item())
