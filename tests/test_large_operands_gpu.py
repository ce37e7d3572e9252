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


# rows of 8192 pieces of 8 elements: this many of them in a launch whose pieces are counted with 31 bits
D, PER_LAUNCH = 65536, 0x7fff0000 // 8192


def _rows(make):
    """A tensor of more rows than a launch takes and the slice around the border that is written and looked at."""
    t = make(PER_LAUNCH + 40)
    return t, slice(PER_LAUNCH - 2, PER_LAUNCH + 40)


# the row count ends behind the border, and before it
@pytest.mark.parametrize("count", [PER_LAUNCH + 20, PER_LAUNCH - 1])
@pytest.mark.parametrize("which", ["silu_and_mul", "group_quant", "moe_sum"])
def test_row_counts_over_several_launches(which, count):
    print(f"case large {which} with a row count of {count}", flush=True)
    _need({"silu_and_mul": 97, "group_quant": 50, "moe_sum": 66}[which])
    wide = 2 * D if which == "silu_and_mul" else D
    x, part = _rows(lambda n: torch.empty(n, wide, dtype=torch.float16, device="cuda"))
    x[part] = torch.randn(x[part].shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(2)).half()
    size = torch.tensor([count], dtype=torch.int32, device="cuda")
    live = count - part.start
    small = x[part].clone()
    if which == "silu_and_mul":
        out, want = torch.empty(x.shape[0], D, dtype=torch.float16, device="cuda"), torch.full((42, D), 7.0, dtype=torch.float16, device="cuda")
        out[part] = 7.0
        torch.ops._C.silu_and_mul_pad(out, x, size)
        torch.ops._C.silu_and_mul(want[:live], small[:live])
    elif which == "group_quant":
        out, want = (torch.empty(n, D, dtype=torch.float8_e4m3fn, device="cuda") for n in (x.shape[0], 42))
        out[part], want[:] = 7.0, 7.0
        sc, wsc = torch.zeros(x.shape[0], D // 128, device="cuda"), torch.zeros(42, D // 128, device="cuda")
        torch.ops._C.dynamic_per_token_group_fp8_quant_with_size(out, sc, x, size, 128)
        torch.ops._C.dynamic_per_token_group_fp8_quant(want[:live], wsc[:live], small[:live], 128)
        assert torch.equal(sc[part], wsc)
        out, want = out.view(torch.uint8), want.view(torch.uint8)
    else:
        out, want = torch.empty(x.shape, dtype=torch.float16, device="cuda"), torch.full((42, D), 7.0, dtype=torch.float16, device="cuda")
        out[part] = 7.0
        torch.ops._moe_C.moe_sum_pad(out, x[:, None], size, 1, False)
        want[:live] = small[:live]
    assert torch.equal(out[part], want)
