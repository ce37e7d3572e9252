"""The row-in-registers quantisers and norms at the edges of their launch shapes: rows that end inside a piece, one
piece short of and past a whole number of pieces, fewer and more rows than the rule's steps, rows too long for
registers and rows whose address or length needs the one-element loops."""
import ctypes
import os

import pytest
import torch

from vllm_gcu_amd import _lib
from vllm_gcu_amd.kernels import _custom_ops  # noqa: F401  (registers the ops)

pytestmark = pytest.mark.gpu
SHAPES = [(1, 8), (3, 13), (2, 2040), (2, 2056), (700, 2048), (1100, 1032), (3, 8192 + 8), (600, 16384), (2, 65536), (2, 65544)]


def over(a, b):
    """a / b as one division (torch multiplies by the reciprocal where one side is a plain number)"""
    t = a if torch.is_tensor(a) else b
    return (a if torch.is_tensor(a) else torch.full_like(t, a)) / (b if torch.is_tensor(b) else torch.full_like(t, b))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,K", SHAPES)
def test_dynamic_row_quantisers(rows, K, dtype):
    print(f"case row quantisers {rows} x {K} {dtype}", flush=True)
    torch.manual_seed(rows * K)
    x = torch.randn(rows, K, device="cuda").to(dtype)
    x[0] = 0
    flat = torch.empty(rows * K + 1, dtype=dtype, device="cuda")
    flat[1:] = x.view(-1)
    for src in (x, flat[1:].view(rows, K)):                      # the second one off the 16-byte grid
        q, s = torch.empty(rows, K, dtype=torch.int8, device="cuda"), torch.empty(rows, 1, device="cuda")
        torch.ops._C.dynamic_scaled_int8_quant(q, src, s, None)
        mx = x.float().abs().amax(dim=1, keepdim=True)
        assert torch.equal(s, over(mx, 127.0))
        want = torch.nan_to_num(x.float() * over(127.0, mx), nan=0.0).round().clamp(-128, 127).to(torch.int8)
        assert torch.equal(q, want)
        f, fs = torch.empty(rows, K, dtype=torch.float8_e4m3fn, device="cuda"), torch.empty(rows, 1, device="cuda")
        torch.ops._C.dynamic_per_token_scaled_fp8_quant(f, src, fs, None)
        assert torch.equal(fs, over(mx.clamp_min(1e-10), 448.0))
        assert torch.equal(f.view(torch.uint8), (x.float() / fs).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,K", [(1, 8), (3, 13), (5, 2056), (300, 520)])
def test_static_int8_quant_with_scales_of_either_type(rows, K, dtype):
    print(f"case static int8 {rows} x {K} {dtype}", flush=True)
    torch.manual_seed(rows * K)
    x = torch.randn(rows, K, device="cuda").to(dtype)
    sc = (torch.rand(K, device="cuda") * 0.03 + 0.01).to(dtype)
    want = (x.float() * (1.0 / sc.float()).to(dtype).float()).round().clamp(-128, 127).to(torch.int8)
    for scale in (sc, sc.float()):
        q = torch.empty(rows, K, dtype=torch.int8, device="cuda")
        torch.ops._C.static_scaled_int8_quant(q, x, scale, None)
        assert torch.equal(q, want)
        torch.ops._C.static_scaled_int8_quant(q, x, scale[:1], None)
        one = (x.float() * (1.0 / sc[:1].float()).to(dtype).float()).round().clamp(-128, 127).to(torch.int8)
        assert torch.equal(q, one)


@pytest.mark.parametrize("rows,d", [(1, 8), (3, 1544), (700, 1408), (2048, 2048)])
def test_silu_and_sum_index_arithmetic(rows, d):
    print(f"case silu / sum {rows} x {d}", flush=True)
    torch.manual_seed(rows + d)
    x = torch.randn(rows, 2 * d, device="cuda").half()
    out = torch.full((rows, d), float("nan"), device="cuda").half()
    torch.ops._C.silu_and_mul(out, x)
    want = torch.nn.functional.silu(x[:, :d].float()) * x[:, d:].float()
    torch.testing.assert_close(out.float(), want, rtol=2e-3, atol=2e-3)
    x3 = torch.randn(rows, 3, d, device="cuda").half()
    n = torch.tensor([max(1, rows - 1)], dtype=torch.int32, device="cuda")
    total = torch.full((rows, d), float("nan"), device="cuda").half()
    torch.ops._moe_C.moe_sum_pad(total, x3, n, 1, False)
    m = int(n)
    torch.testing.assert_close(total[:m].float(), x3[:m].float().sum(1), rtol=2e-3, atol=2e-3)
    assert torch.isnan(total[m:]).all()
    if d % 128 == 0:
        q = torch.empty(rows, d, dtype=torch.float8_e4m3fn, device="cuda")
        s = torch.empty(rows, d // 128, device="cuda")
        torch.ops._C.silu_mul_per_token_group_quant(q, s, x, 128)
        g = out.float().view(rows, d // 128, 128)
        assert torch.equal(s, over(g.abs().amax(-1).clamp_min(1e-10), 448.0))
        assert torch.equal(q.view(torch.uint8), (g / s[..., None]).clamp(-448, 448).view(rows, d).to(torch.float8_e4m3fn).view(torch.uint8))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_group_fp8_codes_of_every_pair(dtype):
    """Every fraction against every largest one, over the ten binades whose codes are normal (test_short_forms_give_the_bits_of_the_plain_ones has all pairs): the code is that
    of the IEEE quotient, as torch has it.  An infinity in the group makes zeros of the rest, with their signs."""
    bits = 10 if dtype == torch.float16 else 7
    one = 0x3C00 if dtype == torch.float16 else 0x3F80
    print(f"case group fp8 codes of every pair {dtype}", flush=True)
    n = 1 << bits
    small = torch.arange(-10 * n, n, device="cuda") + one                  # ten binades below and that of the largest
    small = torch.where(small % 2 == 1, small | 0x8000, small)
    for m0 in range(0, n, 256):
        mx = torch.arange(m0, min(m0 + 256, n), device="cuda") + one
        groups = (small.numel() + 126) // 127
        x = torch.zeros(mx.numel(), groups, 128, dtype=torch.int32, device="cuda")
        x[:, :, 1:] = torch.nn.functional.pad(small, (0, groups * 127 - small.numel())).view(groups, 127)
        x[:, :, 1:] = torch.where((x[:, :, 1:] & 0x7FFF) > mx[:, None, None], mx[:, None, None].int(), x[:, :, 1:])
        x[:, :, 0] = mx[:, None]
        x = x.to(torch.int16).view(dtype).view(mx.numel(), -1)
        q, s = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device="cuda"), torch.empty(mx.numel(), groups, device="cuda")
        torch.ops._C.dynamic_per_token_group_fp8_quant(q, s, x, 128)
        assert torch.equal(s, over(x.view(mx.numel(), groups, 128)[:, :, 0].float(), 448.0))
        want = (x.float().view(mx.numel(), groups, 128) / s[:, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
        assert torch.equal(q.view(torch.uint8), want.view(torch.uint8).view(q.shape))
    x = torch.randn(1, 128, device="cuda").to(dtype)
    x[0, 5], x[0, 7] = float("inf"), -0.0
    q, s = torch.empty(1, 128, dtype=torch.float8_e4m3fn, device="cuda"), torch.empty(1, 1, device="cuda")
    torch.ops._C.dynamic_per_token_group_fp8_quant(q, s, x, 128)
    rest = torch.arange(128, device="cuda") != 5
    assert s.isinf().all() and torch.equal(q.view(torch.uint8)[0, rest], (torch.signbit(x[0, rest]).to(torch.uint8) * 128))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_silu_of_every_gate(dtype):
    """Every gate there is, also those whose sigmoid is no normal number, against the product in 64 bits: half a unit of the type's last place, and 2^-20
    for the exponential, the reciprocal and the products in fp32; the smallest step of the type; and where the exponential is beyond fp32, 2^128 and more, a
    sigmoid of 0 in place of up to 2^-128."""
    print(f"case silu of every gate {dtype}", flush=True)
    gate = torch.arange(65536, device="cuda").to(torch.int32).to(torch.int16).view(dtype)
    gate = gate[gate.float().isfinite()].view(1, -1)
    gate = gate[:, :gate.numel() // 8 * 8]
    x = torch.cat([gate, torch.ones_like(gate)], dim=1).contiguous()
    y = torch.empty_like(gate)
    torch.ops._C.silu_and_mul(y, x)
    a = gate.double()
    want = a / (1 + torch.exp(-a))
    digits, least = (11, 2.0 ** -24) if dtype == torch.float16 else (8, 2.0 ** -126)
    bound = want.abs() * (2.0 ** -digits + 2.0 ** -20) + least + a.abs() * 2.0 ** -128
    assert ((y.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("what,dtype", [("reciprocal", torch.float16), ("gate", torch.float16), ("gate", torch.bfloat16), ("codes", torch.float16), ("codes", torch.bfloat16)])
def test_short_forms_give_the_bits_of_the_plain_ones(what, dtype):
    """On the GPU, over every operand: the reciprocal of three instructions from 1 to 2^126; the gate of eight with every gate and up value there is; the fp8 codes of every
    value against every largest magnitude of a row."""
    print(f"case short forms {what} {dtype}", flush=True)
    check = ctypes.CDLL(os.path.join(os.path.dirname(_lib.LIB_PATH), "libmi355q_bench.so")).mi355q_bench_check_arithmetic
    check.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
    wrong = torch.zeros(1, dtype=torch.int64, device="cuda")
    assert check(["reciprocal", "gate", "codes"].index(what), {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}[dtype], wrong.data_ptr(),
                 torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert wrong.item() == 0
