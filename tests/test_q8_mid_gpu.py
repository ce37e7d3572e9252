"""The 8-bit kernel for a few dozen to 1536 rows (csrc/q8_mid.hip) through the operators that choose it:
row counts around every tile edge and to the end of its range, column counts that are and are not a multiple of eight column tiles, odd numbers of K
blocks, one and several K ranges, with and without bias.  int8 is exact; fp8 is compared with a float64 product."""
import pytest
import torch

from test_q8_plans_cpu import NO_ROOM, tile, way
from vllm_gcu_amd.kernels import _custom_ops as ops
from vllm_gcu_amd.kernels import _runtime as rt
from vllm_gcu_amd.kernels.quantization import rearrange

pytestmark = pytest.mark.gpu
# (M, N, K): tiles of every height, with and without K ranges
SHAPES = [(17, 64, 384), (31, 320, 128), (33, 512, 4096), (48, 1024, 7168), (63, 640, 640), (64, 4096, 2048), (65, 1024, 1024),
          (96, 3072, 3584), (127, 256, 4096), (129, 1024, 5120), (130, 4096, 7168), (200, 2048, 1408), (257, 4608, 3584),
          (511, 4096, 4096), (512, 8192, 2048), (700, 512, 7168), (768, 1024, 4096), (1000, 3072, 3584), (1024, 4096, 4096),
          (1300, 640, 2048), (1535, 1536, 3584), (1536, 2048, 2048),
          (67, 5760, 768), (193, 8448, 768), (323, 6656, 768), (399, 6912, 768), (467, 6656, 2048), (163, 5632, 1536),
          # with K ranges; 144 and 160 rows with block scales
          (65, 1920, 3968), (66, 5504, 6272), (36, 8448, 3456), (84, 8576, 7552), (195, 2816, 6400), (131, 5504, 5888), (151, 5504, 6016)]
BLOCK, SCALED, INT8 = 0, 1, 2            # kinds of mi355q_q8_mid_plan
FEW = 12                                 # the kernel for few rows (csrc/q8_decode.hip) among the tiles of mi355q_q8_mid_way


def _planned(kind, M, N, K):
    want = rt.host.q8_mid_plan(kind, M, N, K)
    print(f"case q8 mid kind={kind} M={M} N={N} K={K} workspace={want}", flush=True)
    assert want >= 0 and way(kind, M, N, K)[0] < FEW, "another kernel takes this shape: the case tests nothing"


@pytest.mark.parametrize("kind", [BLOCK, SCALED, INT8])
def test_the_shapes_take_every_tile(kind):
    tall = {144, 160} if kind == BLOCK else set()
    tiles = [tile(kind, *s) for s in SHAPES if s[1] % 128 == 0]
    assert {t[0] for t in tiles} == {32, 48, 64, 80, 96, 112, 128} | tall
    assert {t[0] for t in tiles if t[2] > 1} >= {32, 64, 80} | tall


@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int8(M, N, K, with_bias):
    _planned(INT8, M, N, K)
    torch.manual_seed(M + N + K)
    x = torch.randint(-128, 128, (M, K), dtype=torch.int8, device="cuda")
    w = torch.randint(-128, 128, (N, K), dtype=torch.int8, device="cuda")
    xs, ws = torch.rand(M, 1, device="cuda") * 0.1, torch.rand(N, 1, device="cuda") * 0.01
    bias = torch.randn(N, device="cuda").half() if with_bias else None
    out = torch.full((M, N), float("nan"), device="cuda").half()
    torch.ops._C.cutlass_scaled_mm(out, x, rearrange.to_kslab(w).t(), xs, ws, bias)
    acc = (x.double() @ w.double().t()).float()              # exact: below 2^53, and below 2^24 where it matters not
    want = acc * xs * ws.view(1, N)
    if with_bias:
        want = want + bias.float()
    assert torch.equal(out, want.half())


@pytest.mark.parametrize("M,N,K", [s for s in SHAPES if s[1] % 128 == 0])
def test_fp8_block_and_scaled(M, N, K):
    torch.manual_seed(M + N + K)
    x = (torch.randn(M, K, device="cuda") * 40).to(torch.float8_e4m3fn)
    w = (torch.randn(N, K, device="cuda") * 40).to(torch.float8_e4m3fn)
    wk = rearrange.to_kslab(w)
    xb, wb = torch.rand(M, K // 128, device="cuda") * 0.01 + 0.001, torch.rand(N // 128, K // 128, device="cuda") * 0.01 + 0.001
    xd = x.double().view(M, K // 128, 128) * xb.double()[..., None]
    wd = w.double().view(N // 128, 128, K // 128, 128) * wb.double()[:, None, :, None]
    want = xd.view(M, K) @ wd.view(N, K).t()
    _planned(BLOCK, M, N, K)
    for bias in (None, torch.randn(N, device="cuda").bfloat16()):
        out = torch.full((M, N), float("nan"), device="cuda").bfloat16()
        torch.ops._C.linear_quant(out, x, wk, bias, xb, wb)
        ref = want if bias is None else want + bias.double()
        assert float((out.double() - ref).norm() / ref.norm()) < 3e-3        # one rounding to bf16
    _planned(SCALED, M, N, K)
    for xs, ws in ((torch.rand(M, 1, device="cuda") * 0.01, torch.rand(N, 1, device="cuda") * 0.01),
                   (torch.full((1,), 0.01, device="cuda"), torch.full((1,), 0.003, device="cuda"))):
        out = torch.full((M, N), float("nan"), device="cuda").half()
        torch.ops._C.cutlass_scaled_mm(out, x, wk.t(), xs, ws, None)
        ref = (x.double() @ w.double().t()) * xs.double().view(-1, 1) * ws.double().view(1, -1)
        assert float((out.double() - ref).norm() / ref.norm()) < 1e-3


@pytest.mark.parametrize("M,N,K", [(48, 1024, 7168), (84, 8576, 7552), (65, 1024, 1024), (399, 6912, 768)])
def test_other_output_types(M, N, K):
    """fp8 with block scales to fp16 and int8 to fp32, with and without K ranges."""
    from vllm_gcu_amd import _lib
    _planned(BLOCK, M, N, K), _planned(INT8, M, N, K)
    torch.manual_seed(M + N + K)
    st = torch.cuda.current_stream().cuda_stream
    ws = torch.zeros(80 << 20, dtype=torch.uint8, device="cuda")
    x, w = ((torch.randn(r, K, device="cuda") * 40).to(torch.float8_e4m3fn) for r in (M, N))
    xb, wb = torch.rand(M, K // 128, device="cuda") * 1e-4 + 1e-5, torch.rand(N // 128, K // 128, device="cuda") + 0.1
    out = torch.full((M, N), float("nan"), device="cuda").half()
    _lib.call("mi355q_fp8_block_gemm_ws", out.data_ptr(), x.data_ptr(), rearrange.to_kslab(w).data_ptr(), xb.data_ptr(), wb.data_ptr(), None, M, N, K, K,
              0, N, _lib.F16, ws.data_ptr(), ws.numel(), st)
    want = (x.double().view(M, -1, 128) * xb.double()[..., None]).view(M, K) @ (
        w.double().view(N // 128, 128, K // 128, 128) * wb.double()[:, None, :, None]).view(N, K).t()
    assert float((out.double() - want).norm() / want.norm()) < 1e-3
    x, w = (torch.randint(-128, 128, (r, K), dtype=torch.int8, device="cuda") for r in (M, N))
    xs, wsc = torch.rand(M, device="cuda") * 0.1, torch.rand(N, device="cuda") * 0.01
    out = torch.full((M, N), float("nan"), device="cuda")
    _lib.call("mi355q_w8a8_int8_gemm_ws", out.data_ptr(), None, x.data_ptr(), rearrange.to_kslab(w).data_ptr(), xs.data_ptr(), 1, wsc.data_ptr(), 1,
              None, 1, M, N, K, K, 0, N, _lib.F32, ws.data_ptr(), ws.numel(), st)
    assert torch.equal(out, (x.double() @ w.double().t()).float() * xs.view(-1, 1) * wsc)


# 160 rows of 30 MB, 64 of 80 MB: further apart than 32 bits of bytes, also within a tile (160 rows are two of 80 or 96, one of 256)
@pytest.mark.parametrize("M,N,K,ldx,kslab", [(160, 16512, 128, 30_000_000, True), (160, 16512, 128, 30_000_000, False),
                                               (160, 260, 256, 30_000_000, False), (64, 16512, 128, 80_000_000, True)])
def test_int8_rows_far_apart(M, N, K, ldx, kslab):
    """Row strides at which the rows of a tile do not fit 32-bit offsets: the same outputs and sums as for dense rows."""
    from vllm_gcu_amd import _lib
    print(f"case q8 rows far apart M={M} N={N} K={K} ldx={ldx} kslab={kslab}", flush=True)
    torch.manual_seed(M + N)
    dense = torch.randint(-128, 128, (M, K), dtype=torch.int8, device="cuda")
    w = torch.randint(-128, 128, (N, K), dtype=torch.int8, device="cuda")
    wt, ldw = (rearrange.to_kslab(w), 0) if kslab else (w, K)
    xs, wsc = torch.rand(M, device="cuda") * 0.1, torch.rand(N, device="cuda") * 0.01
    x = torch.empty(M * ldx, dtype=torch.int8, device="cuda").as_strided((M, K), (ldx, 1))
    x.copy_(dense)
    ws, st = torch.zeros(80 << 20, dtype=torch.uint8, device="cuda"), torch.cuda.current_stream().cuda_stream
    want = dense.double() @ w.double().t()
    for acc in (None, torch.zeros(M, N, dtype=torch.int32, device="cuda")):
        out = torch.full((M, N), float("nan"), device="cuda")
        _lib.call("mi355q_w8a8_int8_gemm_ws", out.data_ptr(), None if acc is None else acc.data_ptr(), x.data_ptr(), wt.data_ptr(), xs.data_ptr(), 1,
                  wsc.data_ptr(), 1, None, 0, M, N, K, ldx, ldw, N, _lib.F32, ws.data_ptr(), ws.numel(), st)
        assert torch.equal(out, want.float() * xs.view(-1, 1) * wsc)
        assert acc is None or torch.equal(acc, want.int())


def test_fp8_rows_far_apart():
    """The same for fp8: what the tile of the plan reaches is computed, more is refused."""
    from vllm_gcu_amd import _lib
    N, K, ldx = 8320, 768, 30_000_000
    w = rearrange.to_kslab((torch.randn(N, K, device="cuda") * 40).to(torch.float8_e4m3fn))
    x = torch.empty(160 * 40_000_000, dtype=torch.uint8, device="cuda").view(torch.float8_e4m3fn).as_strided((160, K), (ldx, 1))
    x.copy_((torch.randn(160, K, device="cuda") * 40).to(torch.float8_e4m3fn))
    dense, xs, wsc = x.contiguous(), torch.rand(160, device="cuda"), torch.rand(N, device="cuda")
    st = torch.cuda.current_stream().cuda_stream

    def call(M, rows, stride):
        out = torch.full((M, N), float("nan"), device="cuda").bfloat16()
        _lib.call("mi355q_fp8_scaled_gemm_ws", out.data_ptr(), rows.data_ptr(), w.data_ptr(), xs.data_ptr(), 1, wsc.data_ptr(), 1, None, M, N, K,
                  stride, 0, N, _lib.BF16, None, 0, st)
        return out
    assert 0 < tile(SCALED, 160, N, K)[0] <= 128
    assert torch.equal(call(160, x, ldx), call(160, dense, K))
    with pytest.raises(RuntimeError, match="fits neither kernel"):
        call(160, x, 40_000_000)


# (kind, M, N, K) -> tile and K ranges: sums added in the kernel (up to 56 KiB of other ranges) or by a second launch
RANGES = [(BLOCK, 54, 1152, 2560, (32, 32, 3)), (INT8, 46, 768, 7936, (32, 32, 5)), (SCALED, 47, 128, 3968, (32, 32, 6)), (BLOCK, 100, 1024, 3584, (32, 32, 2)),
          (SCALED, 47, 128, 10880, (32, 32, 15)), (INT8, 49, 128, 11648, (32, 32, 16)), (INT8, 17, 192, 10624, None), (BLOCK, 33, 1408, 4224, (32, 64, 5)),
          (BLOCK, 33, 896, 8832, (32, 64, 9)), (SCALED, 100, 2176, 4480, (64, 64, 3)), (SCALED, 129, 1024, 5120, (64, 64, 5)), (INT8, 129, 128, 10880, (32, 64, 11))]


@pytest.mark.parametrize("kind,M,N,K,plan", RANGES)
def test_k_ranges_leave_the_counters_at_zero(kind, M, N, K, plan):
    """Products and sums that are exact, over a workspace whose first MiB is zero and whose rest is not, twice: the output to the bit, the
    counters as they were."""
    from vllm_gcu_amd import _lib
    assert plan is None or tile(kind, M, N, K) == plan
    need = rt.host.q8_mid_plan(kind, M, N, K)
    print(f"case q8 ranges kind={kind} M={M} N={N} K={K} workspace={need}", flush=True)
    assert need > 1 << 20
    torch.manual_seed(M + N + K)
    ws = torch.full((need,), 0xff, dtype=torch.uint8, device="cuda")
    ws[:1 << 20] = 0
    x, w = (torch.randint(-3, 4, (r, K), device="cuda").to(torch.int8 if kind == INT8 else torch.float8_e4m3fn) for r in (M, N))
    wk, st = rearrange.to_kslab(w), torch.cuda.current_stream().cuda_stream
    xs = 2.0 ** torch.randint(-2, 3, (M, K // 128) if kind == BLOCK else (M, 1), device="cuda").float()
    sc = 2.0 ** torch.randint(-2, 3, (N // 128, K // 128) if kind == BLOCK else (N, 1), device="cuda").float()
    if kind == BLOCK:
        xd, wd = x.double() * xs.double().repeat_interleave(128, 1), w.double() * sc.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    else:
        xd, wd = x.double() * xs.double(), w.double() * sc.double()
    want = (xd @ wd.t()).bfloat16()
    for _ in range(2):
        out = torch.full((M, N), float("nan"), device="cuda").bfloat16()
        if kind == INT8:
            _lib.call("mi355q_w8a8_int8_gemm_ws", out.data_ptr(), None, x.data_ptr(), wk.data_ptr(), xs.data_ptr(), 1, sc.data_ptr(), 1, None, 0,
                      M, N, K, K, 0, N, _lib.BF16, ws.data_ptr(), need, st)
        elif kind == SCALED:
            _lib.call("mi355q_fp8_scaled_gemm_ws", out.data_ptr(), x.data_ptr(), wk.data_ptr(), xs.data_ptr(), 1, sc.data_ptr(), 1, None, M, N, K,
                      K, 0, N, _lib.BF16, ws.data_ptr(), need, st)
        else:
            _lib.call("mi355q_fp8_block_gemm_ws", out.data_ptr(), x.data_ptr(), wk.data_ptr(), xs.data_ptr(), sc.data_ptr(), None, M, N, K, K, 0, N,
                      _lib.BF16, ws.data_ptr(), need, st)
        assert torch.equal(out, want) and not ws[:1 << 20].any()


# with RANGES and SHAPES: every tile of every kind whole, with ranges that the kernel adds and with ranges that a second launch adds, where the plans
# have such launches (test_q8_plans_cpu.py looks whether they are all here)
MORE = [(BLOCK, 17, 128, 14336), (BLOCK, 129, 1152, 3968), (BLOCK, 121, 2432, 10240), (BLOCK, 129, 128, 2048), (BLOCK, 207, 1152, 9088),
        (BLOCK, 129, 128, 9088), (BLOCK, 97, 2176, 8192), (BLOCK, 339, 2176, 6400), (BLOCK, 1285, 3072, 384), (BLOCK, 1450, 3072, 384),
        (SCALED, 17, 64, 14336), (SCALED, 129, 64, 2048), (SCALED, 33, 4096, 14336), (SCALED, 129, 64, 9088), (SCALED, 129, 1408, 14336),
        (SCALED, 152, 1408, 14336), (INT8, 33, 1408, 5120), (INT8, 129, 1152, 3968), (INT8, 106, 2432, 6400), (INT8, 129, 64, 3072), (INT8, 70, 1024, 8192),
        (INT8, 97, 3072, 9088), (INT8, 482, 2432, 10880),
        # the kernel for few rows; an int8 layer of it to fp32, which is the tile's, with ranges
        (BLOCK, 33, 512, 1152), (SCALED, 24, 1024, 2048), (INT8, 33, 512, 1152), (INT8, 32, 128, 3328)]


@pytest.mark.parametrize("zeroed", [True, False])
@pytest.mark.parametrize("kind,M,N,K,plan", RANGES + [(*m, None) for m in MORE])
def test_k_ranges_leave_the_first_mib_as_it_was(kind, M, N, K, plan, zeroed):
    """Products and sums that are exact, in two output types, over a workspace that nobody cleared but for, where the call says so, the counters: the output to
    the bit, the counters at zero, and without them the first MiB neither read nor written."""
    from vllm_gcu_amd import _lib
    assert plan is None or tile(kind, M, N, K) == plan
    need = rt.host.q8_mid_plan(kind, M, N, K)
    print(f"case q8 ranges kind={kind} M={M} N={N} K={K} workspace={need} zeroed={zeroed} way={way(kind, M, N, K)}", flush=True)
    assert need > 1 << 20 or (need == 0 and way(kind, M, N, K)[1] == 1)
    torch.manual_seed(M + N + K)
    ws = torch.randint(0, 256, (max(need, 1 << 20),), dtype=torch.uint8, device="cuda")
    ws[1 << 20:] = 0xff
    if zeroed:
        ws[:1 << 16] = 0
    before, flag = ws[:1 << 20].clone(), _lib.ZEROED_COUNTERS if zeroed else 0
    x, w = (torch.randint(-3, 4, (r, K), device="cuda").to(torch.int8 if kind == INT8 else torch.float8_e4m3fn) for r in (M, N))
    wk, st = rearrange.to_kslab(w), torch.cuda.current_stream().cuda_stream
    xs = 2.0 ** torch.randint(-2, 3, (M, K // 128) if kind == BLOCK else (M, 1), device="cuda").float()
    sc = 2.0 ** torch.randint(-2, 3, (N // 128, K // 128) if kind == BLOCK else (N, 1), device="cuda").float()
    if kind == BLOCK:
        xd, wd = x.double() * xs.double().repeat_interleave(128, 1), w.double() * sc.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    else:
        xd, wd = x.double() * xs.double(), w.double() * sc.double()
    want = xd @ wd.t()
    for dtype in (torch.bfloat16, torch.float32 if kind == INT8 else torch.float16):
        out, code = torch.full((M, N), float("nan"), dtype=dtype, device="cuda"), rt.dtype_code(dtype) | flag
        if kind == INT8:
            _lib.call("mi355q_w8a8_int8_gemm_ws", out.data_ptr(), None, x.data_ptr(), wk.data_ptr(), xs.data_ptr(), 1, sc.data_ptr(), 1, None, 0,
                      M, N, K, K, 0, N, code, ws.data_ptr(), need, st)
        elif kind == SCALED:
            _lib.call("mi355q_fp8_scaled_gemm_ws", out.data_ptr(), x.data_ptr(), wk.data_ptr(), xs.data_ptr(), 1, sc.data_ptr(), 1, None, M, N, K,
                      K, 0, N, code, ws.data_ptr(), need, st)
        else:
            _lib.call("mi355q_fp8_block_gemm_ws", out.data_ptr(), x.data_ptr(), wk.data_ptr(), xs.data_ptr(), sc.data_ptr(), None, M, N, K, K, 0, N,
                      code, ws.data_ptr(), need, st)
        assert torch.equal(out, want.to(dtype)) and torch.equal(ws[:1 << 20], before)


@pytest.mark.parametrize("kind,M,N,K", NO_ROOM)
def test_without_room_for_k_ranges(kind, M, N, K):
    """Shapes whose plan cuts K, through the entry points without a workspace: sums that are exact, to the bit."""
    from vllm_gcu_amd import _lib
    assert way(kind, M, N, K, 0)[0] < FEW
    print(f"case q8 without a workspace kind={kind} M={M} N={N} K={K}", flush=True)
    torch.manual_seed(M + N + K)
    x, w = (torch.randint(-3, 4, (r, K), device="cuda").to(torch.int8 if kind == INT8 else torch.float8_e4m3fn) for r in (M, N))
    wk, st = rearrange.to_kslab(w), torch.cuda.current_stream().cuda_stream
    xs, sc = (torch.ones(r, K // 128 if kind == BLOCK else 1, device="cuda") for r in (M, N // 128 if kind == BLOCK else N))
    out = torch.full((M, N), float("nan"), device="cuda").bfloat16()
    if kind == INT8:
        _lib.call("mi355q_w8a8_int8_gemm", out.data_ptr(), None, x.data_ptr(), wk.data_ptr(), xs.data_ptr(), 1, sc.data_ptr(), 1, None, 0, M, N, K, K, 0,
                  N, _lib.BF16, st)
    else:
        _lib.call("mi355q_fp8_block_gemm", out.data_ptr(), x.data_ptr(), wk.data_ptr(), xs.data_ptr(), sc.data_ptr(), None, M, N, K, K, 0, N, _lib.BF16,
                  st)
    assert torch.equal(out, (x.double() @ w.double().t()).bfloat16())
