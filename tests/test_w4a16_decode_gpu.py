"""The W4A16 kernels for up to 16 rows (csrc/w4a16_decode.hip), through the library's own choice, over small layers -- 1, 2 and 4 column
tiles per workgroup, 8 and 16 wavefronts, one to seven K blocks each (the last ones without a block), row counts around each load of
four rows, groups of 128 to K, zero-points and none, bias, exact inputs bit for bit, and a row of infinities -- and over blocks of 16
slots of a fused-MoE layer."""
import numpy as np
import pytest
import torch

from oracle import w4 as ow4
from vllm_gcu_amd.kernels import _custom_ops as ops
from vllm_gcu_amd.kernels.quantization import rearrange

pytestmark = pytest.mark.gpu
# (K, N, group): K blocks 1 .. 64, N on both sides of 256 tiles of 16 and of 32 columns
SHAPES = [(128, 128, 128), (640, 1024, 128), (1024, 4096, 1024), (1152, 4224, 128), (2048, 384, 256), (2176, 8192, 128), (3072, 256, 1536),
          (4096, 512, 128), (4096, 8320, 256), (4224, 1024, 128), (6144, 4352, 128), (8192, 512, 4096), (1024, 16384, 128), (2944, 8448, 128),
          (1024, 8192, 256), (1280, 8320, 128), (3968, 4224, 128), (4352, 8320, 128), (6400, 4224, 128)]
# K blocks 65 .. 112: five to seven of a wavefront, on either side of the rows where it takes them (test_w4a16_decode_cpu.py has the plans)
DEEP = [(8320, 2048, 128), (10240, 3072, 1024), (10368, 4096, 128), (12288, 2048, 256), (12416, 3072, 128), (14336, 4096, 128), (10240, 4352, 128),
        (8448, 8192, 256)]


def _data(K, N, g, dtype, exact):
    rng = np.random.default_rng(K + N)
    q = rng.integers(0, 16, size=(K, N), dtype=np.uint8)
    z = rng.integers(0, 16, size=(K // g, N), dtype=np.uint8)
    s = 2.0 ** -rng.integers(4, 8, size=(K // g, N)) if exact else rng.uniform(0.001, 0.01, size=(K // g, N))
    x = rng.integers(-4, 5, size=(16, K)) if exact else rng.standard_normal((16, K))
    w, zp = rearrange.rearrange_uint4_int32_gptq(torch.from_numpy(ow4.gptq_pack_weight(q)).cuda(), torch.from_numpy(ow4.gptq_pack_zeros(z)).cuda())
    w8, _ = rearrange.rearrange_uint4_int32_gptq(torch.from_numpy(ow4.gptq_pack_weight(q)).cuda(), None)
    return q, z, torch.from_numpy(s.astype(np.float32)).to(dtype), torch.from_numpy(x.astype(np.float32)).to(dtype), w, zp, w8


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,N,g", SHAPES)
def test_rows_1_to_16(K, N, g, dtype):
    q, z, s, x, w, zp, w8 = _data(K, N, g, dtype, False)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(K)).to(dtype)
    want = ow4.w4a16_gemm(x.float().numpy(), q, z, s.float().numpy(), g, bias=bias.float().numpy())
    plain = ow4.w4a16_gemm(x.float().numpy(), q, None, s.float().numpy(), g)
    for M in (1, 4, 5, 8, 9, 16):
        print(f"case w4a16 decode M={M} K={K} N={N} g={g} {dtype}", flush=True)
        xm = x[:M].cuda()
        got = ops.w4a16_gemm(xm, w, s.cuda(), zp, bias.cuda(), g, out=torch.full((M, N), float("nan"), dtype=dtype, device="cuda"))
        np.testing.assert_allclose(got.float().cpu().numpy(), want[:M], rtol=1e-2, atol=1e-2)
        got = ops.w4a16_gemm(xm, w8, s.cuda(), None, None, g, out=torch.full((M, N), float("nan"), dtype=dtype, device="cuda"))
        np.testing.assert_allclose(got.float().cpu().numpy(), plain[:M], rtol=1e-2, atol=1e-2)
    # a row of infinities stays in its row
    bad = x.clone()
    bad[2, 5] = float("inf")
    for M in (3, 7, 16):
        a, b = (ops.w4a16_gemm(t[:M].cuda(), w, s.cuda(), zp, None, g) for t in (bad, x))
        keep = [i for i in range(M) if i != 2]
        assert torch.equal(a[keep], b[keep]) and not torch.isfinite(a[2]).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,N,g", SHAPES)
def test_exact(K, N, g, dtype):
    """Sums that fp32 holds exactly: bit for bit the oracle's, and the streaming kernel's."""
    q, z, s, x, w, zp, _ = _data(K, N, g, dtype, True)
    want = torch.from_numpy(ow4.w4a16_gemm(x.float().numpy(), q, z, s.float().numpy(), g)).to(dtype)
    for M in (1, 6, 16):
        assert torch.equal(ops.w4a16_gemm(x[:M].cuda(), w, s.cuda(), zp, None, g).cpu(), want[:M])
        assert torch.equal(ops.w4a16_gemm(x[:M].cuda(), w, s.cuda(), zp, None, g, family=1).cpu(), want[:M])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("E,K,N,g,counts", [
    (3, 128, 256, 128, (1, 0, 16)), (2, 1152, 384, 384, (4, 5)),                 # few slabs of weights: quarters of one to a workgroup
    (1, 640, 16384, 128, (3,)), (4, 384, 4096, 128, (1, 2, 8, 9)),               # up to a slab per CU: halves
    (4, 256, 8192, 128, (33, 4, 5, 16)), (1, 1408, 32768, 1408, (12,)),          # about one: whole slabs, eight wavefronts
    (8, 384, 8192, 384, (1, 2, 3, 1, 4, 1, 2, 3)), (8, 640, 8192, 128, (5, 8, 20, 7, 9, 1, 6, 17))])   # more: few rows each, many
def test_grouped_blocks_of_16(E, K, N, g, counts, dtype):
    """Fused-MoE launches over blocks of 16 slots: every workgroup shape, blocks with 1 .. 16 slots, pads in the middle of a block too, an
    expert out of range (zero rows), a layer with both forms of slot numbering and routing weights.  Sums that fp32 holds exactly: bit
    for bit."""
    from vllm_gcu_amd.kernels import fused_moe
    print(f"case w4a16 grouped decode E={E} K={K} N={N} g={g} {counts} {dtype}", flush=True)
    rng = np.random.default_rng(K + N + E)
    numel = sum(counts) + 3
    slots = rng.permutation(numel).astype(np.int32)
    q = rng.integers(0, 16, size=(E, K, N), dtype=np.uint8)
    z = rng.integers(0, 16, size=(E, K // g, N), dtype=np.uint8)
    s = torch.from_numpy((2.0 ** -rng.integers(4, 8, size=(E, K // g, N))).astype(np.float32)).to(dtype)
    w, zp = rearrange.rearrange_uint4_int32_gptq(torch.from_numpy(np.stack([ow4.gptq_pack_weight(a) for a in q])).cuda(),
                                                 torch.from_numpy(np.stack([ow4.gptq_pack_zeros(a) for a in z])).cuda())
    ids, experts, at, of = [], [], 0, np.full(numel, -1)
    for e, n in list(enumerate(counts)) + [(-1, 3)]:
        for i in range(0, n, 16):
            part = slots[at:at + min(16, n - i)]
            block = np.full(16, numel, dtype=np.int32)
            block[(16 - len(part)) // 2 * (len(experts) & 1):][:len(part)] = part       # every other block starts with pads
            ids.append(block), experts.append(e)
            of[part] = e
            at += len(part)
    used = 16 * len(experts)
    ids.append(np.full(16, -1, dtype=np.int32)), experts.append(0)                      # past the padded count: not read
    ids, experts = torch.from_numpy(np.concatenate(ids)).cuda(), torch.tensor(experts, dtype=torch.int32).cuda()
    npp = torch.tensor([used], dtype=torch.int32).cuda()
    rw = torch.from_numpy((2.0 ** rng.integers(-2, 2, size=numel)).astype(np.float32))
    for topk in (1, 2) if numel % 2 == 0 else (1, 3) if numel % 3 == 0 else (1,):
        x = torch.from_numpy(rng.integers(-4, 5, size=(numel // topk, K)).astype(np.float32)).to(dtype)
        want = np.zeros((numel, N), dtype=np.float32)
        for e in range(E):
            rows = np.nonzero(of == e)[0]
            if rows.size:
                want[rows] = x.float().numpy()[rows // topk] @ ow4.dequantize(q[e], z[e], s[e].float().numpy(), g)
        for weigh in (False, True):
            out = torch.full((numel // topk, topk, N), float("nan"), dtype=dtype, device="cuda")
            fused_moe.invoke_fused_moe_kernel(x.cuda(), w, out, None, s.cuda(), zp, rw.view(-1, topk).cuda(),
                                              torch.zeros(numel // topk, topk, dtype=torch.int32).cuda(), ids, experts, npp, weigh, topk,
                                              {"BLOCK_SIZE_M": 16}, use_fp8_w8a8=False, use_int8_w8a8=False,
                                              use_int8_w8a16=False, use_int4_w4a16=True, block_shape=[0, g])
            ref = torch.from_numpy(want * (rw.numpy()[:, None] if weigh else 1)).to(dtype)
            assert torch.equal(out.view(-1, N).cpu(), ref)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("ids_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("E,K,N", [(1, 384, 256), (3, 128, 4096), (8, 256, 8192), (60, 384, 768), (200, 128, 256), (1, 256, 32768)])
def test_unsorted_slots(E, K, N, ids_dtype, dtype):
    """Up to 64 slots given by their experts: bit for bit the aligned launch, for experts with 1 .. 64 slots and ids that are none of them
    (their rows are left alone), both forms of slot numbering, no alignment launch."""
    from vllm_gcu_amd import _lib
    from vllm_gcu_amd.kernels import fused_moe
    lib, g, code = _lib.load(), 128, _lib.F16 if dtype == torch.float16 else _lib.BF16
    gen = torch.Generator().manual_seed(E + N)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (E, K // 8, N), dtype=torch.int32, generator=gen).cuda()
    s = (torch.rand(E, K // g, N, generator=gen) * 0.01).to(dtype).cuda()
    zp = torch.randint(-2 ** 31, 2 ** 31 - 1, (E, K // g, N // 8), dtype=torch.int32, generator=gen).cuda()
    for numel in (1, 2, 15, 16, 17, 40, 63, 64):
        for few in (E, 1, min(E, 3)):
            print(f"case w4a16 unsorted E={E} K={K} N={N} numel={numel} of {few} {ids_dtype} {dtype}", flush=True)
            ids = torch.randint(0, few, (numel,), generator=gen).to(ids_dtype)
            if numel > 2:
                ids[1], ids[-1] = -1, E
            rw = torch.rand(numel, generator=gen).cuda()
            for topk in (1, 2) if numel % 2 == 0 else (1,):
                x = torch.randn(numel // topk, K, generator=gen).to(dtype).cuda()
                idd = ids.view(-1, topk).cuda()
                so, ex, n = fused_moe.moe_align_block_size(idd, 16, E)
                want, got = (torch.full((numel, N), float("nan"), dtype=dtype, device="cuda") for _ in range(2))
                st = torch.cuda.current_stream().cuda_stream
                _lib.check(lib.mi355q_moe_gemm(want.data_ptr(), x.data_ptr(), w.data_ptr(), None, s.data_ptr(), zp.data_ptr(), _lib.ZP_PACKED, 0, g,
                                               rw.data_ptr(), so.data_ptr(), ex.data_ptr(), n.data_ptr(), numel, topk, 16, ex.numel(), E, K, N,
                                               code, code, 0, None, 0, st), "moe_gemm")
                _lib.check(lib.mi355q_moe_w4a16_unsorted(got.data_ptr(), x.data_ptr(), w.data_ptr(), s.data_ptr(), zp.data_ptr(), _lib.ZP_PACKED, g,
                                                         rw.data_ptr(), idd.data_ptr(), int(ids_dtype == torch.int64), numel, topk, E, K, N, 0,
                                                         code, st), "moe_w4a16_unsorted")
                keep = (ids >= 0) & (ids < E)
                assert torch.equal(got[keep.cuda()], want[keep.cuda()]) and got[~keep.cuda()].isnan().all() and not got[keep.cuda()].isnan().any()
                # gate and up in one launch: the operator's own bits of the sums without routing weights
                _lib.check(lib.mi355q_moe_w4a16_unsorted(want.data_ptr(), x.data_ptr(), w.data_ptr(), s.data_ptr(), zp.data_ptr(), _lib.ZP_PACKED, g,
                                                         None, idd.data_ptr(), int(ids_dtype == torch.int64), numel, topk, E, K, N, 0, code, st),
                           "moe_w4a16_unsorted")
                act, glu = (torch.full((numel, N // 2), float("nan"), dtype=dtype, device="cuda") for _ in range(2))
                _lib.check(lib.mi355q_silu_and_mul(act.data_ptr(), want.data_ptr(), numel, N // 2, code, None, 1, st), "silu_and_mul")
                _lib.check(lib.mi355q_moe_w4a16_unsorted(glu.data_ptr(), x.data_ptr(), w.data_ptr(), s.data_ptr(), zp.data_ptr(), _lib.ZP_PACKED, g,
                                                         None, idd.data_ptr(), int(ids_dtype == torch.int64), numel, topk, E, K, N, 1, code, st),
                           "moe_w4a16_unsorted")
                assert torch.equal(glu[keep.cuda()], act[keep.cuda()]) and glu[~keep.cuda()].isnan().all() and not glu[keep.cuda()].isnan().any()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind", ["none", "packed", "pre-scaled"])
@pytest.mark.parametrize("E,K,N,g", [(2, 1152, 256, 384), (1, 1152, 16384, 1152), (1, 640, 32768, 128), (4, 1152, 16384, 128), (4, 512, 16384, 256)])
def test_unsorted_slots_of_every_form(E, K, N, g, kind, dtype):
    """Every workgroup shape with up to nine K blocks (a wavefront then has several or none), groups of one to nine of them, each kind of
    zero-points: the aligned launch against a float64 product, the unsorted one and SiLU of gate and up against it bit for bit."""
    from vllm_gcu_amd import _lib
    from vllm_gcu_amd.kernels import fused_moe
    lib, code = _lib.load(), _lib.F16 if dtype == torch.float16 else _lib.BF16
    gen = torch.Generator(device="cuda").manual_seed(E + K + N)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (E, K // 8, N), dtype=torch.int32, device="cuda", generator=gen)
    s = (torch.rand(E, K // g, N, device="cuda", generator=gen) * 0.009 + 0.001).to(dtype)
    zk, zp = _lib.ZP_NONE, None
    dense = rearrange.unpack_slab(w).to(torch.float32).view(E, K // g, g, N)
    if kind == "packed":
        z = torch.randint(0, 16, (E, K // g, N), dtype=torch.uint8, device="cuda", generator=gen)
        zk = _lib.ZP_PACKED
        zp = torch.stack([rearrange.rearrange_uint4_int32_gptq(w[0], torch.from_numpy(ow4.gptq_pack_zeros(a.cpu().numpy())).cuda())[1] for a in z])
        dense = (dense - z[:, :, None].float()) * s[:, :, None].float()
    elif kind == "pre-scaled":                               # fractions of the scale, as they are
        zk, zp = _lib.ZP_PRESCALED, (s.float() * torch.rand(s.shape, device="cuda", generator=gen) * 15).to(dtype)
        dense = dense * s[:, :, None].float() - zp[:, :, None].float()
    else:
        dense = (dense - 8) * s[:, :, None].float()
    dense = dense.view(E, K, N)
    st = torch.cuda.current_stream().cuda_stream
    for numel, topk in ((1, 1), (5, 1), (18, 2), (60, 1)):
        print(f"case w4a16 unsorted {kind} E={E} K={K} N={N} g={g} numel={numel} {dtype}", flush=True)
        ids = torch.randint(0, E, (numel // topk, topk), device="cuda", generator=gen)
        if numel > 2:
            ids.view(-1)[1], ids.view(-1)[-1] = -1, E
        x = torch.randn(numel // topk, K, device="cuda", generator=gen).to(dtype)
        rw = torch.rand(numel, device="cuda", generator=gen)
        so, ex, n = fused_moe.moe_align_block_size(ids, 16, E)

        def unsorted(weights, glu):
            out = torch.full((numel, N // 2 if glu else N), float("nan"), dtype=dtype, device="cuda")
            _lib.check(lib.mi355q_moe_w4a16_unsorted(out.data_ptr(), x.data_ptr(), w.data_ptr(), s.data_ptr(), None if zp is None else zp.data_ptr(),
                                                     zk, g, None if weights is None else weights.data_ptr(), ids.data_ptr(), 1, numel, topk, E, K,
                                                     N, glu, code, st), "moe_w4a16_unsorted")
            return out
        aligned = torch.full((numel, N), float("nan"), dtype=dtype, device="cuda")
        _lib.check(lib.mi355q_moe_gemm(aligned.data_ptr(), x.data_ptr(), w.data_ptr(), None, s.data_ptr(), None if zp is None else zp.data_ptr(), zk, 0,
                                       g, rw.data_ptr(), so.data_ptr(), ex.data_ptr(), n.data_ptr(), numel, topk, 16, ex.numel(), E, K, N, code,
                                       code, 0, None, 0, st), "moe_gemm")
        flat = ids.view(-1)
        keep = (flat >= 0) & (flat < E)
        got = unsorted(rw, 0)
        assert torch.equal(got[keep], aligned[keep]) and got[~keep].isnan().all()
        rows = keep.nonzero().view(-1).tolist()
        want = torch.stack([(x[r // topk].double() @ dense[flat[r]].double()) * rw[r].double() for r in rows])
        err = float((got[rows].double() - want).norm() / want.norm())
        assert err < (1e-3 if dtype == torch.float16 else 6e-3)                          # one rounding to 16 bits
        if zk != _lib.ZP_PRESCALED:
            plain, glu = unsorted(None, 0), unsorted(None, 1)
            act = torch.full((numel, N // 2), float("nan"), dtype=dtype, device="cuda")
            _lib.check(lib.mi355q_silu_and_mul(act.data_ptr(), plain.data_ptr(), numel, N // 2, code, None, 1, st), "silu_and_mul")
            assert torch.equal(glu[keep], act[keep]) and glu[~keep].isnan().all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("E,K,N,rows,topk,ranges", [(8, 6272, 4096, 2, 2, 2), (8, 6144, 4096, 3, 2, 4), (8, 3072, 4096, 3, 2, 2), (8, 2944, 4096, 3, 2, 1),
                                                    (16, 6272, 3072, 16, 2, 2), (3, 256, 512, 64, 1, 1), (60, 384, 256, 10, 6, 1)])
def test_unsorted_sum(E, K, N, rows, topk, ranges, dtype):
    """The second GEMM whose K ranges and slots are added by one launch: the bits of the GEMM and moe_sum one after the other where every
    sum along K is exact, for the ranges the shape is cut into (also uneven ones)."""
    from vllm_gcu_amd import _lib
    lib, g, numel = _lib.load(), 128, rows * topk
    code = _lib.F16 if dtype == torch.float16 else _lib.BF16
    gen = torch.Generator(device="cuda").manual_seed(E + K + N)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (E, K // 8, N), dtype=torch.int32, device="cuda", generator=gen)
    zp = torch.randint(-2 ** 31, 2 ** 31 - 1, (E, K // g, N // 8), dtype=torch.int32, device="cuda", generator=gen)
    s = (2.0 ** torch.randint(-9, -6, (E, K // g, N), device="cuda", generator=gen)).to(dtype)
    x = torch.randint(-4, 5, (numel, K), device="cuda", generator=gen).to(dtype)
    rw = torch.rand(numel, device="cuda", generator=gen)
    ids = torch.randint(0, E, (rows, topk), device="cuda", generator=gen, dtype=torch.int32)
    st = torch.cuda.current_stream().cuda_stream
    need = lib.mi355q_moe_w4a16_unsorted_sum_bytes(numel, E, K, N)
    assert need == ranges * numel * N * 4
    ws = torch.full((need // 4,), float("nan"), device="cuda")
    got, want = (torch.full((rows, N), float("nan"), dtype=dtype, device="cuda") for _ in range(2))
    slots = torch.empty(numel, N, dtype=dtype, device="cuda")
    common = (w.data_ptr(), s.data_ptr(), zp.data_ptr(), _lib.ZP_PACKED, g, rw.data_ptr(), ids.data_ptr(), 0)
    _lib.check(lib.mi355q_moe_w4a16_unsorted_sum(got.data_ptr(), x.data_ptr(), *common, rows, topk, E, K, N, code, ws.data_ptr(), need, st),
               "moe_w4a16_unsorted_sum")
    _lib.check(lib.mi355q_moe_w4a16_unsorted(slots.data_ptr(), x.data_ptr(), *common, numel, 1, E, K, N, 0, code, st), "moe_w4a16_unsorted")
    _lib.check(lib.mi355q_moe_sum(want.data_ptr(), slots.data_ptr(), rows, topk, N, code, code, None, st), "moe_sum")
    assert torch.equal(got, want)
    assert lib.mi355q_moe_w4a16_unsorted_sum(got.data_ptr(), x.data_ptr(), *common, rows, topk, E, K, N, code, ws.data_ptr(), need - 4, st) != 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("E,K,N,rows,topk", [(8, 6144, 4096, 6, 2), (8, 2944, 4096, 6, 2), (60, 384, 256, 10, 6)])
def test_unsorted_sum_passes_infinities_and_nan(E, K, N, rows, topk, dtype):
    """Rows with an infinity of either sign, a NaN and the largest finite value, and an infinite weight: what the GEMM and moe_sum make of them (exact
    sums elsewhere), and no other token touched by them."""
    from vllm_gcu_amd import _lib
    print(f"case unsorted sum, inf and nan E={E} K={K} N={N} rows={rows} topk={topk} {dtype}", flush=True)
    lib, g, numel = _lib.load(), 128, rows * topk
    code = _lib.F16 if dtype == torch.float16 else _lib.BF16
    gen = torch.Generator(device="cuda").manual_seed(E + K + N)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (E, K // 8, N), dtype=torch.int32, device="cuda", generator=gen)
    s = (2.0 ** torch.randint(-9, -6, (E, K // g, N), device="cuda", generator=gen)).to(dtype)
    x = torch.randint(-4, 5, (numel, K), device="cuda", generator=gen).to(dtype)
    for i, v in enumerate((float("inf"), -float("inf"), float("nan"), torch.finfo(dtype).max)):
        x[topk * i, 61 * i + 3] = v                          # tokens 0 .. 3
    rw = torch.rand(numel, device="cuda", generator=gen)
    rw[topk * 4] = float("inf")                              # token 4
    ids, st = torch.randint(0, E, (rows, topk), device="cuda", generator=gen, dtype=torch.int32), torch.cuda.current_stream().cuda_stream
    need = lib.mi355q_moe_w4a16_unsorted_sum_bytes(numel, E, K, N)
    ws = torch.full((need // 4,), float("nan"), device="cuda")
    got, want = (torch.full((rows, N), 7.0, dtype=dtype, device="cuda") for _ in range(2))
    slots = torch.empty(numel, N, dtype=dtype, device="cuda")
    common = (w.data_ptr(), s.data_ptr(), None, _lib.ZP_NONE, g, rw.data_ptr(), ids.data_ptr(), 0)
    _lib.check(lib.mi355q_moe_w4a16_unsorted_sum(got.data_ptr(), x.data_ptr(), *common, rows, topk, E, K, N, code, ws.data_ptr(), need, st),
               "moe_w4a16_unsorted_sum")
    _lib.check(lib.mi355q_moe_w4a16_unsorted(slots.data_ptr(), x.data_ptr(), *common, numel, 1, E, K, N, 0, code, st), "moe_w4a16_unsorted")
    _lib.check(lib.mi355q_moe_sum(want.data_ptr(), slots.data_ptr(), rows, topk, N, code, code, None, st), "moe_sum")
    assert not got[:3].isfinite().all() and not got[4].isfinite().all()
    for t in range(rows):
        if t == 3:                                           # (sums that are not exact: 2^16 and more beside small products)
            assert torch.equal(got[t].isfinite(), want[t].isfinite())
            fin = want[t].isfinite()
            assert torch.allclose(got[t][fin].double(), want[t][fin].double(), rtol=1e-2)
        else:
            assert torch.equal(got[t].nan_to_num(11.0, 12.0, 13.0), want[t].nan_to_num(11.0, 12.0, 13.0)) and (t < 5 or got[t].isfinite().all())


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("E,K,N,rows,topk", [(8, 6144, 4096, 3, 2), (8, 2944, 4096, 3, 2), (5, 384, 256, 64, 1), (60, 384, 256, 10, 6)])
def test_unsorted_sum_without_slots_of_no_expert(E, K, N, rows, topk, dtype, wide):
    """Slots of ids outside [0, E) add nothing, whatever the workspace held: the bits of the GEMM into zeroed rows and moe_sum."""
    from vllm_gcu_amd import _lib
    print(f"case unsorted sum, dropped slots E={E} K={K} N={N} rows={rows} topk={topk} {dtype} wide={wide}", flush=True)
    lib, g, numel = _lib.load(), 128, rows * topk
    code = _lib.F16 if dtype == torch.float16 else _lib.BF16
    gen = torch.Generator(device="cuda").manual_seed(E + K + N)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (E, K // 8, N), dtype=torch.int32, device="cuda", generator=gen)
    zp = torch.randint(-2 ** 31, 2 ** 31 - 1, (E, K // g, N // 8), dtype=torch.int32, device="cuda", generator=gen)
    s = (2.0 ** torch.randint(-9, -6, (E, K // g, N), device="cuda", generator=gen)).to(dtype)
    x = torch.randint(-4, 5, (numel, K), device="cuda", generator=gen).to(dtype)
    rw = torch.rand(numel, device="cuda", generator=gen)
    ids = torch.randint(0, E, (rows, topk), device="cuda", generator=gen, dtype=torch.int64 if wide else torch.int32)
    ids[0, 0], ids[-1, :], ids[1, -1] = E, -1, E + 3
    rw[0] = float("nan")                                     # (of a slot that adds nothing)
    st = torch.cuda.current_stream().cuda_stream
    need = lib.mi355q_moe_w4a16_unsorted_sum_bytes(numel, E, K, N)
    ws = torch.full((need // 4,), float("nan"), device="cuda")
    got, want = (torch.full((rows, N), float("nan"), dtype=dtype, device="cuda") for _ in range(2))
    slots = torch.zeros(numel, N, dtype=dtype, device="cuda")
    common = (w.data_ptr(), s.data_ptr(), zp.data_ptr(), _lib.ZP_PACKED, g, rw.data_ptr(), ids.data_ptr(), wide)
    _lib.check(lib.mi355q_moe_w4a16_unsorted_sum(got.data_ptr(), x.data_ptr(), *common, rows, topk, E, K, N, code, ws.data_ptr(), need, st),
               "moe_w4a16_unsorted_sum")
    _lib.check(lib.mi355q_moe_w4a16_unsorted(slots.data_ptr(), x.data_ptr(), *common, numel, 1, E, K, N, 0, code, st), "moe_w4a16_unsorted")
    _lib.check(lib.mi355q_moe_sum(want.data_ptr(), slots.data_ptr(), rows, topk, N, code, code, None, st), "moe_sum")
    assert torch.equal(got, want) and (got[-1] == 0).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,N,g", DEEP)
def test_deep_k(K, N, g, dtype):
    """Five to seven K blocks of a wavefront, on either side of the depths where it takes them, one and two tiles."""
    test_rows_1_to_16(K, N, g, dtype)
    test_exact(K, N, g, dtype)
