"""The W4A16 kernel for a few dozen to some hundred rows (csrc/w4a16_rows.hip): every tile it has at row counts around the
tile's edges, odd and even numbers of K blocks (one range of a workgroup then holds one less, or none), K split over
workgroups, column tiles that are and are not a multiple of eight, groups of 32 to K, every kind of zero-points, bias, and
exact inputs bit for bit; then the choice the library makes by itself."""
import numpy as np
import pytest
import torch

from oracle import w4 as ow4
from vllm_gcu_amd.kernels import _custom_ops as ops
from vllm_gcu_amd.kernels.quantization import rearrange

pytestmark = pytest.mark.gpu
TILES = [(2, 1), (3, 1), (4, 1), (2, 2), (3, 2), (4, 2), (5, 2), (6, 2)]     # rows / 16, columns / 64
# (K, N, group, K ranges)
SHAPES = [(128, 128, 128, 1), (384, 1024, 128, 1), (1280, 384, 256, 1), (2304, 640, 64, 2), (1152, 256, 32, 3), (1024, 512, 1024, 4)]


def _case(seed, M, K, N, g, dtype, exact=False):
    rng = np.random.default_rng(seed)
    q = rng.integers(0, 16, size=(K, N), dtype=np.uint8)
    z = rng.integers(0, 16, size=(K // g, N), dtype=np.uint8)
    s = 2.0 ** -rng.integers(4, 8, size=(K // g, N)) if exact else rng.uniform(0.001, 0.01, size=(K // g, N))
    x = rng.integers(-4, 5, size=(M, K)) if exact else rng.standard_normal((M, K))
    return q, z, torch.from_numpy(s.astype(np.float32)).to(dtype), torch.from_numpy(x.astype(np.float32)).to(dtype)


def _want(q, z, s, x, g, bias=None):
    return ow4.w4a16_gemm(x.float().numpy(), q, z, s.float().numpy(), g, bias=None if bias is None else bias.float().numpy())


def _run(q, z, s, x, g, bias=None, **kw):
    w, zp = rearrange.rearrange_uint4_int32_gptq(torch.from_numpy(ow4.gptq_pack_weight(q)).cuda(),
                                                 None if z is None else torch.from_numpy(ow4.gptq_pack_zeros(z)).cuda())
    out = torch.full((x.shape[0], q.shape[1]), float("nan"), dtype=x.dtype, device="cuda")
    return ops.w4a16_gemm(x.cuda(), w, s.cuda(), zp, None if bias is None else bias.cuda(), g, out=out, **kw).cpu()


def _close(got, want):
    np.testing.assert_allclose(got.float().numpy(), want, rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,N,g,splits", SHAPES)
@pytest.mark.parametrize("mt,nt", TILES)
def test_tiles(mt, nt, K, N, g, splits, dtype, monkeypatch):
    kw = dict(family=4, split_k=splits | mt << 8 | nt << 16)
    for M in (1, 16 * mt - 15, 16 * mt, 16 * mt + 1, 40 * mt):
        print(f"case w4a16 rows {16 * mt}x{64 * nt} M={M} K={K} N={N} g={g} splits={splits} {dtype}", flush=True)
        q, z, s, x = _case(M + K, M, K, N, g, dtype)
        bias = torch.randn(N, generator=torch.Generator().manual_seed(M)).to(dtype)
        _close(_run(q, z, s, x, g, bias, **kw), _want(q, z, s, x, g, bias))
        _close(_run(q, None, s, x, g, **kw), _want(q, None, s, x, g))
    # z * s in the activation type, as some checkpoints hold it: the kernel recovers the integer
    monkeypatch.setattr(ops, "_RECOVER_INTEGER_ZEROS", False)
    w, _ = rearrange.rearrange_uint4_int32_gptq(torch.from_numpy(ow4.gptq_pack_weight(q)).cuda(), None)
    zs = (torch.from_numpy(z.astype(np.float32)) * s.float()).to(dtype)
    _close(ops.w4a16_gemm(x.cuda(), w, s.cuda(), zs.cuda(), None, g, **kw).cpu(), _want(q, z, s, x, g))
    q, z, s, x = _case(5, 16 * mt + 3, K, N, g, dtype, exact=True)
    assert torch.equal(_run(q, z, s, x, g, **kw), torch.from_numpy(_want(q, z, s, x, g)).to(dtype))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("g", [128, 32])
@pytest.mark.parametrize("mt,nt", [(2, 1), (3, 1), (2, 2)])
def test_one_and_two_workgroups_per_cu(mt, nt, g, dtype):
    """The tiles that fit twice on a CU have a ring for it and another for a launch of no more workgroups than CUs (test_tiles' are all of those): on both
    sides of the line, with fewer K blocks than either ring has stages and with more."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for K, tiles in ((128, cus), (128, cus + 2), (1152, cus), (1152, cus + 2)):
        M, N = 16 * mt - 3, tiles * 64 * nt
        print(f"case w4a16 rows {16 * mt}x{64 * nt} M={M} K={K} N={N} g={g} {dtype}", flush=True)
        q, z, s, x = _case(K + mt, M, K, N, g, dtype, exact=True)
        assert torch.equal(_run(q, z, s, x, g, family=4, split_k=1 | mt << 8 | nt << 16), torch.from_numpy(_want(q, z, s, x, g)).to(dtype))


@pytest.mark.parametrize("M,K,N,g", [(5, 1024, 1024, 64), (20, 4096, 16384, 128), (24, 2048, 512, 32), (33, 1024, 128, 128),
                                     (48, 4096, 1024, 128), (64, 2048, 4096, 128), (65, 3584, 512, 128), (96, 1024, 14336, 128),
                                     (130, 2048, 1024, 64), (333, 1024, 2048, 128), (700, 1024, 1024, 128), (4095, 512, 128, 128),
                                     (4096, 512, 128, 64), (4097, 512, 128, 64)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_automatic(M, K, N, g, dtype):
    """What the library takes by itself equals this kernel's result (its sums are exact on these inputs, so they prove
    that the numbers are right whatever it took)."""
    print(f"case w4a16 rows automatic M={M} K={K} N={N} g={g} {dtype}", flush=True)
    q, z, s, x = _case(M, M, K, N, g, dtype, exact=True)
    want = torch.from_numpy(_want(q, z, s, x, g)).to(dtype)
    assert torch.equal(_run(q, z, s, x, g), want)
    assert torch.equal(_run(q, z, s, x, g, family=4), want)


@pytest.mark.parametrize("M,K,N,g,dtype", [(170, 28672, 8192, 128, torch.bfloat16), (1536, 4096, 6144, 64, torch.bfloat16),
                                           (333, 7168, 9344, 64, torch.bfloat16), (700, 5120, 5120, 32, torch.bfloat16),
                                           (256, 3584, 37888, 32, torch.float16), (700, 5120, 5120, 64, torch.float16)])
def test_taken_where_the_tiles_loop_is_the_slow_one(M, K, N, g, dtype):
    """The 64-row tiles run a slower loop for groups of 64 and 32 and for bf16 rows that are not staged as fp16; this kernel is 18 to 40 %
    ahead of it at these shapes.  Sums in another order round differently, so equal bits say which kernel ran."""
    print(f"case w4a16 slow loop M={M} K={K} N={N} g={g} {dtype}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(M)
    w, zp = (torch.randint(-2**31, 2**31, shape, dtype=torch.int32, device="cuda", generator=gen) for shape in ((K // 8, N), (K // g, N // 8)))
    scales = (torch.rand(K // g, N, device="cuda", generator=gen) * 0.01).to(dtype)
    x = torch.randn(M, K, device="cuda", generator=gen).to(dtype)
    assert torch.equal(ops.w4a16_gemm(x, w, scales, zp, None, g), ops.w4a16_gemm(x, w, scales, zp, None, g, family=4))


@pytest.mark.parametrize("N", [7168, 8192])
@pytest.mark.parametrize("M", [16, 24])
def test_streaming_kernel_halves_of_slabs_in_two_ranges(M, N):
    """Dealt out to the XCDs by slabs, and in turn where they fill the chip: every column is written either way."""
    print(f"case w4a16 stream halves M={M} N={N}", flush=True)
    q, z, s, x = _case(M + N, M, 1024, N, 128, torch.float16, exact=True)
    assert torch.equal(_run(q, z, s, x, 128, family=1, split_k=2 | 4 << 8), torch.from_numpy(_want(q, z, s, x, 128)).half())


@pytest.mark.parametrize("M,K,N,dtype,family", [(17, 2560, 14336, torch.float16, 4), (32, 1408, 19328, torch.float16, 4), (24, 7168, 2560, torch.float16, 1),
                                                (32, 14080, 4352, torch.float16, 1), (30, 14336, 4096, torch.bfloat16, 1), (24, 2432, 18944, torch.bfloat16, 4)])
def test_17_to_32_rows_without_a_second_launch(M, K, N, dtype, family):
    """Wide layers come here unsplit; those that K ranges would serve stay with the streaming kernel, one launch (K in another order, so equal bits say which ran)."""
    print(f"case w4a16 17..32 rows M={M} K={K} N={N} {dtype}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(M)
    w, zp = (torch.randint(-2**31, 2**31, shape, dtype=torch.int32, device="cuda", generator=gen) for shape in ((K // 8, N), (K // 128, N // 8)))
    scales = (torch.rand(K // 128, N, device="cuda", generator=gen) * 0.01).to(dtype)
    x = torch.randn(M, K, device="cuda", generator=gen).to(dtype)
    assert torch.equal(ops.w4a16_gemm(x, w, scales, zp, None, 128), ops.w4a16_gemm(x, w, scales, zp, None, 128, family=family))


def test_activations_of_four_gib():
    """The last row below 4 GiB of activations is addressed in 32 bits; from 4 GiB on the problem is refused."""
    K, N, M = 1 << 24, 128, 127
    print(f"case w4a16 rows M={M} K={K} N={N}", flush=True)
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 24 << 30:
        pytest.skip("needs 24 GiB of GPU memory")
    q, z, s, x = _case(1, M, 256, N, 128, torch.float16, exact=True)
    packed = torch.zeros(K // 8, N, dtype=torch.int32, device="cuda")
    packed[-32:] = torch.from_numpy(ow4.gptq_pack_weight(q)).cuda()
    zeros = torch.zeros(K // 128, N // 8, dtype=torch.int32, device="cuda")
    zeros[-2:] = torch.from_numpy(ow4.gptq_pack_zeros(z)).cuda()
    w, zp = rearrange.rearrange_uint4_int32_gptq(packed, zeros)
    del packed
    scales = torch.ones(K // 128, N, dtype=torch.float16, device="cuda")
    scales[-2:] = s.cuda()
    xs = torch.zeros(M + 1, K, dtype=torch.float16, device="cuda")
    xs[:M, -256:] = x.cuda()
    got = ops.w4a16_gemm(xs[:M], w, scales, zp, None, 128, family=4)
    assert torch.equal(got.cpu(), torch.from_numpy(_want(q, z, s, x, 128)).half())
    for family in (0, 4):
        with pytest.raises(RuntimeError, match="4 GiB"):
            ops.w4a16_gemm(xs, w, scales, zp, None, 128, family=family)
