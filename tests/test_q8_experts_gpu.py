"""fp8 experts of a few tokens without an alignment (csrc/q8_experts.hip) against a float64 evaluation of the quantised sequence: every width of a workgroup and
ring, one and several blocks of an expert's slots, ragged last workgroups, repeated and foreign ids, both id types, output in place of the input."""
import pytest
import torch

from vllm_gcu_amd import _lib
from vllm_gcu_amd.kernels.quantization import rearrange

pytestmark = pytest.mark.gpu
DT = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}
# tokens, slots per token, experts, K, I
SHAPES = [(1, 1, 1, 128, 128), (1, 8, 128, 2304, 1152), (2, 6, 64, 1024, 640), (4, 2, 4, 384, 512), (3, 8, 256, 7168, 2048), (3, 3, 3, 640, 256), (4, 8, 16, 2176, 384),
          (4, 4, 40, 4096, 1024), (2, 2, 2, 32768, 128), (1, 16, 64, 8320, 2432), (4, 16, 128, 2560, 896),
          (1, 1, 2, 131072, 128), (1, 2, 2, 128, 65536), (1, 1, 2, 256, 65664)]


def _quantise(x):
    """Groups of 128: e4m3fn values and scales, as doubles."""
    g = x.float().view(*x.shape[:-1], -1, 128)
    s = g.abs().amax(-1, keepdim=True).clamp_min(1e-10)
    s = s / torch.full_like(s, 448.0)                          # (by a number torch multiplies with its reciprocal)
    q = (g / s).clamp(-448, 448).to(torch.float8_e4m3fn)
    return (q.double() * s.double()).view(x.shape)


def _dense(w, s):
    return w.double() * s.double().repeat_interleave(128, -2).repeat_interleave(128, -1)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,T,E,K,I", SHAPES)
@pytest.mark.parametrize("ids_of", ["distinct", "one expert", "foreign"])
def test_against_the_sequence(M, T, E, K, I, ids_of, dtype):
    print(f"case q8 experts M={M} T={T} E={E} K={K} I={I} {ids_of} {dtype}", flush=True)
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(M * K + I)
    x = torch.randn(M, K, device="cuda", generator=gen).to(dtype)
    w1 = (torch.randn(E, 2 * I, K, device="cuda", generator=gen) * 60).to(torch.float8_e4m3fn)
    w2 = (torch.randn(E, K, I, device="cuda", generator=gen) * 60).to(torch.float8_e4m3fn)
    s1 = (torch.rand(E, 2 * I // 128, K // 128, device="cuda", generator=gen) + 0.5) * (1.0 / 60 / K ** 0.5)
    s2 = (torch.rand(E, K // 128, I // 128, device="cuda", generator=gen) + 0.5) * (1.0 / 60 / I ** 0.5)
    tw = torch.rand(M, T, device="cuda", generator=gen) + 0.1
    if ids_of == "one expert":
        ids = torch.full((M, T), E - 1, device="cuda")                   # (up to 64 slots of one expert: several blocks)
    else:
        ids = torch.stack([torch.randperm(E, device="cuda", generator=gen)[:T] if T <= E else torch.randint(0, E, (T,), device="cuda", generator=gen) for _ in range(M)])
    if ids_of == "foreign":
        ids[0, 0], ids[M - 1, T - 1] = -1, E
    ids = ids.to(torch.int32 if M % 2 else torch.int64).contiguous()
    need = lib.mi355q_moe_fp8_unsorted_bytes(M, T, E, K, I)
    assert need == M * T * (2 * I + K) * 2
    ws = torch.full((need,), 0xff, dtype=torch.uint8, device="cuda")     # NaN wherever nothing is written
    want = torch.zeros(M, K, dtype=torch.float64, device="cuda")
    xq = _quantise(x)
    for m in range(M):
        for t in range(T):
            e = int(ids[m, t])
            if 0 <= e < E:
                gu = (xq[m] @ _dense(w1[e], s1[e]).t()).to(dtype).float()
                act = (torch.nn.functional.silu(gu[:I]) * gu[I:]).to(dtype)
                want[m] += (_quantise(act) @ _dense(w2[e], s2[e]).t()) * tw[m, t].double()
    out, k1, k2 = x.clone(), rearrange.to_kslab(w1), rearrange.to_kslab(w2)
    rc = lib.mi355q_moe_fp8_unsorted(out.data_ptr(), out.data_ptr(), k1.data_ptr(), s1.data_ptr(), k2.data_ptr(), s2.data_ptr(),
                                     tw.data_ptr(), ids.data_ptr(), int(ids.dtype == torch.int64), M, T, E, K, I, DT[dtype], ws.data_ptr(), need,
                                     torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    _lib.check(rc, "moe_fp8_unsorted")
    # a sum that rounds the other way to 16 bits moves an intermediate value by a step of e4m3fn, 2^-4 of it at most, now and then: some of I values
    assert (out.double() - want).norm() <= 1e-2 * want.norm() + 1e-30
    if ids_of == "foreign" and M == T == 1:
        assert not out.any()


def test_what_is_not_covered():
    lib = _lib.load()
    need = lib.mi355q_moe_fp8_unsorted_bytes
    assert need(5, 1, 8, 1024, 1024) == 0 and need(4, 17, 128, 1024, 1024) == 0 and need(1, 1, 8, 1024 + 64, 1024) == 0 and need(4, 1, 8, 32768 + 128, 128) == 0
    assert need(1, 2, 8, 65536, 128) and not need(1, 2, 8, 65536 + 128, 128) and need(1, 1, 8, 128, 131072) and not need(1, 1, 8, 128, 131072 + 128)
    assert lib.mi355q_moe_fp8_unsorted_wanted(1, 8, 256, 7168, 2048) and not lib.mi355q_moe_fp8_unsorted_wanted(4, 8, 256, 7168, 2048)
    x = torch.zeros(1024, dtype=torch.uint8, device="cuda").data_ptr()
    assert lib.mi355q_moe_fp8_unsorted(x, x, x, x, x, x, x, x, 0, 1, 1, 1, 128, 128, _lib.BF16, x, 8, None) != 0         # workspace too small
    assert lib.mi355q_moe_fp8_unsorted(x, x + 2, x, x, x, x, x, x, 0, 1, 1, 1, 128, 128, _lib.BF16, x, 1024, None) != 0
