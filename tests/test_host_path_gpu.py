"""The native host path (csrc/host/module.cpp) against the general Python path of the same methods: the same
kernels run on the same operands, so the outputs are equal bit for bit; operands the kernels cannot read as they
are are declined and still give the general path's result."""
import pytest
import torch

pytestmark = pytest.mark.gpu
K, N = 512, 384


@pytest.fixture(autouse=True)
def _seed():
    torch.manual_seed(3)


def _layer(method, dtype, **kw):
    layer = torch.nn.Module()
    with torch.device("cuda"):
        method.create_weights(layer, K, [N], K, N, dtype, **kw)
    return layer


def _int4(which, dtype):
    from vllm_gcu_amd.kernels.quantization import awq, gptq
    m = (gptq.GPTQGCUConfig(4, 128) if which == "gptq" else awq.AWQGCUConfig(4, 128)).get_quant_method()
    layer = _layer(m, dtype)
    layer.qweight.data.random_()
    layer.qzeros.data.random_()
    layer.scales.data.uniform_(0.001, 0.01)
    m.process_weights_after_loading(layer)
    return m, layer, m.apply


def _int8(which, dtype):
    from vllm_gcu_amd.kernels.quantization import w8a8
    if which == "int8 static":
        m = w8a8.W8A8Config().get_quant_method()
        layer = _layer(m, dtype)
        layer.in_scales.data.uniform_(0.02, 0.04)
        layer.out_scales.data.uniform_(0.0001, 0.0005)
        apply = m.apply
    else:
        m, layer = w8a8.CompressedTensorMMLinearKernel(), torch.nn.Module()
        layer.weight = torch.nn.Parameter(torch.empty(N, K, dtype=torch.int8, device="cuda"), requires_grad=False)
        layer.weight_scale = torch.nn.Parameter(torch.rand(N, 1, device="cuda") * 0.01, requires_grad=False)
        apply = m.apply_weights
    layer.weight.data.random_(-127, 128)
    m.process_weights_after_loading(layer)
    return m, layer, apply


def _fp8(which, dtype):
    from vllm_gcu_amd.kernels.quantization import fp8
    block = which == "fp8 block"
    scheme = "static" if which == "fp8 static" else "dynamic"
    m = fp8.Fp8GCUConfig((128, 128) if block else None, scheme).get_quant_method()
    layer = _layer(m, dtype)
    layer.weight.data.copy_(torch.randn(N, K, device="cuda") * 50)
    if block:
        layer.weight_scale_inv.data.uniform_(0.001, 0.002)
    else:
        layer.weight_scale.data.fill_(0.001)
        if scheme == "static":
            layer.input_scale.data.fill_(0.01)
    m.process_weights_after_loading(layer)
    return m, layer, m.apply


MAKE = {"gptq": _int4, "awq": _int4, "int8 static": _int8, "int8 dynamic": _int8, "fp8 block": _fp8, "fp8 token": _fp8,
        "fp8 static": _fp8}


@pytest.mark.parametrize("M", [1, 40, 300])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("which", sorted(MAKE))
def test_linear_methods_match_the_general_path(which, dtype, M, monkeypatch):
    from vllm_gcu_amd.kernels import _custom_ops as ops
    print(f"case host path {which} {dtype} M={M}", flush=True)
    _, layer, apply = MAKE[which](which, dtype)
    wide = torch.randn(M, 2 * K, device="cuda", dtype=dtype)
    bias = torch.randn(N, device="cuda", dtype=dtype)
    for x in (wide[:, :K].contiguous(), wide[:, :K].contiguous().reshape(1, M, K), wide[:, K:]):    # the last one strided
        for b in (None, bias):
            got = [apply(layer, x, b) for _ in range(2)][-1]      # (the first call may verify and convert)
            with monkeypatch.context() as mp:
                mp.setattr(ops, "eager", lambda: False)
                want = apply(layer, x, b)
            assert got.shape == want.shape and got.dtype == want.dtype
            assert torch.equal(got, want)


@pytest.mark.parametrize("M", [1, 5, 70])
@pytest.mark.parametrize("which", ["w4a16", "w4a16 bf16", "fp8", "int8"])
def test_fused_experts_match_the_general_path(which, M, monkeypatch):
    from vllm_gcu_amd.kernels import _custom_ops as ops
    from vllm_gcu_amd.kernels.quantization import fp8, moe_wna16, w8a8
    print(f"case host path experts {which} M={M}", flush=True)
    E, H, I, T = 8, 256, 384, 2
    dtype = torch.bfloat16 if which in ("fp8", "w4a16 bf16") else torch.float16
    m = (fp8.Fp8GCUConfig().get_quant_method(moe=True) if which == "fp8" else
         w8a8.W8A8Config().get_quant_method(moe=True) if which == "int8" else
         moe_wna16.MoeWNA16GCUConfig("gptq", 4, 128, True).get_quant_method())
    layer = torch.nn.Module()
    with torch.device("cuda"):
        m.create_weights(layer, E, H, I, dtype)
    for name, p in layer.named_parameters():
        if p.dtype == torch.float8_e4m3fn:
            p.data.copy_(torch.randn(p.shape, device="cuda") * 50)
        elif name.endswith("g_idx"):
            p.data.copy_((torch.arange(p.shape[1], device="cuda") // 128).expand_as(p))
        elif p.dtype in (torch.int32, torch.int8):
            p.data.random_()
        else:
            p.data.uniform_(0.001, 0.002)
    m.process_weights_after_loading(layer)
    x, logits = torch.randn(M, H, device="cuda", dtype=dtype), torch.randn(M, E, device="cuda")
    for kw in (dict(), dict(use_grouped_topk=True, num_expert_group=4, topk_group=2)):
        a, b = x.clone(), x.clone()
        got = m.apply(layer, a, logits, T, True, **kw)
        with monkeypatch.context() as mp:
            mp.setattr(ops, "eager", lambda: False)
            want = m.apply(layer, b, logits, T, True, **kw)
        assert got.data_ptr() == a.data_ptr() and torch.isfinite(want).all()
        assert torch.equal(got, want)


def test_declined_operands():
    from vllm_gcu_amd.kernels import _runtime as rt
    _, layer, apply = _int4("awq", torch.float16)
    x = torch.randn(2, K, device="cuda", dtype=torch.float16)
    h = rt.host
    args = (layer.qweight, layer.qzeros, layer.scales, None, None, 128)
    assert h.w4a16(x, *args) is not None
    for bad in (x.cpu(), x.float(), x[:, :K - 128], x[:0], torch.randn(2, 2 * K, device="cuda").half()[:, :K], None):
        assert h.w4a16(bad, *args) is None
    assert h.w4a16(x, layer.qweight, layer.qzeros, layer.scales[:1], None, None, 128) is None       # too few scales
    assert h.w4a16(x, layer.qweight, layer.qzeros, layer.scales, None, x[0, :8], 128) is None       # too short a bias
    g = torch.arange(K, device="cuda", dtype=torch.int32) // 128
    assert h.w4a16(x, layer.qweight, layer.qzeros, layer.scales, g, None, 128) is None              # not verified yet
    with torch.enable_grad():
        assert h.w4a16(x.clone().requires_grad_(), *args) is None

OPERATOR = {"gptq": "gptq_gemm_gcu", "awq": "awq_gemm_gcu", "int8 static": "dot_bias_quant", "int8 dynamic": "cutlass_scaled_mm",
            "fp8 block": "linear_quant", "fp8 token": "cutlass_scaled_mm", "fp8 static": "cutlass_scaled_mm"}


def _traced_or_refused(fn, a, b):
    """torch.jit.trace of ``fn`` on ``a`` computes ``fn(b)`` too; -> False where torch refuses to trace (it does not take
    operators whose schema writes to a plain ``Tensor!``).  What must not happen is a result recorded as a constant."""
    try:
        traced = torch.jit.trace(fn, (a,), check_trace=False)
    except RuntimeError as e:
        assert "observable data dependence" not in str(e)
        return False
    assert torch.equal(traced(b), fn(b)) and torch.equal(traced(a), fn(a))
    return True


@pytest.mark.parametrize("which", sorted(MAKE))
def test_tracing_sees_the_operator(which):
    print(f"case host path traced {which}", flush=True)
    _, layer, apply = MAKE[which](which, torch.float16)
    a, b = (torch.randn(5, K, device="cuda", dtype=torch.float16) for _ in range(2))
    apply(layer, a, None)                                       # (may verify and convert)
    traced = _traced_or_refused(lambda t: apply(layer, t, None) + t[:, :1], a, b)
    assert traced or which not in ("gptq", "awq")


@pytest.mark.parametrize("grouped", [False, True])
def test_tracing_sees_the_routing(grouped):
    from vllm_gcu_amd.kernels import fused_moe as fmoe
    print(f"case host path traced routing grouped={grouped}", flush=True)
    a, b = (torch.randn(5, 8, device="cuda") for _ in range(2))
    for i in (0, 1):
        _traced_or_refused(lambda g: fmoe.select_experts(g, g, 2, grouped, True, topk_group=2, num_expert_group=4)[i] + g[:, :2], a, b)


@pytest.mark.parametrize("which", sorted(MAKE))
def test_subclasses_and_function_modes_see_the_operator(which):
    print(f"case host path overridden {which}", flush=True)
    seen = []

    class Seen(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return super().__torch_function__(func, types, args, kwargs or {})

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    _, layer, apply = MAKE[which](which, torch.float16)
    x = torch.randn(5, K, device="cuda", dtype=torch.float16)
    want = [apply(layer, x, None) for _ in range(2)][-1]
    got = apply(layer, x.as_subclass(Seen), None)
    assert any(OPERATOR[which] in s for s in seen) and torch.equal(got.as_subclass(torch.Tensor), want)
    seen.clear()
    with Mode():
        got = apply(layer, x, None)
    assert any(OPERATOR[which] in s for s in seen) and torch.equal(got, want)
    # a parameter class that leaves torch's functions alone, and a default device, are nothing to stand aside for
    class Weight(torch.nn.Parameter):
        pass
    from vllm_gcu_amd.kernels import _runtime as rt
    if which == "awq":
        qw = Weight(layer.qweight.data, requires_grad=False)
        with torch.device("cuda"):
            assert torch.equal(rt.host.w4a16(x, qw, layer.qzeros, layer.scales, None, None, 128), want)


@pytest.mark.parametrize("which", ["gptq", "awq"])
def test_vmap(which):
    print(f"case host path vmap {which}", flush=True)
    _, layer, apply = MAKE[which](which, torch.float16)
    x = torch.randn(3, 5, K, device="cuda", dtype=torch.float16)
    want = torch.stack([apply(layer, t, None) for t in x])
    assert torch.equal(torch.vmap(lambda t: apply(layer, t, None))(x), want)
