"""The work that a serving program has this package do, as cases that can be timed.

A case is a plain dict; ``kind`` says which public entry points a pass goes through:

* ``w4a16_linear`` -- one int4 linear layer (GPTQ or AWQ checkpoint) through its quantization method;
* ``w4a16_layer``  -- the quantized part of one decoder layer with int4 weights: norm, qkv, o, norm, gate_up,
  SiLU gate, down (attention itself is not part of this package: its output is an input of the pass);
* ``int8_linear``  -- one W8A8 layer: activation quantisation (static per channel or dynamic per token) and GEMM;
* ``fp8_mlp``      -- one gated MLP with 128 x 128 block-scaled fp8 weights and the fused norm + quantise and
  SiLU + quantise prologues;
* ``fp8_linear``   -- one fp8 layer with per-token activation and per-channel weight scales;
* ``moe_w4a16``    -- one fused-MoE layer with int4 experts: norm, routing, alignment, both expert GEMMs, sum;
* ``moe_fp8``      -- the same with block-scaled fp8 experts and grouped top-k routing.

Layers are made by the methods' own ``create_weights`` and ``process_weights_after_loading``, as a model loader
makes them; weights and activations are synthetic, with the distributions of BASELINE.json's configurations.
"""
import math

import torch

from vllm_gcu_amd.kernels import _custom_ops as ops
from vllm_gcu_amd.kernels.quantization.awq import AWQGCUConfig
from vllm_gcu_amd.kernels.quantization.fp8 import Fp8GCUConfig
from vllm_gcu_amd.kernels.quantization.gptq import GPTQGCUConfig
from vllm_gcu_amd.kernels.quantization.moe_wna16 import MoeWNA16GCUConfig
from vllm_gcu_amd.kernels.quantization.w8a8 import CompressedTensorMMLinearKernel, W8A8Config

DEVICE = "cuda"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
EPS = 1e-6

# (hidden, qkv columns, intermediate) of decoder layers: Llama-3-8B, Llama-2-7B, Qwen2-7B, and generic ones
LAYERS = [(4096, 6144, 14336), (4096, 12288, 11008), (3584, 4608, 18944), (2048, 3072, 5632), (5120, 7168, 13824)]
# (K, N) of single linear layers, from the same models, Llama-3-70B, DeepSeek-V3 and generic ones
LINEARS = [(4096, 6144), (4096, 4096), (4096, 28672), (14336, 4096), (8192, 10240), (8192, 8192), (8192, 28672),
           (3584, 4608), (3584, 37888), (18944, 3584), (5120, 13824), (2048, 11008), (7168, 4096), (2048, 7168),
           (11008, 4096), (1024, 1024), (6144, 2048)]


def listed():
    return [
        # one token through the o projection of Llama-3-8B: the smallest call there is, once per layer and token
        dict(name="w4a16 linear, 1 token", kind="w4a16_linear", tokens=1, K=4096, N=4096, group=128, method="gptq",
             dtype="f16", bias=False),
        # a decode step of 16 sequences through one Llama-3-8B layer from an AWQ checkpoint
        dict(name="w4a16 layer, decode 16", kind="w4a16_layer", tokens=16, hidden=4096, qkv=6144, inter=14336,
             group=128, method="awq", dtype="bf16", bias=False),
        # a chunk of prefill tokens beside running decodes: an odd number of rows, qkv with a bias (Qwen2-7B)
        dict(name="w4a16 layer, chunk of 333", kind="w4a16_layer", tokens=333, hidden=3584, qkv=4608, inter=18944,
             group=128, method="gptq", dtype="f16", bias=True),
        # prefill of 2048 tokens through the largest linear of Llama-3-8B
        dict(name="w4a16 linear, prefill 2048", kind="w4a16_linear", tokens=2048, K=4096, N=28672, group=128,
             method="gptq", dtype="f16", bias=False),
        # int8 decode of 24 sequences, qkv of Qwen2-7B with its bias, static activation scales
        dict(name="int8 linear, decode 24", kind="int8_linear", tokens=24, K=3584, N=4608, scheme="static",
             dtype="bf16", bias=True),
        # int8 prefill of one Llama-3-70B MLP layer, dynamic per-token activation scales
        dict(name="int8 linear, prefill 2048", kind="int8_linear", tokens=2048, K=8192, N=28672, scheme="dynamic",
             dtype="f16", bias=False),
        # the shared expert of a DeepSeek-V3-style layer: a decode batch, and a ragged prefill batch
        dict(name="fp8 mlp, decode 48", kind="fp8_mlp", tokens=48, hidden=7168, inter=2048),
        dict(name="fp8 mlp, prefill 1537", kind="fp8_mlp", tokens=1537, hidden=7168, inter=2048),
        # speculative decoding / many sequences: a row count just above a tile, down projection of Llama-3-8B
        dict(name="fp8 linear, 130 tokens", kind="fp8_linear", tokens=130, K=14336, N=4096, dtype="bf16", bias=False),
        # a few decoding sequences, and a prefill batch, through one Mixtral-8x7B layer
        dict(name="moe w4a16, decode 5", kind="moe_w4a16", tokens=5, hidden=4096, inter=14336, experts=8, topk=2,
             group=128, dtype="f16"),
        dict(name="moe w4a16, prefill 512", kind="moe_w4a16", tokens=512, hidden=4096, inter=14336, experts=8, topk=2,
             group=128, dtype="f16"),
        # a decode batch through one DeepSeek-V3-style layer: nearly every expert's weights are read
        dict(name="moe fp8, decode 256", kind="moe_fp8", tokens=256, hidden=7168, inter=2048, experts=256, topk=8,
             groups=8, topk_group=4),
    ]


def _tokens(rng, top):
    """1 .. top, spread over the logarithm; whole powers of two as often as serving pads batches to them."""
    if rng.random() < 0.2:
        return 1 << rng.randint(0, int(math.log2(top)))
    return max(1, min(top, int(round(math.exp(rng.uniform(0.0, math.log(top)))))))


def _dim(rng, low, high):
    """A multiple of 128, spread over the logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high))) / 128)) * 128))


def _linear_shape(rng):
    return rng.choice(LINEARS) if rng.random() < 0.5 else (_dim(rng, 1024, 16384), _dim(rng, 1024, 28672))


def draw(rng):
    kind = rng.choice(["w4a16_linear", "w4a16_layer", "int8_linear", "fp8_mlp", "fp8_linear", "moe_w4a16", "moe_fp8"])
    dtype = rng.choice(["f16", "bf16"])
    if kind == "w4a16_linear":
        K, N = _linear_shape(rng)
        return dict(kind=kind, tokens=_tokens(rng, 2048), K=K, N=N, group=rng.choice([128, 128, 128, 64]),
                    method=rng.choice(["gptq", "awq"]), dtype=dtype, bias=rng.random() < 0.25)
    if kind == "w4a16_layer":
        h, q, i = rng.choice(LAYERS) if rng.random() < 0.6 else (_dim(rng, 2048, 5120), _dim(rng, 3072, 8192),
                                                                 _dim(rng, 5632, 14336))
        return dict(kind=kind, tokens=_tokens(rng, 2048), hidden=h, qkv=q, inter=i, group=128,
                    method=rng.choice(["gptq", "awq"]), dtype=dtype, bias=rng.random() < 0.25)
    if kind == "int8_linear":
        K, N = _linear_shape(rng)
        return dict(kind=kind, tokens=_tokens(rng, 2048), K=K, N=N, scheme=rng.choice(["static", "dynamic"]),
                    dtype=dtype, bias=rng.random() < 0.25)
    if kind == "fp8_mlp":
        return dict(kind=kind, tokens=_tokens(rng, 2048), hidden=rng.choice([7168, _dim(rng, 2048, 8192)]),
                    inter=rng.choice([2048, _dim(rng, 1024, 8192)]))
    if kind == "fp8_linear":
        K, N = _linear_shape(rng)
        return dict(kind=kind, tokens=_tokens(rng, 2048), K=K, N=N, dtype=dtype, bias=rng.random() < 0.25)
    if kind == "moe_w4a16":
        h, i, e, t = rng.choice([(4096, 14336, 8, 2), (2048, 1408, 60, 4), (2048, 1024, 64, 6),
                                 (_dim(rng, 1024, 4096), _dim(rng, 1024, 8192), 16, 2)])
        return dict(kind=kind, tokens=_tokens(rng, 1024), hidden=h, inter=i, experts=e, topk=t, group=128, dtype=dtype)
    h, i, e = rng.choice([(7168, 2048, 256), (7168, 2048, 64), (_dim(rng, 2048, 7168), _dim(rng, 512, 2048), 128)])
    return dict(kind=kind, tokens=_tokens(rng, 256), hidden=h, inter=i, experts=e, topk=rng.choice([6, 8]), groups=8,
                topk_group=4)


# --- what a program has in hand before the call ------------------------------------------------------------
def _uniform(gen, shape, low, high, dtype):
    return (torch.rand(shape, generator=gen, device=DEVICE) * (high - low) + low).to(dtype)


def _normal(gen, shape, std, dtype):
    return torch.empty(shape, dtype=dtype, device=DEVICE).normal_(0.0, std, generator=gen)


def _bits(gen, t):
    """Random bytes: int4 weights and zero-points uniform over 0 .. 15, int8 weights uniform."""
    raw = t.view(torch.uint8).view(-1)
    raw.random_(0, 256, generator=gen)


def _int4_linear(gen, method, K, N, dtype):
    layer = torch.nn.Module()
    with torch.device(DEVICE):
        method.create_weights(layer, K, [N], K, N, dtype)
    _bits(gen, layer.qweight.data)
    _bits(gen, layer.qzeros.data)
    layer.scales.data.copy_(_uniform(gen, layer.scales.shape, 0.001, 0.01, dtype))
    method.process_weights_after_loading(layer)
    return layer


def _fp8_codes(gen, t):
    """Block-scaled codes of weights ~ N(0, 0.02): the largest of a block of 16384 lies near four deviations."""
    for part in t.view(-1).split(1 << 29):
        part.copy_(_normal(gen, part.shape, 112.0, torch.bfloat16).clamp_(-448.0, 448.0))


def _block_scales(gen, t):
    t.copy_(_uniform(gen, t.shape, 0.9, 1.1, torch.float32) * (0.08 / 448.0))


def _int4_method(case):
    return (GPTQGCUConfig(4, case["group"]) if case["method"] == "gptq" else AWQGCUConfig(4, case["group"])).get_quant_method()


def _fp8_linear_layer(gen, method, K, N, dtype):
    layer = torch.nn.Module()
    with torch.device(DEVICE):
        method.create_weights(layer, K, [N], K, N, dtype)
    _fp8_codes(gen, layer.weight.data)
    if method.block_quant:
        _block_scales(gen, layer.weight_scale_inv.data)
    else:
        layer.weight_scale = torch.nn.Parameter(_uniform(gen, (N,), 0.9, 1.1, torch.float32) * (0.08 / 448.0),
                                                requires_grad=False)
    method.process_weights_after_loading(layer)
    return layer


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind, M = case["kind"], case["tokens"]
    dtype = DTYPES[case.get("dtype", "bf16")]
    s = {"kind": kind}
    if kind == "w4a16_linear":
        s["method"] = _int4_method(case)
        s["layer"] = _int4_linear(gen, s["method"], case["K"], case["N"], dtype)
        s["x"] = _normal(gen, (M, case["K"]), 1.0, dtype)
        s["bias"] = _normal(gen, (case["N"],), 1.0, dtype) if case["bias"] else None
    elif kind == "w4a16_layer":
        H, Q, I = case["hidden"], case["qkv"], case["inter"]
        s["method"] = m = _int4_method(case)
        s["qkv"], s["o"] = _int4_linear(gen, m, H, Q, dtype), _int4_linear(gen, m, H, H, dtype)
        s["gate_up"], s["down"] = _int4_linear(gen, m, H, 2 * I, dtype), _int4_linear(gen, m, I, H, dtype)
        s["norm1"], s["norm2"] = _uniform(gen, (H,), 0.5, 1.5, dtype), _uniform(gen, (H,), 0.5, 1.5, dtype)
        s["x"], s["attn"] = _normal(gen, (M, H), 1.0, dtype), _normal(gen, (M, H), 1.0, dtype)
        s["bias"] = _normal(gen, (Q,), 1.0, dtype) if case["bias"] else None
    elif kind == "int8_linear":
        K, N = case["K"], case["N"]
        s["layer"] = layer = torch.nn.Module()
        scales = _uniform(gen, (N,), 0.001, 0.02, torch.float32)
        if case["scheme"] == "static":
            s["method"] = W8A8Config().get_quant_method()
            with torch.device(DEVICE):
                s["method"].create_weights(layer, K, [N], K, N, dtype)
            layer.in_scales.data.copy_(_uniform(gen, (K,), 0.02, 0.04, dtype))
            layer.out_scales.data.copy_(scales * 0.03)
        else:
            s["method"] = CompressedTensorMMLinearKernel()
            layer.weight = torch.nn.Parameter(torch.empty((N, K), dtype=torch.int8, device=DEVICE), requires_grad=False)
            layer.weight_scale = torch.nn.Parameter(scales.reshape(N, 1), requires_grad=False)
        layer.weight.data.random_(-127, 128, generator=gen)
        s["method"].process_weights_after_loading(layer)
        s["x"] = _normal(gen, (M, K), 1.0, dtype)
        s["bias"] = _normal(gen, (N,), 1.0, dtype) if case["bias"] else None
        s["scheme"] = case["scheme"]
    elif kind == "fp8_mlp":
        H, I = case["hidden"], case["inter"]
        s["method"] = m = Fp8GCUConfig((128, 128)).get_quant_method()
        s["gate_up"], s["down"] = _fp8_linear_layer(gen, m, H, 2 * I, dtype), _fp8_linear_layer(gen, m, I, H, dtype)
        s["norm"] = _uniform(gen, (H,), 0.5, 1.5, dtype)
        s["x"] = _normal(gen, (M, H), 1.0, dtype)
    elif kind == "fp8_linear":
        s["method"] = Fp8GCUConfig(None).get_quant_method()
        s["layer"] = _fp8_linear_layer(gen, s["method"], case["K"], case["N"], dtype)
        s["x"] = _normal(gen, (M, case["K"]), 1.0, dtype)
        s["bias"] = _normal(gen, (case["N"],), 1.0, dtype) if case["bias"] else None
    else:
        H, I, E = case["hidden"], case["inter"], case["experts"]
        s["layer"] = layer = torch.nn.Module()
        if kind == "moe_w4a16":
            s["method"] = m = MoeWNA16GCUConfig("gptq", 4, case["group"], True).get_quant_method()
            with torch.device(DEVICE):
                m.create_weights(layer, E, H, I, dtype)
            for name in ("w13", "w2"):
                _bits(gen, getattr(layer, name + "_qweight").data)
                _bits(gen, getattr(layer, name + "_qzeros").data)
                sc = getattr(layer, name + "_scales").data
                sc.copy_(_uniform(gen, sc.shape, 0.001, 0.01, dtype))
                rows = getattr(layer, name + "_g_idx").data
                rows.copy_((torch.arange(rows.shape[1], device=DEVICE) // case["group"]).expand_as(rows))
            s["routing"] = dict(top_k=case["topk"], renormalize=True)
            s["norm"] = _uniform(gen, (H,), 0.5, 1.5, dtype)
        else:
            s["method"] = m = Fp8GCUConfig((128, 128)).get_quant_method(moe=True)
            with torch.device(DEVICE):
                m.create_weights(layer, E, H, I, dtype)
            for name in ("w13", "w2"):
                _fp8_codes(gen, getattr(layer, name + "_weight").data)
                _block_scales(gen, getattr(layer, name + "_weight_scale_inv").data)
            s["routing"] = dict(top_k=case["topk"], renormalize=True, use_grouped_topk=True,
                                num_expert_group=case["groups"], topk_group=case["topk_group"])
            s["norm"] = _uniform(gen, (H,), 0.5, 1.5, dtype)
        m.process_weights_after_loading(layer)
        s["x"] = _normal(gen, (M, H), 1.0, dtype)
        s["logits"] = _normal(gen, (M, E), 1.0, torch.float32)
    return s


# --- one pass ----------------------------------------------------------------------------------------------
def _rms_norm(x, weight):
    out = torch.empty_like(x)
    torch.ops._C.rms_norm(out, x, weight, EPS)
    return out


def run(s):
    kind, method, x = s["kind"], s["method"], s["x"]
    if kind in ("w4a16_linear", "fp8_linear"):
        return method.apply(s["layer"], x, s["bias"])
    if kind == "w4a16_layer":
        qkv = method.apply(s["qkv"], _rms_norm(x, s["norm1"]), s["bias"])
        o = method.apply(s["o"], s["attn"])
        gate_up = method.apply(s["gate_up"], _rms_norm(o, s["norm2"]))
        act = torch.empty((x.shape[0], gate_up.shape[1] // 2), dtype=x.dtype, device=x.device)
        torch.ops._C.silu_and_mul(act, gate_up)
        return qkv, o, method.apply(s["down"], act)
    if kind == "int8_linear":
        if s["scheme"] == "static":
            return method.apply(s["layer"], x, s["bias"])
        return method.apply_weights(s["layer"], x, s["bias"])
    if kind == "fp8_mlp":
        # the norm and the gate quantise in the same pass (what the fusion pass of a compiled model puts there)
        M, H = x.shape
        q = torch.empty((M, H), dtype=torch.float8_e4m3fn, device=x.device)
        sc = torch.empty((M, H // 128), dtype=torch.float32, device=x.device)
        torch.ops._C.rms_norm_per_token_group_quant_fp8(q, sc, x, s["norm"], EPS, 128)
        gate_up = method.apply(s["gate_up"], q, None, sc)
        I = gate_up.shape[1] // 2
        a = torch.empty((M, I), dtype=torch.float8_e4m3fn, device=x.device)
        asc = torch.empty((M, I // 128), dtype=torch.float32, device=x.device)
        torch.ops._C.silu_mul_per_token_group_quant(a, asc, gate_up, 128)
        return method.apply(s["down"], a, None, asc)
    # the experts write their sum over the normed hidden states, which a model makes anew in every layer
    return method.apply(s["layer"], _rms_norm(x, s["norm"]), s["logits"], **s["routing"])


# --- what a pass cannot do without -------------------------------------------------------------------------
def _int4_bytes(K, N, group):
    return K * N // 2 + K // group * N * 2 + K // group * N // 2


def _experts_hit(case):
    """Experts that at least one token is expected to reach, by evenly spread routing."""
    return case["experts"] * (1.0 - (1.0 - case["topk"] / case["experts"]) ** case["tokens"])


def work(case):
    kind, M = case["kind"], case["tokens"]
    bias = 2 * case.get("N", case.get("qkv", 0)) if case.get("bias") else 0
    if kind == "w4a16_linear":
        K, N = case["K"], case["N"]
        return {"bytes": _int4_bytes(K, N, case["group"]) + 2 * M * (K + N) + bias, "flops": 2.0 * M * K * N}
    if kind == "w4a16_layer":
        H, Q, I, g = case["hidden"], case["qkv"], case["inter"], case["group"]
        weights = _int4_bytes(H, Q, g) + _int4_bytes(H, H, g) + _int4_bytes(H, 2 * I, g) + _int4_bytes(I, H, g)
        return {"bytes": weights + 4 * H + 2 * M * (2 * H + Q + 2 * H) + bias,
                "flops": 2.0 * M * (H * Q + H * H + 3.0 * H * I)}
    if kind == "int8_linear":
        K, N = case["K"], case["N"]
        return {"bytes": K * N + 4 * N + 2 * M * (K + N) + bias + (2 * K if case["scheme"] == "static" else 0),
                "flops": 2.0 * M * K * N}
    if kind == "fp8_mlp":
        H, I = case["hidden"], case["inter"]
        return {"bytes": 3 * H * I + 3 * H * I // 16384 * 4 + 2 * H + 4 * M * H, "flops": 6.0 * M * H * I}
    if kind == "fp8_linear":
        K, N = case["K"], case["N"]
        return {"bytes": K * N + 4 * N + 2 * M * (K + N) + bias, "flops": 2.0 * M * K * N}
    H, I, E, T = case["hidden"], case["inter"], case["experts"], case["topk"]
    if kind == "moe_w4a16":
        one = _int4_bytes(H, 2 * I, case["group"]) + _int4_bytes(I, H, case["group"])
    else:
        one = 3 * H * I + 3 * H * I // 16384 * 4
    return {"bytes": _experts_hit(case) * one + 2 * H + 4 * M * H + 4 * M * E, "flops": 6.0 * M * T * H * I}


def tolerance(case):
    kind, bf16 = case["kind"], case.get("dtype", "bf16") == "bf16"
    if kind in ("fp8_mlp", "moe_fp8"):
        # a sum that rounds the other way moves an intermediate value by an fp8 step
        return {"rel": 1e-2}
    if kind in ("w4a16_layer", "moe_w4a16"):
        return {"rel": 1e-2 if bf16 else 2e-3}              # intermediate results rounded to 16 bits
    return {"rel": 4e-3 if bf16 else 1e-3}                  # one rounding to 16 bits
