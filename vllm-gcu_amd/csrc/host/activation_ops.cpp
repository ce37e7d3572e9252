// The operators without a weight matrix, registered as boxed kernels so that a call through torch.ops ends in
// the C ABI without entering Python: csrc/torch_bindings.cpp:163-175, 254-317, 291, 714-766, 803-871, 974,
// 1052-1189, 1390-1431 of the reference.  Boxed, because the schema may belong to another extension that spells
// an optional argument as a plain Tensor: the arguments are taken off the stack by position.
#include <ATen/core/stack.h>
#include <torch/library.h>

#include <memory>
#include <vector>

#include "host.h"

namespace mi355q_host {
namespace {

using c10::IValue;
using torch::jit::Stack;

Tensor tensor_or_none(const IValue& v) { return v.isNone() ? Tensor() : v.toTensor(); }

void require_gpu(std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    TORCH_CHECK(!t->defined() || t->is_cuda(), "mi355q operators need tensors on the GPU; got a ", t->device(),
                " tensor (there is no CPU fallback)");
}

// rows and length of the last dimension
struct Rows {
  int64_t rows, len;
  explicit Rows(const Tensor& t) : len(t.size(-1)) { rows = t.numel() / len; }
};

Tensor as(const Tensor& t, at::ScalarType d) { return t.scalar_type() == d ? t.contiguous() : t.to(d).contiguous(); }

// `size` counts entries of the leading dimension (tokens); the kernels work on rows flattened over every
// dimension but the last.  The product is taken on the device, so a captured graph whose count tensor is
// rewritten between replays sees the new value.
struct Count {
  Tensor t;
  int rows_per_count = 1;
  Count() = default;
  Count(const Tensor& data, const Tensor& size) {
    if (!size.defined()) return;
    t = size.scalar_type() == at::kInt ? size : size.to(at::kInt);
    const int64_t lead = std::max<int64_t>(data.size(0), 1);
    rows_per_count = static_cast<int>(std::max<int64_t>(data.numel() / data.size(-1) / lead, 1));
  }
  const int32_t* p() const { return static_cast<const int32_t*>(ptr(t)); }
};

bool same_lead(const Tensor& out, const Tensor& x, int64_t last) {
  if (out.dim() != x.dim() || out.size(-1) != last) return false;
  for (int64_t i = 0; i + 1 < x.dim(); ++i)
    if (out.size(i) != x.size(i)) return false;
  return true;
}

void fp8_out_ok(const Tensor& out, const Tensor& x, int64_t last) {
  TORCH_CHECK((out.scalar_type() == at::kFloat8_e4m3fn || out.scalar_type() == at::kByte) && out.is_contiguous() &&
                  same_lead(out, x, last),
              "fp8 output must be a contiguous float8_e4m3fn tensor of the input's rows x ", last);
}

Tensor single_scale(const Tensor& scale, const char* what) {
  TORCH_CHECK(scale.numel() == 1, what, " takes a single scale");
  return scale.scalar_type() == at::kFloat ? scale : scale.to(at::kFloat);
}

// ---- SiLU gate ------------------------------------------------------------------------------------------
void silu_and_mul(const Tensor& out, const Tensor& input, const Tensor& size) {
  require_gpu({&out, &input, &size});
  if (input.numel() == 0) return;
  const Tensor x = input.contiguous();
  const Rows r(x);
  TORCH_CHECK(out.is_contiguous() && out.size(-1) * 2 == r.len && out.scalar_type() == x.scalar_type(),
              "silu_and_mul: out must be contiguous [..., d] of the input dtype for input [..., 2d]");
  const Count n(x, size);
  const OnDevice on(x);
  check(mi355q_silu_and_mul(out.data_ptr(), x.data_ptr(), r.rows, r.len / 2, require_dtype(x.scalar_type()), n.p(),
                            n.rows_per_count, on.stream()),
        "silu_and_mul");
}

// ---- fp8 quantisers -------------------------------------------------------------------------------------
void group_quant(const Tensor& out, const Tensor& scale, const Tensor& input, const Tensor& size, int64_t group, bool fuse) {
  require_gpu({&out, &scale, &input, &size});
  if (input.numel() == 0) return;
  const Tensor x = input.contiguous();
  const Rows r(x);
  const int64_t K = fuse ? r.len / 2 : r.len;
  fp8_out_ok(out, x, K);
  TORCH_CHECK(group > 0 && scale.scalar_type() == at::kFloat && scale.is_contiguous() && scale.numel() == r.rows * (K / group),
              "per-token-group quant: scale must be contiguous float32 [..., K / group_size]");
  const Count n(x, size);
  const OnDevice on(x);
  check(mi355q_fp8_group_quant(static_cast<uint8_t*>(out.data_ptr()), static_cast<float*>(scale.data_ptr()), x.data_ptr(),
                               r.rows, K, group, fuse, require_dtype(x.scalar_type()), n.p(), n.rows_per_count, on.stream()),
        "fp8_group_quant");
}

void token_quant(const Tensor& out, const Tensor& input, const Tensor& scale) {
  require_gpu({&out, &input, &scale});
  if (input.numel() == 0) return;
  const Tensor x = input.contiguous();
  const Rows r(x);
  fp8_out_ok(out, x, r.len);
  const OnDevice on(x);
  check(mi355q_fp8_token_quant(static_cast<uint8_t*>(out.data_ptr()), static_cast<float*>(scale.data_ptr()), x.data_ptr(),
                               r.rows, r.len, require_dtype(x.scalar_type()), nullptr, on.stream()),
        "fp8_token_quant");
}

void static_fp8(const Tensor& out, const Tensor& input, const Tensor& scale, const Tensor& size, int fuse) {
  require_gpu({&out, &input, &scale, &size});
  if (input.numel() == 0) return;
  const Tensor x = input.contiguous();
  const Rows r(x);
  const int64_t K = fuse ? r.len / 2 : r.len;
  fp8_out_ok(out, x, K);
  const Tensor sc = single_scale(scale, "static fp8 quant");
  const Count n(x, size);
  const OnDevice on(x);
  check(mi355q_fp8_static_quant(static_cast<uint8_t*>(out.data_ptr()), x.data_ptr(), static_cast<const float*>(sc.data_ptr()),
                                r.rows, K, fuse, require_dtype(x.scalar_type()), n.p(), n.rows_per_count, on.stream()),
        "fp8_static_quant");
}

// ---- int8 quantisers ------------------------------------------------------------------------------------
void dynamic_int8(const Tensor& out, const Tensor& input, const Tensor& scales, bool azp) {
  require_gpu({&out, &input, &scales});
  TORCH_CHECK(!azp, "dynamic_scaled_int8_quant: asymmetric quantisation (azp) is not supported");
  if (input.numel() == 0) return;
  const Tensor x = input.contiguous();
  const Rows r(x);
  TORCH_CHECK(out.is_contiguous() && scales.is_contiguous() && scales.scalar_type() == at::kFloat,
              "dynamic_scaled_int8_quant: output and fp32 scales must be contiguous");
  const OnDevice on(x);
  check(mi355q_dynamic_int8_quant(static_cast<int8_t*>(out.data_ptr()), static_cast<float*>(scales.data_ptr()), x.data_ptr(),
                                  r.rows, r.len, require_dtype(x.scalar_type()), nullptr, on.stream()),
        "dynamic_int8_quant");
}

void static_int8(const Tensor& out, const Tensor& input, const Tensor& scale) {
  require_gpu({&out, &input, &scale});
  if (input.numel() == 0) return;
  const Tensor x = input.contiguous();
  const Rows r(x);
  const Tensor sc = as(scale, scale.scalar_type() == x.scalar_type() ? x.scalar_type() : at::kFloat);
  TORCH_CHECK(sc.numel() == 1 || sc.numel() == r.len, "static_scaled_int8_quant: scale must have 1 or K=", r.len,
              " entries, got ", sc.numel());
  const OnDevice on(x);
  check(mi355q_static_int8_quant_typed(static_cast<int8_t*>(out.data_ptr()), x.data_ptr(), sc.data_ptr(), dtype_code(sc.scalar_type()),
                                       sc.numel() > 1, r.rows, r.len, require_dtype(x.scalar_type()), on.stream()),
        "static_int8_quant");
}

// a 0-d scale is per tensor, anything else per channel of the gated half (silu_mul_static_int8_quant.cpp:11-28)
void silu_mul_static_int8(const Tensor& out, const Tensor& input, const Tensor& scale) {
  require_gpu({&out, &input, &scale});
  if (input.numel() == 0) return;
  const Tensor x = input.contiguous();
  const Rows r(x);
  const int64_t d = r.len / 2;
  TORCH_CHECK(out.scalar_type() == at::kChar && same_lead(out, x, d) && out.is_contiguous(),
              "silu_mul_static_int8_quant: result must be contiguous int8 of the input's rows x ", d);
  const Tensor sc = as(scale, at::kFloat);
  TORCH_CHECK(sc.numel() == 1 || sc.numel() == d, "silu_mul_static_int8_quant: scale must have 1 or ", d, " entries, got ",
              sc.numel());
  const OnDevice on(x);
  check(mi355q_silu_mul_static_int8_quant(static_cast<int8_t*>(out.data_ptr()), x.data_ptr(),
                                          static_cast<const float*>(sc.data_ptr()), sc.numel() > 1, r.rows, d,
                                          require_dtype(x.scalar_type()), on.stream()),
        "silu_mul_static_int8_quant");
}

// ---- sum over the top-k slots ---------------------------------------------------------------------------
void moe_sum(const Tensor& out, const Tensor& input, const Tensor& size, int64_t dim, bool keepdim) {
  require_gpu({&out, &input, &size});
  if (input.numel() == 0) return;
  TORCH_CHECK(input.dim() == 3 && dim == 1 && !keepdim, "moe_sum_pad: expects input [M, topk, K], dim=1, keepdim=False");
  const Tensor x = input.contiguous();
  const int64_t M = x.size(0), T = x.size(1), K = x.size(2);
  TORCH_CHECK(out.is_contiguous() && out.dim() == 2 && out.size(0) == M && out.size(1) == K,
              "moe_sum_pad: out must be contiguous [M, K]");
  Tensor n;
  if (size.defined()) n = size.scalar_type() == at::kInt ? size : size.to(at::kInt);
  const OnDevice on(x);
  check(mi355q_moe_sum(out.data_ptr(), x.data_ptr(), M, T, K, require_dtype(x.scalar_type()), require_dtype(out.scalar_type()),
                       static_cast<const int32_t*>(ptr(n)), on.stream()),
        "moe_sum");
}

// ---- RMS norm and its fusions with the quantisers -------------------------------------------------------
void rms_norm(const Tensor& out, const Tensor& out_scales, const Tensor& input, const Tensor& residual, const Tensor& weight,
              const Tensor& scale, double eps, int mode, int64_t group) {
  require_gpu({&out, &out_scales, &input, &residual, &weight, &scale});
  if (input.numel() == 0) return;
  const at::ScalarType dt = input.scalar_type();
  TORCH_CHECK(is_16bit(dt), "rms_norm: input must be f16/bf16, got ", dt);
  TORCH_CHECK(input.is_contiguous() && out.is_contiguous(), "rms_norm: input and output must be contiguous");
  const Rows r(input);
  TORCH_CHECK(weight.numel() == r.len, "rms_norm: weight has ", weight.numel(), " elements for rows of ", r.len);
  TORCH_CHECK(out.sizes() == input.sizes(), "rms_norm: output shape ", out.sizes(), " != input shape ", input.sizes());
  const at::ScalarType want = mode == 0 ? dt : mode == 3 ? at::kChar : at::kFloat8_e4m3fn;
  TORCH_CHECK(out.scalar_type() == want, "rms_norm: output must be ", want, ", got ", out.scalar_type());
  TORCH_CHECK(!residual.defined() ||
                  (residual.scalar_type() == dt && residual.sizes() == input.sizes() && residual.is_contiguous()),
              "rms_norm: residual must match the input (dtype, shape, contiguous)");
  const Tensor w = as(weight, dt);
  Tensor sc;
  if (mode == 1 || mode == 3) sc = single_scale(scale, "rms_norm + static quant");
  TORCH_CHECK(mode != 2 || (group > 0 && out_scales.scalar_type() == at::kFloat && out_scales.is_contiguous() &&
                            out_scales.numel() == r.rows * (r.len / group)),
              "rms_norm + group quant: scales must be contiguous f32 [.., K / group_size]");
  const OnDevice on(input);
  check(mi355q_rms_norm(out.data_ptr(), static_cast<float*>(ptr(out_scales)), input.data_ptr(), ptr(residual), w.data_ptr(),
                        static_cast<const float*>(ptr(sc)), static_cast<float>(eps), r.rows, r.len, mode, group,
                        dtype_code(dt), on.stream()),
        "rms_norm");
}

// ---- routing --------------------------------------------------------------------------------------------
void topk_softmax(const Tensor& weights, const Tensor& ids, const Tensor& token_expert, const Tensor& gating) {
  require_gpu({&weights, &ids, &token_expert, &gating});
  if (gating.numel() == 0) return;
  const Tensor g = gating.contiguous();
  TORCH_CHECK(g.dim() == 2, "topk_softmax: gating_output must be [M, E]");
  TORCH_CHECK(weights.scalar_type() == at::kFloat && ids.scalar_type() == at::kInt,
              "topk_softmax: topk_weights must be float32 and topk_indices int32");
  TORCH_CHECK(weights.is_contiguous() && ids.is_contiguous(), "topk_softmax: outputs must be contiguous");
  TORCH_CHECK(!token_expert.defined() || (token_expert.scalar_type() == at::kInt && token_expert.is_contiguous()),
              "topk_softmax: token_expert_indices must be contiguous int32");
  const OnDevice on(g);
  check(mi355q_topk_softmax(static_cast<float*>(weights.data_ptr()), static_cast<int32_t*>(ids.data_ptr()),
                            static_cast<int32_t*>(ptr(token_expert)), g.data_ptr(), g.size(0), g.size(1), weights.size(-1), 0,
                            require_dtype(g.scalar_type()), on.stream()),
        "topk_softmax");
}

void grouped_topk(const Tensor& weights, const Tensor& ids, const Tensor& gating, int64_t topk, bool renormalize, int64_t groups,
                  int64_t topk_group, const Tensor& bias, c10::string_view scoring) {
  require_gpu({&weights, &ids, &gating, &bias});
  if (gating.numel() == 0) return;
  TORCH_CHECK(scoring == "softmax" || scoring == "sigmoid", "fused_grouped_topk: unsupported scoring function '", scoring, "'");
  const Tensor g = gating.contiguous();
  TORCH_CHECK(g.dim() == 2, "fused_grouped_topk: gating_output must be [M, E]");
  Tensor b;
  if (bias.defined()) b = as(bias, at::kFloat);
  TORCH_CHECK(weights.scalar_type() == at::kFloat && ids.scalar_type() == at::kInt,
              "fused_grouped_topk: topk_weights must be float32 and topk_ids int32");
  const OnDevice on(g);
  check(mi355q_grouped_topk(static_cast<float*>(weights.data_ptr()), static_cast<int32_t*>(ids.data_ptr()), g.data_ptr(),
                            static_cast<const float*>(ptr(b)), g.size(0), g.size(1), topk, renormalize, groups, topk_group,
                            scoring == "sigmoid", require_dtype(g.scalar_type()), on.stream()),
        "grouped_topk");
}

void align(const Tensor& topk_ids, const Tensor& valid, int64_t experts, int64_t block, const Tensor& map, const Tensor& sorted,
           const Tensor& expert_ids, const Tensor& post_pad) {
  require_gpu({&topk_ids, &valid, &map, &sorted, &expert_ids, &post_pad});
  const Tensor ids = topk_ids.contiguous();
  TORCH_CHECK(ids.scalar_type() == at::kInt || ids.scalar_type() == at::kLong,
              "moe_align_block_size: topk_ids must be int32 or int64, got ", ids.scalar_type());
  const int64_t numel = ids.numel(), top = ids.dim() > 1 ? ids.size(-1) : 1;
  const int64_t cap = numel + experts * (block - 1);
  TORCH_CHECK(sorted.numel() >= cap && expert_ids.numel() >= cap / block,
              "moe_align_block_size: output buffers are smaller than numel + num_experts * (block_size - 1)");
  for (const Tensor* t : {&sorted, &expert_ids, &post_pad})
    TORCH_CHECK(t->scalar_type() == at::kInt && t->is_contiguous(), "moe_align_block_size: outputs must be contiguous int32");
  Tensor v, m;
  if (valid.defined()) v = valid.scalar_type() == at::kInt ? valid : valid.to(at::kInt);
  if (map.defined()) m = as(map, at::kInt);
  const OnDevice on(ids);
  check(mi355q_moe_align_block_size(ids.data_ptr(), ids.scalar_type() == at::kLong, numel, top,
                                    static_cast<const int32_t*>(ptr(v)), experts, block, static_cast<const int32_t*>(ptr(m)),
                                    static_cast<int32_t*>(sorted.data_ptr()), static_cast<int32_t*>(expert_ids.data_ptr()),
                                    static_cast<int32_t*>(post_pad.data_ptr()), on.stream()),
        "moe_align_block_size");
}

// ---- boxed kernels: N arguments off the stack, nothing returned ------------------------------------------
struct Args {
  Stack* s;
  size_t n;
  const IValue& operator[](size_t i) const { return torch::jit::peek(*s, i, n); }
  Tensor t(size_t i) const { return tensor_or_none((*this)[i]); }
  int64_t i(size_t i) const { return (*this)[i].toInt(); }
  double d(size_t i) const { return (*this)[i].toDouble(); }
  bool b(size_t i) const { return (*this)[i].toBool(); }
  c10::string_view str(size_t i) const { return (*this)[i].toStringView(); }
};


template <size_t N, void (*F)(const Args&)>
void boxed(const c10::OperatorHandle&, Stack* stack) {
  F(Args{stack, N});
  torch::jit::drop(*stack, N);
}

const Tensor none;

#define MQ_OP(NAME, N, ...) \
  void NAME(const Args& a) { __VA_ARGS__; }

MQ_OP(op_silu_and_mul, 2, silu_and_mul(a.t(0), a.t(1), none))
MQ_OP(op_silu_and_mul_pad, 3, silu_and_mul(a.t(0), a.t(1), a.t(2)))
MQ_OP(op_group_quant, 4, group_quant(a.t(0), a.t(1), a.t(2), none, a.i(3), false))
MQ_OP(op_group_quant_size, 5, group_quant(a.t(0), a.t(1), a.t(2), a.t(3), a.i(4), false))
MQ_OP(op_silu_group_quant, 4, group_quant(a.t(0), a.t(1), a.t(2), none, a.i(3), true))
MQ_OP(op_silu_group_quant_size, 5, group_quant(a.t(0), a.t(1), a.t(2), a.t(3), a.i(4), true))
// (scale_ub is ignored, as in the reference: dynamic_per_token_scaled_fp8_quant.cpp:32-34)
MQ_OP(op_token_quant, 4, token_quant(a.t(0), a.t(1), a.t(2)))
MQ_OP(op_static_fp8, 3, static_fp8(a.t(0), a.t(1), a.t(2), none, 0))
MQ_OP(op_silu_static_fp8, 4, static_fp8(a.t(0), a.t(1), a.t(2), a.t(3), 1))
MQ_OP(op_mul_static_fp8, 4, static_fp8(a.t(0), a.t(1), a.t(2), a.t(3), 2))
MQ_OP(op_dynamic_int8, 4, dynamic_int8(a.t(0), a.t(1), a.t(2), a.t(3).defined()))
MQ_OP(op_static_int8, 4, static_int8(a.t(0), a.t(1), a.t(2)))
MQ_OP(op_silu_static_int8, 3, silu_mul_static_int8(a.t(0), a.t(1), a.t(2)))
MQ_OP(op_moe_sum, 5, moe_sum(a.t(0), a.t(1), a.t(2), a.i(3), a.b(4)))
MQ_OP(op_rms_norm, 4, rms_norm(a.t(0), none, a.t(1), none, a.t(2), none, a.d(3), 0, 0))
MQ_OP(op_add_rms_norm, 4, rms_norm(a.t(0), none, a.t(0), a.t(1), a.t(2), none, a.d(3), 0, 0))
MQ_OP(op_rms_norm_fp8, 5, rms_norm(a.t(0), none, a.t(1), none, a.t(2), a.t(3), a.d(4), 1, 0))
MQ_OP(op_add_rms_norm_fp8, 6, rms_norm(a.t(0), none, a.t(1), a.t(2), a.t(3), a.t(4), a.d(5), 1, 0))
MQ_OP(op_rms_norm_group, 6, rms_norm(a.t(0), a.t(1), a.t(2), none, a.t(3), none, a.d(4), 2, a.i(5)))
MQ_OP(op_add_rms_norm_group, 7, rms_norm(a.t(0), a.t(2), a.t(3), a.t(1), a.t(4), none, a.d(5), 2, a.i(6)))
MQ_OP(op_rms_norm_int8, 5, rms_norm(a.t(0), none, a.t(1), none, a.t(2), a.t(3), a.d(4), 3, 0))
MQ_OP(op_add_rms_norm_int8, 6, rms_norm(a.t(0), none, a.t(1), a.t(2), a.t(3), a.t(5), a.d(4), 3, 0))
MQ_OP(op_topk_softmax, 4, topk_softmax(a.t(0), a.t(1), a.t(2), a.t(3)))
MQ_OP(op_grouped_topk, 9, grouped_topk(a.t(0), a.t(1), a.t(2), a.i(3), a.b(4), a.i(5), a.i(6), a.t(7), a.str(8)))
MQ_OP(op_align, 6, align(a.t(0), none, a.i(1), a.i(2), none, a.t(3), a.t(4), a.t(5)))
MQ_OP(op_align_pad, 7, align(a.t(0), a.t(1), a.i(2), a.i(3), none, a.t(4), a.t(5), a.t(6)))
MQ_OP(op_align_exts, 8, align(a.t(3), a.t(4), a.i(6), a.i(7), a.t(5), a.t(0), a.t(1), a.t(2)))
#undef MQ_OP

}  // namespace

void register_activation_ops() {
  // kept for the life of the process: a Library object takes its registrations back when it ends
  static torch::Library& c = *new torch::Library(torch::Library::IMPL, "_C", c10::DispatchKey::CUDA, __FILE__, __LINE__);
  static torch::Library& moe = *new torch::Library(torch::Library::IMPL, "_moe_C", c10::DispatchKey::CUDA, __FILE__, __LINE__);
#define MQ_IMPL(LIB, OP, N, F) LIB.impl(OP, torch::CppFunction::makeFromBoxedFunction<&boxed<N, &F>>())
  MQ_IMPL(c, "silu_and_mul", 2, op_silu_and_mul);
  MQ_IMPL(c, "silu_and_mul_pad", 3, op_silu_and_mul_pad);
  MQ_IMPL(c, "dynamic_per_token_group_fp8_quant", 4, op_group_quant);
  MQ_IMPL(c, "dynamic_per_token_group_fp8_quant_with_size", 5, op_group_quant_size);
  MQ_IMPL(c, "silu_mul_per_token_group_quant", 4, op_silu_group_quant);
  MQ_IMPL(c, "silu_mul_per_token_group_quant_with_size", 5, op_silu_group_quant_size);
  MQ_IMPL(c, "dynamic_per_token_scaled_fp8_quant", 4, op_token_quant);
  MQ_IMPL(c, "static_scaled_fp8_quant", 3, op_static_fp8);
  MQ_IMPL(c, "silu_mul_static_fp8_quant", 4, op_silu_static_fp8);
  MQ_IMPL(c, "mul_static_fp8_quant", 4, op_mul_static_fp8);
  MQ_IMPL(c, "dynamic_scaled_int8_quant", 4, op_dynamic_int8);
  MQ_IMPL(c, "static_scaled_int8_quant", 4, op_static_int8);
  MQ_IMPL(c, "silu_mul_static_int8_quant", 3, op_silu_static_int8);
  MQ_IMPL(moe, "moe_sum_pad", 5, op_moe_sum);
  MQ_IMPL(c, "rms_norm", 4, op_rms_norm);
  MQ_IMPL(c, "fused_add_rms_norm", 4, op_add_rms_norm);
  MQ_IMPL(c, "rms_norm_static_fp8_quant", 5, op_rms_norm_fp8);
  MQ_IMPL(c, "fused_add_rms_norm_static_fp8_quant", 6, op_add_rms_norm_fp8);
  MQ_IMPL(c, "rms_norm_per_token_group_quant_fp8", 6, op_rms_norm_group);
  MQ_IMPL(c, "fused_add_rms_norm_per_token_group_quant_fp8", 7, op_add_rms_norm_group);
  MQ_IMPL(c, "rms_norm_static_int8_quant", 5, op_rms_norm_int8);
  MQ_IMPL(c, "fused_add_rms_norm_static_int8_quant", 6, op_add_rms_norm_int8);
  MQ_IMPL(moe, "topk_softmax", 4, op_topk_softmax);
  MQ_IMPL(c, "fused_grouped_topk", 9, op_grouped_topk);
  MQ_IMPL(moe, "moe_align_block_size", 6, op_align);
  MQ_IMPL(moe, "sgl_moe_align_block_size", 6, op_align);
  MQ_IMPL(c, "moe_align_block_size_pad", 7, op_align_pad);
  MQ_IMPL(c, "exts_moe_align_block_size", 8, op_align_exts);
#undef MQ_IMPL
}

}  // namespace mi355q_host
