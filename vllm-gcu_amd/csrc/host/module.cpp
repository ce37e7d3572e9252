// vllm_gcu_amd._mi355q_host: the calls a model's forward makes, from torch tensors to the C ABI in one step.
//
// Every function here is a fast path: it takes operands that the kernels can read as they are (GPU tensors,
// contiguous, weights in this library's layouts, matching types and sizes), allocates the outputs and launches.
// Anything else -- a conversion, a reference-layout weight, a tensor subclass or a mode that must see the
// operator (torch.jit tracing, __torch_function__ and __torch_dispatch__ in classes and modes, functionalisation,
// functorch's transforms, gradients), a wrong size -- makes it return None before any work is enqueued, and the
// Python caller goes on with its general path, which calls the operator, converts or raises.
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/PyInterpreter.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "host.h"

namespace mi355q_host {
namespace {

// launches may wait for room in the queue: other Python threads run meanwhile
struct NoGil {
  PyThreadState* s = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(s); }
};

struct Bytes {                     // a name looked up often
  PyObject* o;
  explicit Bytes(const char* s) : o(PyUnicode_InternFromString(s)) {}
};

// ---- which tensors a fast path takes ---------------------------------------------------------------------
constexpr c10::DispatchKeySet kSpecial({
    c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::Functionalize,
    c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched,
    c10::DispatchKey::Conjugate, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});

// what a thread turns on to see every operator: tracing records it, functorch runs it level by level
constexpr c10::DispatchKeySet kWatching = kSpecial | c10::DispatchKeySet({
    c10::DispatchKey::Tracer, c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
    c10::DispatchKey::FuncTorchDynamicLayerBackMode});

// looked up when the module is loaded: the __torch_function__ of classes that leave torch's functions alone (parameters among
// them), and the type of the mode behind torch.device(..) contexts and torch.set_default_device, which acts on the functions that
// make tensors only
PyObject* g_disabled_torch_function = nullptr;
PyObject* g_device_context = nullptr;

bool function_mode_active() {
  using TLS = at::impl::PythonTorchFunctionTLS;
  if (!at::impl::torch_function_mode_enabled()) return false;
  for (int64_t i = 0; i < TLS::stack_len(); ++i)
    if (reinterpret_cast<PyObject*>(Py_TYPE(TLS::get_stack_at(i)->ptr(getPyInterpreter()))) != g_device_context) return true;
  return false;
}

bool modes_active() {
  const auto inc = c10::impl::tls_local_dispatch_key_set().included_;
  return inc.has_any(kWatching) || c10::impl::TorchDispatchModeTLS::any_modes_set() || function_mode_active();
}

// a tensor of a class whose __torch_function__ has to see the call
bool overrides_torch_function(PyObject* o) {
  static const Bytes name("__torch_function__");
  if (THPVariable_CheckExact(o)) return false;
  PyObject* f = PyObject_GetAttr(reinterpret_cast<PyObject*>(Py_TYPE(o)), name.o);
  if (!f) PyErr_Clear();
  Py_XDECREF(f);                   // (the class holds it)
  return f != g_disabled_torch_function;
}

bool plain(const Tensor& t) {
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(kSpecial) &&
         !(t.requires_grad() && at::GradMode::is_enabled());
}

const Tensor* as_tensor(PyObject* o) {
  if (!o || !THPVariable_Check(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  return plain(t) && !overrides_torch_function(o) ? &t : nullptr;
}

// None or no object -> an undefined tensor; false for anything a fast path does not take
bool optional_tensor(PyObject* o, Tensor& t) {
  if (!o || o == Py_None) return true;
  const Tensor* p = as_tensor(o);
  if (!p) return false;
  t = *p;
  return true;
}

bool dense(const Tensor& t, at::ScalarType d) { return t.scalar_type() == d && t.is_contiguous(); }
bool dense(const Tensor& t, at::ScalarType d, int64_t numel) { return dense(t, d) && t.numel() == numel; }
bool none_or_dense(const Tensor& t, at::ScalarType d, int64_t numel) { return !t.defined() || dense(t, d, numel); }

// an attribute of a layer the way nn.Module looks it up, without the exception its own look-up goes through;
// a new reference, null (and no error set) where there is none
PyObject* layer_attr(PyObject* layer, const Bytes& name) {
  static const Bytes params("_parameters");
  PyObject** dict = _PyObject_GetDictPtr(layer);
  if (dict && *dict) {
    PyObject* v = PyDict_GetItem(*dict, name.o);
    if (!v) {
      PyObject* p = PyDict_GetItem(*dict, params.o);
      if (p && PyDict_Check(p)) v = PyDict_GetItem(p, name.o);
    }
    if (v) {
      Py_INCREF(v);
      return v;
    }
  }
  PyObject* v = PyObject_GetAttr(layer, name.o);
  if (!v) PyErr_Clear();
  return v;
}

struct Ref {                       // owns one reference
  PyObject* o;
  explicit Ref(PyObject* p) : o(p) {}
  Ref(const Ref&) = delete;
  ~Ref() { Py_XDECREF(o); }
};

PyObject* no() { Py_RETURN_NONE; }

c10::SmallVector<int64_t, 5> with_last(const Tensor& x, int64_t last) {
  c10::SmallVector<int64_t, 5> s(x.sizes().begin(), x.sizes().end());
  s.back() = last;
  return s;
}

// ---- kslab registry ----------------------------------------------------------------------------------------
struct Alloc {
  int64_t bytes;
  int64_t live;                    // tensor objects that carry the flag
};
std::mutex g_kslab_mu;
std::unordered_map<uintptr_t, Alloc>& kslab_map(int64_t dev) {
  static auto& m = *new std::unordered_map<int64_t, std::unordered_map<uintptr_t, Alloc>>;
  return m[dev];
}

PyObject* py_kslab_register(PyObject*, PyObject* const* a, Py_ssize_t) {
  const int64_t dev = PyLong_AsLongLong(a[0]), bytes = PyLong_AsLongLong(a[2]);
  const uintptr_t p = PyLong_AsUnsignedLongLong(a[1]);
  std::lock_guard<std::mutex> lk(g_kslab_mu);
  Alloc& e = kslab_map(dev)[p];
  e.bytes = bytes;
  ++e.live;
  return no();
}

PyObject* py_kslab_unregister(PyObject*, PyObject* const* a, Py_ssize_t) {
  const int64_t dev = PyLong_AsLongLong(a[0]);
  const uintptr_t p = PyLong_AsUnsignedLongLong(a[1]);
  std::lock_guard<std::mutex> lk(g_kslab_mu);
  auto& m = kslab_map(dev);
  auto it = m.find(p);
  if (it != m.end() && --it->second.live <= 0) m.erase(it);
  return no();
}

PyObject* py_is_kslab(PyObject*, PyObject* const* a, Py_ssize_t) {
  if (!THPVariable_Check(a[0])) Py_RETURN_FALSE;
  const Tensor& t = THPVariable_Unpack(a[0]);
  if (t.is_cuda() && !t.key_set().has_any(kSpecial) && is_kslab(t)) Py_RETURN_TRUE;
  Py_RETURN_FALSE;
}

// ---- W4A16 -------------------------------------------------------------------------------------------------
struct W4 {
  Tensor qweight, zeros, scales;
};

// x[.., K] @ dequant(qweight) (+ bias), or an undefined tensor where the operands are not what the kernels read
Tensor w4a16(const Tensor& x, const W4& w, const Tensor& bias, int64_t group) {
  const at::ScalarType dt = x.scalar_type();
  const Tensor& qw = w.qweight;
  if (!is_16bit(dt) || x.dim() < 1 || !x.is_contiguous() || x.numel() == 0) return {};
  if (qw.dim() != 2 || !dense(qw, at::kInt)) return {};
  const int64_t K = x.size(-1), N = qw.size(1), M = x.numel() / K;
  const int64_t groups = group > 0 ? K / group : 1;
  if (qw.size(0) * 8 != K || !dense(w.scales, dt, groups * N) || !none_or_dense(bias, dt, N)) return {};
  const bool zp = w.zeros.defined() && w.zeros.numel() != 0;
  if (zp && !dense(w.zeros, at::kInt, groups * N / 8)) return {};
  const OnDevice on(x);
  void* stream = on.stream();
  const Scratch ws = workspace(x, stream, mi355q_w4a16_workspace_bytes(M, K, N));
  const NoGil free_gil;
  Tensor out = empty(with_last(x, N), dt, x);
  check(mi355q_w4a16_gemm(out.data_ptr(), x.data_ptr(), static_cast<const int32_t*>(qw.data_ptr()), w.scales.data_ptr(),
                          zp ? w.zeros.data_ptr() : nullptr, zp ? MI355Q_ZP_PACKED : MI355Q_ZP_NONE, ptr(bias), M, K, N,
                          group, dtype_code(dt), ws.p, ws.bytes, stream),
        "w4a16_gemm");
  return out;
}

// a g_idx that the general path has verified (it leaves its tag on the tensor), or none at all
bool g_idx_ok(PyObject* g, int64_t group) {
  static const Bytes tag("_mi355q_trivial");
  if (!g || g == Py_None) return true;
  if (!THPVariable_Check(g)) return false;
  const Tensor& t = THPVariable_Unpack(g);
  if (t.key_set().has_any(kSpecial) || overrides_torch_function(g)) return false;
  if (t.numel() == 0) return true;
  PyObject** dict = _PyObject_GetDictPtr(g);
  PyObject* v = dict && *dict ? PyDict_GetItem(*dict, tag.o) : nullptr;
  return v && PyTuple_Check(v) && PyTuple_GET_SIZE(v) == 3 &&
         PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(v, 0)) == reinterpret_cast<uintptr_t>(t.data_ptr()) &&
         PyLong_AsLongLong(PyTuple_GET_ITEM(v, 1)) == static_cast<int64_t>(t._version()) &&
         PyLong_AsLongLong(PyTuple_GET_ITEM(v, 2)) == group;
}

PyObject* w4a16_objects(PyObject* x, PyObject* qw, PyObject* zeros, PyObject* scales, PyObject* g_idx, PyObject* bias,
                        int64_t group) {
  const Tensor *xt = as_tensor(x), *qt = as_tensor(qw), *st = as_tensor(scales);
  Tensor zt, bt;
  if (!xt || !qt || !st || !optional_tensor(zeros, zt) || !optional_tensor(bias, bt) || !g_idx_ok(g_idx, group) || modes_active())
    return no();
  Tensor out = w4a16(*xt, W4{*qt, zt, *st}, bt, group);
  if (!out.defined()) return no();
  return THPVariable_Wrap(std::move(out));
}

// (x, qweight, zeros, scales, g_idx, bias, group_size)
PyObject* py_w4a16(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  return w4a16_objects(a[0], a[1], a[2], a[3], a[4], a[5], PyLong_AsLongLong(a[6]));
  END_HANDLE_TH_ERRORS
}

// (layer, x, bias, group_size): the operands from the layer's qweight / qzeros / scales / g_idx
PyObject* py_w4a16_layer(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  static const Bytes n_qw("qweight"), n_qz("qzeros"), n_sc("scales"), n_gi("g_idx");
  const Ref qw(layer_attr(a[0], n_qw)), qz(layer_attr(a[0], n_qz)), sc(layer_attr(a[0], n_sc)), gi(layer_attr(a[0], n_gi));
  if (!qw.o || !sc.o) return no();
  return w4a16_objects(a[1], qw.o, qz.o, sc.o, gi.o, a[2], PyLong_AsLongLong(a[3]));
  END_HANDLE_TH_ERRORS
}

// ---- W8A8 int8 ---------------------------------------------------------------------------------------------
// Up to how many rows the weight-streaming kernel takes a kslab layer (measured on MI355X, us, streaming / MFMA
// tile kernel; `top` = 64 is its last single pass).  The streaming kernel gives a layer of few columns 32 or 16
// columns per workgroup, so every CU streams a share; the tile kernel's wavefronts without rows only copy, and on
// layers of at most 128 column tiles it cuts K into ranges that fill the chip.  The streaming kernel's time grows
// with the rows (in steps at 17, 33), the split tile kernel's hardly does: they cross at 25..32 rows behind a very
// long K -- 28672 x 8192: M = 24 45.4 / 50.5, M = 32 51.5 / 50.7, M = 64 67.1 / 49.7; at 33..40 where K >= 2 N --
// 16384 x 7168: M = 32 26.2 / 29.6, M = 40 31.0 / 30.3; 14336 x 4096: M = 32 19.5 / 20.1, M = 40 24.4 / 20.2; at
// 41..48 for other K >= 7168 -- 7168 x 4096: M = 40 14.9 / 15.9, M = 48 16.2 / 16.1; 8192 x 8192: M = 48 19.5 / 21.3,
// M = 64 23.0 / 22.0; on wide layers (128 column tiles or more, no split) -- 8192 x 28672: M = 40 49.8 / 52.3,
// M = 48 51.9 / 49.1; a short K stays with the streaming kernel -- 4096 x 4096: M = 64 13.4 / 15.6.
int64_t int8_stream_rows(int64_t K, int64_t N, int64_t top) {
  if (N % 128 != 0) return top;
  if (N >= 128 * 128) return top * 5 / 8;
  if (K >= 24576) return top * 3 / 8;
  if (K >= 2 * N && K >= 7168) return top / 2;
  if (K >= 7168) return top * 5 / 8;
  return top;
}

PyObject* py_int8_stream_rows(PyObject*, PyObject* const* a, Py_ssize_t) {
  return PyLong_FromLongLong(int8_stream_rows(PyLong_AsLongLong(a[0]), PyLong_AsLongLong(a[1]), PyLong_AsLongLong(a[2])));
}

struct Int8Mm {
  Tensor w, ws, bias;              // kslab weight of N x K, f32 scales [N], bias in the output type
  int64_t N, K;
  at::ScalarType out_dtype;
  bool ok() const {
    return w.scalar_type() == at::kChar && is_kslab(w) && K % 128 == 0 && N % 64 == 0 && N > 1 && dense(ws, at::kFloat, N) &&
           is_16bit(out_dtype) && none_or_dense(bias, out_dtype, N);
  }
};

// q [M, K] int8 with one f32 scale per row (or none): GIL held on entry, `ws` is the stream's scratch
void int8_mm(const Int8Mm& m, const Tensor& q, const Tensor& xs, const Tensor& out, int64_t M, int64_t top, bool mid,
             const Scratch& ws, void* stream) {
  const float* xp = static_cast<const float*>(ptr(xs));
  const float* wp = static_cast<const float*>(m.ws.data_ptr());
  // decode-sized M: the weight-streaming kernel (same int32 sums, same epilogue order: bit-identical results)
  // reads kslab weights about twice as fast as the tile kernel
  if (!mid && M <= int8_stream_rows(m.K, m.N, top)) {
    check(mi355q_kcontig_gemm(out.data_ptr(), q.data_ptr(), m.w.data_ptr(), xp, wp, ptr(m.bias), 2, 0, M, m.K, m.N, MI355Q_F16,
                              dtype_code(m.out_dtype), 1, stream),
          "kcontig_gemm");
    return;
  }
  check(mi355q_w8a8_int8_gemm_ws(out.data_ptr(), nullptr, static_cast<const int8_t*>(q.data_ptr()),
                                 static_cast<const int8_t*>(m.w.data_ptr()), xp, xp && xs.numel() > 1, wp, 1, ptr(m.bias), 0, M,
                                 m.N, m.K, m.K, 0, m.N, dtype_code(m.out_dtype) | MI355Q_ZEROED_COUNTERS, ws.p, ws.bytes, stream),
        "w8a8_int8_gemm");
}

// bytes of scratch; mid: the kernel for some hundred rows takes the layer
size_t int8_scratch(const Int8Mm& m, int64_t M, int64_t top, bool& mid) {
  size_t need = 0;
  mid = mi355q_q8_mid_plan(2, M, m.N, m.K, &need);
  if (mid) return need;
  return M <= int8_stream_rows(m.K, m.N, top) ? 0 : mi355q_w8a8_int8_workspace_bytes(M, m.N, m.K);
}

// Whether a call of a few rows goes to the kernel that quantises them itself (kind and quantiser of mi355q_q8_quant_gemm)
bool quantises(int kind, int quant, int64_t M, int64_t N, int64_t K, const Tensor& x, const Tensor& c_scale, const Tensor& w, const Tensor& ws,
               const Tensor& bias) {
  const auto off = [](const Tensor& t, uintptr_t a) { return reinterpret_cast<uintptr_t>(ptr(t)) % a != 0; };
  return M <= 16 && mi355q_q8_quant_gemm_takes(kind, quant, M, N, K) && !off(x, 16) && !off(c_scale, 16) && !off(w, 16) && !off(ws, 16) && !off(bias, 8);
}

// (layer, x, bias, top): quantise with the layer's per-channel in_scales, multiply with out_scales
PyObject* py_w8a8_static_layer(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  static const Bytes n_w("weight"), n_in("in_scales"), n_os("out_scales"), n_dt("out_dtype");
  const Ref w(layer_attr(a[0], n_w)), in(layer_attr(a[0], n_in)), os(layer_attr(a[0], n_os)), od(layer_attr(a[0], n_dt));
  const Tensor *xt = as_tensor(a[1]), *wt = as_tensor(w.o), *it = as_tensor(in.o), *st = as_tensor(os.o);
  const int64_t top = PyLong_AsLongLong(a[3]);
  Int8Mm m;
  if (!xt || !wt || !it || !st || !od.o || !THPDtype_Check(od.o) || !optional_tensor(a[2], m.bias) || modes_active()) return no();
  m.w = *wt, m.ws = *st, m.out_dtype = reinterpret_cast<THPDtype*>(od.o)->scalar_type;
  const Tensor& x = *xt;
  if (wt->dim() != 2 || x.dim() < 1 || x.numel() == 0 || !x.is_contiguous() || !is_16bit(x.scalar_type())) return no();
  m.N = wt->size(0), m.K = wt->size(1);
  if (x.size(-1) != m.K || !m.ok() || !dense(*it, x.scalar_type(), m.K)) return no();
  const int64_t M = x.numel() / m.K;
  const OnDevice on(x);
  void* stream = on.stream();
  Tensor out;
  if (m.out_dtype == x.scalar_type() && quantises(2, 2, M, m.N, m.K, x, *it, m.w, m.ws, m.bias)) {
    const NoGil free_gil;
    out = empty(with_last(x, m.N), m.out_dtype, x);
    check(mi355q_q8_quant_gemm(out.data_ptr(), x.data_ptr(), m.w.data_ptr(), it->data_ptr(), static_cast<const float*>(m.ws.data_ptr()), 1,
                               ptr(m.bias), 2, 2, M, m.N, m.K, dtype_code(m.out_dtype), stream),
          "q8_quant_gemm");
  } else {
    bool mid;
    const size_t need = int8_scratch(m, M, top, mid);
    const Scratch ws = need ? workspace(x, stream, need) : Scratch{nullptr, 0};
    const NoGil free_gil;
    const Tensor q = empty({M, m.K}, at::kChar, x);
    out = empty(with_last(x, m.N), m.out_dtype, x);
    check(mi355q_static_int8_quant_typed(static_cast<int8_t*>(q.data_ptr()), x.data_ptr(), it->data_ptr(), dtype_code(x.scalar_type()),
                                         1, M, m.K, dtype_code(x.scalar_type()), stream),
          "static_int8_quant");
    int8_mm(m, q, Tensor(), out, M, top, mid, ws, stream);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// (layer, x, bias, top): dynamic per-token activation scales, weight_scale per channel
PyObject* py_int8_dynamic_layer(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  static const Bytes n_w("weight"), n_ws("weight_scale"), n_is("input_scale");
  const Ref w(layer_attr(a[0], n_w)), sc(layer_attr(a[0], n_ws)), is(layer_attr(a[0], n_is));
  const Tensor *xt = as_tensor(a[1]), *wt = as_tensor(w.o), *st = as_tensor(sc.o);
  const int64_t top = PyLong_AsLongLong(a[3]);
  Int8Mm m;
  if (!xt || !wt || !st || (is.o && is.o != Py_None) || !optional_tensor(a[2], m.bias) || modes_active()) return no();
  const Tensor& x = *xt;
  if (wt->dim() != 2 || x.dim() < 1 || x.numel() == 0 || !x.is_contiguous() || !is_16bit(x.scalar_type())) return no();
  m.w = *wt, m.ws = *st, m.out_dtype = x.scalar_type(), m.N = wt->size(0), m.K = wt->size(1);
  if (x.size(-1) != m.K || !m.ok()) return no();
  const int64_t M = x.numel() / m.K;
  const OnDevice on(x);
  void* stream = on.stream();
  Tensor out;
  if (quantises(2, 1, M, m.N, m.K, x, Tensor(), m.w, m.ws, m.bias)) {
    const NoGil free_gil;
    out = empty(with_last(x, m.N), m.out_dtype, x);
    check(mi355q_q8_quant_gemm(out.data_ptr(), x.data_ptr(), m.w.data_ptr(), nullptr, static_cast<const float*>(m.ws.data_ptr()), 1, ptr(m.bias),
                               2, 1, M, m.N, m.K, dtype_code(m.out_dtype), stream),
          "q8_quant_gemm");
  } else {
    bool mid;
    const size_t need = int8_scratch(m, M, top, mid);
    const Scratch ws = need ? workspace(x, stream, need) : Scratch{nullptr, 0};
    const NoGil free_gil;
    const Tensor q = empty({M, m.K}, at::kChar, x), xs = empty({M}, at::kFloat, x);
    out = empty(with_last(x, m.N), m.out_dtype, x);
    check(mi355q_dynamic_int8_quant(static_cast<int8_t*>(q.data_ptr()), static_cast<float*>(xs.data_ptr()), x.data_ptr(), M, m.K,
                                    dtype_code(x.scalar_type()), nullptr, stream),
          "dynamic_int8_quant");
    int8_mm(m, q, xs, out, M, top, mid, ws, stream);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ---- fp8 ---------------------------------------------------------------------------------------------------
// Which kernel a block-scaled layer takes: -1 = the weight streamer, else the MFMA tile kernel with that many
// bytes of scratch for its K ranges.  The tile kernel beats the streamer above 64 rows once its tiles fill a
// good part of the chip (measured, K 8192 N 28672 = 224 tiles: M 65..128 69..73 us against 87..119 us, M 64 68 us
// against 73 us for the streamer's last single-block size; K 7168 N 4096 = 32 tiles: 52 us against 37..53 us at
// M 65..128, so few tiles stay with the streamer).  The tile kernel needs about 1 us per K block however few tiles
// there are; the streamer's time grows with the rows: they cross at 48..64 tiles (K 7168 N 4096: 32 tiles 56
// against 31 us, 64 tiles 55 against 58 us, 96 tiles 56 against 85 us; the same on K 4096 N 4096, K 2048 N 7168 and
// K 7168 N 2048).  From 33 rows on a layer of 128 tiles or more: the tile kernel's wavefronts without rows only
// copy (K 8192 x N 28672 at M = 40 / 48 / 64: 59.0 / 62.3 / 68.7 -> 55.5 / 56.3 / 53.6 us; 112 tiles: the streamer
// stays ahead).  And, whatever the tile count, where the library plans K ranges side by side that fill the chip:
// from 65 rows, and from 25 / 33 rows on where K is long.
int64_t fp8_tile_plan(int64_t M, int64_t N, int64_t K, int64_t min_m, int64_t min_tiles) {
  if (N % 128 || K % 128) return -1;
  const int64_t tiles = (M + 255) / 256 * (N / 128);        // 256 x 128 output tiles, one workgroup each
  const int64_t need = M > min_m / 4 ? static_cast<int64_t>(mi355q_fp8_gemm_workspace_bytes(M, N, K)) : 0;
  if (need || (M > min_m && tiles >= min_tiles) || (M > min_m / 2 && tiles >= 2 * min_tiles)) return need;
  return -1;
}

PyObject* py_fp8_tile_plan(PyObject*, PyObject* const* a, Py_ssize_t) {
  return PyLong_FromLongLong(fp8_tile_plan(PyLong_AsLongLong(a[0]), PyLong_AsLongLong(a[1]), PyLong_AsLongLong(a[2]),
                                           PyLong_AsLongLong(a[3]), PyLong_AsLongLong(a[4])));
}

// (layer, x, x_scale, min_m, min_tiles, stage_scales): block-scaled weight / weight_scale_inv.  x is 16-bit
// (quantised here per token and group of 128) or fp8 with its scales
PyObject* py_fp8_block_layer(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  static const Bytes n_w("weight"), n_ws("weight_scale_inv"), n_is("input_scale");
  const Ref w(layer_attr(a[0], n_w)), sc(layer_attr(a[0], n_ws));
  const Tensor *xt = as_tensor(a[1]), *wt = as_tensor(w.o), *st = as_tensor(sc.o);
  Tensor xs;
  if (!xt || !wt || !st || !optional_tensor(a[2], xs) || modes_active()) return no();
  if (!xs.defined()) {
    const Ref is(layer_attr(a[0], n_is));
    if (is.o && is.o != Py_None) return no();
  }
  const Tensor& x = *xt;
  const bool quantise = !xs.defined();
  if (wt->dim() != 2 || x.dim() < 1 || x.numel() == 0 || !x.is_contiguous()) return no();
  if (quantise ? !is_16bit(x.scalar_type()) : x.scalar_type() != at::kFloat8_e4m3fn) return no();
  const int64_t N = wt->size(0), K = wt->size(1), M = x.numel() / std::max<int64_t>(x.size(-1), 1);
  if (x.size(-1) != K || K % 128 || N % 128 || wt->scalar_type() != at::kFloat8_e4m3fn || !is_kslab(*wt) ||
      !dense(*st, at::kFloat, N / 128 * (K / 128)) || (!quantise && !dense(xs, at::kFloat, M * (K / 128))))
    return no();
  int64_t need = fp8_tile_plan(M, N, K, PyLong_AsLongLong(a[3]), PyLong_AsLongLong(a[4]));
  size_t mid_need = 0;
  const bool mid = mi355q_q8_mid_plan(0, M, N, K, &mid_need);
  if (mid) need = mid_need;
  const at::ScalarType od = quantise ? x.scalar_type() : at::kBFloat16;
  const OnDevice on(x);
  void* stream = on.stream();
  Scratch ws{nullptr, 0};
  if (need >= 0) {
    // behind the partial sums of a K split (or the first MiB): room for the activation scales in K block major order
    const int64_t stage = !mid && PyObject_IsTrue(a[5]) ? (M + 15) / 16 * 16 * (K / 128) * 4 : 0;
    const int64_t total = (need ? need : stage ? (1 << 20) : 0) + stage;
    if (total) ws = workspace(x, stream, total);
  }
  Tensor out;
  {
    const NoGil free_gil;
    Tensor q = x;
    if (quantise) {
      q = empty(x.sizes(), at::kFloat8_e4m3fn, x);
      xs = empty({M, K / 128}, at::kFloat, x);
      check(mi355q_fp8_group_quant(static_cast<uint8_t*>(q.data_ptr()), static_cast<float*>(xs.data_ptr()), x.data_ptr(), M, K, 128,
                                   0, dtype_code(od), nullptr, 1, stream),
            "fp8_group_quant");
    }
    out = empty(with_last(x, N), od, x);
    const float *xp = static_cast<const float*>(xs.data_ptr()), *wp = static_cast<const float*>(st->data_ptr());
    if (need >= 0)
      check(mi355q_fp8_block_gemm_ws(out.data_ptr(), q.data_ptr(), wt->data_ptr(), xp, wp, nullptr, M, N, K, K, 0, N,
                                     dtype_code(od) | MI355Q_ZEROED_COUNTERS, ws.p, ws.bytes, stream),
            "fp8_block_gemm");
    else
      check(mi355q_kcontig_gemm(out.data_ptr(), q.data_ptr(), wt->data_ptr(), xp, wp, nullptr, 1, 128, M, K, N, MI355Q_F16,
                                dtype_code(od), 1, stream),
            "kcontig_gemm");
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// (layer, x, bias): scales outside the K sum.  Static activation scale where the layer has one, else one per token
PyObject* py_fp8_scaled_layer(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  static const Bytes n_w("weight"), n_ws("weight_scale"), n_is("input_scale");
  const Ref w(layer_attr(a[0], n_w)), sc(layer_attr(a[0], n_ws)), is(layer_attr(a[0], n_is));
  const Tensor *xt = as_tensor(a[1]), *wt = as_tensor(w.o), *st = as_tensor(sc.o);
  Tensor bias, xs;
  if (!xt || !wt || !st || !optional_tensor(a[2], bias) || !optional_tensor(is.o, xs) || modes_active()) return no();
  const Tensor& x = *xt;
  if (wt->dim() != 2 || x.dim() < 1 || x.numel() == 0 || !x.is_contiguous() || !is_16bit(x.scalar_type())) return no();
  const int64_t N = wt->size(0), K = wt->size(1), M = x.numel() / std::max<int64_t>(x.size(-1), 1);
  if (x.size(-1) != K || K % 128 || N % 64 || wt->scalar_type() != at::kFloat8_e4m3fn || !is_kslab(*wt) ||
      !dense(*st, at::kFloat) || (st->numel() != N && st->numel() != 1) || !none_or_dense(bias, x.scalar_type(), N) ||
      !none_or_dense(xs, at::kFloat, 1))
    return no();
  const OnDevice on(x);
  void* stream = on.stream();
  const int dt = dtype_code(x.scalar_type());
  Tensor out;
  if (!xs.defined() && quantises(1, 1, M, N, K, x, Tensor(), *wt, *st, bias)) {
    const NoGil free_gil;
    out = empty(with_last(x, N), x.scalar_type(), x);
    check(mi355q_q8_quant_gemm(out.data_ptr(), x.data_ptr(), wt->data_ptr(), nullptr, static_cast<const float*>(st->data_ptr()), st->numel() > 1,
                               ptr(bias), 1, 1, M, N, K, dt, stream),
          "q8_quant_gemm");
  } else {
    size_t need = 0;
    if (!mi355q_q8_mid_plan(1, M, N, K, &need)) need = mi355q_fp8_gemm_workspace_bytes(M, N, K);
    const Scratch ws = need ? workspace(x, stream, need) : Scratch{nullptr, 0};
    const NoGil free_gil;
    const Tensor q = empty({M, K}, at::kFloat8_e4m3fn, x);
    const bool per_row = !xs.defined();
    if (per_row) {
      xs = empty({M}, at::kFloat, x);
      check(mi355q_fp8_token_quant(static_cast<uint8_t*>(q.data_ptr()), static_cast<float*>(xs.data_ptr()), x.data_ptr(), M, K, dt,
                                   nullptr, stream),
            "fp8_token_quant");
    } else {
      check(mi355q_fp8_static_quant(static_cast<uint8_t*>(q.data_ptr()), x.data_ptr(), static_cast<const float*>(xs.data_ptr()), M, K,
                                    0, dt, nullptr, 1, stream),
            "fp8_static_quant");
    }
    out = empty(with_last(x, N), x.scalar_type(), x);
    check(mi355q_fp8_scaled_gemm_ws(out.data_ptr(), q.data_ptr(), wt->data_ptr(), static_cast<const float*>(xs.data_ptr()),
                                    per_row && M > 1, static_cast<const float*>(st->data_ptr()), st->numel() > 1, ptr(bias), M, N, K,
                                    K, 0, N, dt | MI355Q_ZEROED_COUNTERS, ws.p, ws.bytes, stream),
          "fp8_scaled_gemm");
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// (kind, M, N, K) -> bytes of workspace, or -1 where the kernel for some hundred rows does not take the layer
PyObject* py_q8_mid_plan(PyObject*, PyObject* const* a, Py_ssize_t) {
  size_t need = 0;
  const bool mid = mi355q_q8_mid_plan(PyLong_AsLong(a[0]), PyLong_AsLong(a[1]), PyLong_AsLong(a[2]), PyLong_AsLong(a[3]), &need);
  return PyLong_FromLongLong(mid ? static_cast<int64_t>(need) : -1);
}

// ---- fused MoE ---------------------------------------------------------------------------------------------
// (logits, topk, renormalize) -> (weights, ids)
PyObject* py_fused_topk(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  const Tensor* g = as_tensor(a[0]);
  const int64_t topk = PyLong_AsLongLong(a[1]);
  if (!g || g->dim() != 2 || g->numel() == 0 || !g->is_contiguous() || dtype_code(g->scalar_type()) < 0 || topk < 1 || modes_active())
    return no();
  const int renorm = PyObject_IsTrue(a[2]);
  const OnDevice on(*g);
  Tensor w = empty({g->size(0), topk}, at::kFloat, *g), ids = empty({g->size(0), topk}, at::kInt, *g);
  {
    const NoGil free_gil;
    check(mi355q_topk_softmax(static_cast<float*>(w.data_ptr()), static_cast<int32_t*>(ids.data_ptr()), nullptr, g->data_ptr(),
                              g->size(0), g->size(1), topk, renorm, dtype_code(g->scalar_type()), on.stream()),
          "topk_softmax");
  }
  return PyTuple_Pack(2, Ref(THPVariable_Wrap(std::move(w))).o, Ref(THPVariable_Wrap(std::move(ids))).o);
  END_HANDLE_TH_ERRORS
}

// (logits, topk, renormalize, groups, topk_group, sigmoid, bias) -> (weights, ids)
PyObject* py_grouped_topk(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  const Tensor* g = as_tensor(a[0]);
  Tensor bias;
  const int64_t topk = PyLong_AsLongLong(a[1]);
  if (!g || g->dim() != 2 || g->numel() == 0 || !g->is_contiguous() || dtype_code(g->scalar_type()) < 0 || topk < 1 ||
      !optional_tensor(a[6], bias) || !none_or_dense(bias, at::kFloat, g->size(1)) || modes_active())
    return no();
  const int renorm = PyObject_IsTrue(a[2]), sigmoid = PyObject_IsTrue(a[5]);
  const int groups = PyLong_AsLong(a[3]), keep = PyLong_AsLong(a[4]);
  const OnDevice on(*g);
  Tensor w = empty({g->size(0), topk}, at::kFloat, *g), ids = empty({g->size(0), topk}, at::kInt, *g);
  {
    const NoGil free_gil;
    check(mi355q_grouped_topk(static_cast<float*>(w.data_ptr()), static_cast<int32_t*>(ids.data_ptr()), g->data_ptr(),
                              static_cast<const float*>(ptr(bias)), g->size(0), g->size(1), topk, renorm, groups, keep, sigmoid,
                              dtype_code(g->scalar_type()), on.stream()),
          "grouped_topk");
  }
  return PyTuple_Pack(2, Ref(THPVariable_Wrap(std::move(w))).o, Ref(THPVariable_Wrap(std::move(ids))).o);
  END_HANDLE_TH_ERRORS
}

enum Experts { kW4 = 0, kFp8 = 1, kInt8 = 2 };     // as quant_mode of mi355q_moe_gemm

// The whole sequence of the fused experts on one scratch tensor:
// (mode, group_size, block_m, hidden, w1, w2, w1_scale, w2_scale, w1_zp, w2_zp, topk_weights, topk_ids, output);
// output is the caller's tensor and may be `hidden` itself: hidden is last read by the first GEMM, and the sum
// that writes the output comes after the second.  Returns True, or None where the general path has to take over.
PyObject* py_fused_experts(PyObject*, PyObject* const* a, Py_ssize_t) {
  HANDLE_TH_ERRORS
  const int mode = PyLong_AsLong(a[0]);
  int64_t group = PyLong_AsLongLong(a[1]);
  const int64_t block = PyLong_AsLongLong(a[2]);
  const Tensor *xp = as_tensor(a[3]), *w1p = as_tensor(a[4]), *w2p = as_tensor(a[5]), *s1p = as_tensor(a[6]), *s2p = as_tensor(a[7]),
               *twp = as_tensor(a[10]), *idp = as_tensor(a[11]), *outp = as_tensor(a[12]);
  Tensor z1, z2;
  if (!xp || !w1p || !w2p || !s1p || !s2p || !twp || !idp || !outp || !optional_tensor(a[8], z1) || !optional_tensor(a[9], z2) ||
      modes_active())
    return no();
  const Tensor &x = *xp, &w1 = *w1p, &w2 = *w2p, &tw = *twp, &ids = *idp, &out = *outp;
  const at::ScalarType dt = x.scalar_type();
  if (!is_16bit(dt) || x.dim() != 2 || !x.is_contiguous() || x.numel() == 0 || w1.dim() != 3 || w2.dim() != 3 || ids.dim() != 2 ||
      !dense(out, dt, x.numel()) || block <= 0)
    return no();
  const int64_t E = w1.size(0), M = x.size(0), K = x.size(1), T = ids.size(1), numel = M * T;
  const int64_t N = mode == kW4 ? w1.size(2) : w1.size(1), I = N / 2;      // N = gate and up columns
  if (ids.size(0) != M || numel == 0 || !(dense(ids, at::kInt) || dense(ids, at::kLong)) || !dense(tw, at::kFloat, numel) || N % 2)
    return no();
  // weights [E, N, K] and [E, K, I] (int4: slab tensors [E, K/8, N] and [E, I/8, K])
  if (mode == kW4) {
    if (group <= 0 || K % group || I % group) return no();
    if (!dense(w1, at::kInt) || !dense(w2, at::kInt) || w1.size(1) * 8 != K || w2.size(0) != E || w2.size(1) * 8 != I || w2.size(2) != K)
      return no();
    if (!dense(*s1p, dt, E * (K / group) * N) || !dense(*s2p, dt, E * (I / group) * K)) return no();
    if (!none_or_dense(z1, at::kInt, E * (K / group) * (N / 8)) || !none_or_dense(z2, at::kInt, E * (I / group) * (K / 8))) return no();
  } else {
    const at::ScalarType wt = mode == kFp8 ? at::kFloat8_e4m3fn : at::kChar;
    if (mode != kFp8 && mode != kInt8) return no();
    if (w1.scalar_type() != wt || w2.scalar_type() != wt || !is_kslab(w1) || !is_kslab(w2)) return no();
    if (w1.size(2) != K || w2.size(0) != E || w2.size(1) != K || w2.size(2) != I || K % 128 || I % 128 || N % 128) return no();
    const int64_t n1 = mode == kFp8 ? N / 128 * (K / 128) : N, n2 = mode == kFp8 ? K / 128 * (I / 128) : K;
    if (!dense(*s1p, at::kFloat, E * n1) || !dense(*s2p, at::kFloat, E * n2) || z1.defined() || z2.defined()) return no();
    if (mode == kFp8 && group != 128) return no();
    if (mode == kInt8) group = 1;
  }
  const bool ids64 = ids.scalar_type() == at::kLong;
  if (mode == kFp8 && M <= 4 && mi355q_moe_fp8_unsorted_wanted(M, T, E, K, I)) {
    const auto at16 = [](const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
    if (at16(x) && at16(out) && at16(w1) && at16(w2)) {
      const size_t bytes = mi355q_moe_fp8_unsorted_bytes(M, T, E, K, I);
      const OnDevice on(x);
      {
        const NoGil free_gil;
        const Tensor buf = empty({static_cast<int64_t>(bytes)}, at::kByte, x);
        check(mi355q_moe_fp8_unsorted(out.data_ptr(), x.data_ptr(), w1.data_ptr(), static_cast<const float*>(s1p->data_ptr()), w2.data_ptr(),
                                      static_cast<const float*>(s2p->data_ptr()), static_cast<const float*>(tw.data_ptr()), ids.data_ptr(), ids64, M, T,
                                      E, K, I, dtype_code(dt), buf.data_ptr(), bytes, on.stream()),
              "moe_fp8_unsorted");
      }
      Py_RETURN_TRUE;
    }
  }
  const int64_t blocks = (numel + E * (block - 1)) / block;
  const bool quant = mode != kW4;
  // A wavefront's worth of slots in blocks of 16: the GEMMs sort them themselves, and the first applies the gate, where its launch counts:
  // sixty experts of 2048 x 2816 at 1 / 8 / 16 tokens 32.2 / 39.9 / 51.2 -> 29.5 / 37.8 / 49.3 us, sixteen of 3072 x 8192 at 3 / 16 39.2 / 63.7 ->
  // 36.7 / 62.7; eight of 4096 x 28672 at 1 / 5 / 16 48.6 / 103.2 / 132.5 and 47.5 / 104.1 / 132.4: two streams of weights instead of one.
  const bool unsorted = mode == kW4 && block == 16 && numel <= 64 && group % 128 == 0 && K % 128 == 0 && N % 128 == 0 && I % 128 == 0;
  const bool gate = unsorted && N * K <= (1 << 26);
  const bool sorted_gate = mode == kW4 && !unsorted && mi355q_moe_w4a16_gates(block, K, N, group, z1.defined() ? MI355Q_ZP_PACKED : MI355Q_ZP_NONE);
  const bool gate_up = mode == kFp8 && block <= 64 && N % 256 == 0;       // the first GEMM applies the gate and quantises
  // one allocation: quantised inputs of both GEMMs with their scales, the three intermediate matrices, the alignment
  int64_t total = 0;
  auto room = [&total](int64_t bytes) {
    const int64_t at = total;
    total += (bytes + 255) / 256 * 256;
    return at;
  };
  const int64_t s_cols1 = mode == kFp8 ? K / 128 : 1, s_cols2 = mode == kFp8 ? I / 128 : 1;
  const int64_t o_q1 = room(quant ? M * K : 0), o_s1 = room(quant ? M * s_cols1 * 4 : 0);
  // first GEMM, unless it leaves gated columns, then (dead by then) the second one, unless its sums are f32
  const int64_t o_c1 = room(std::max(gate || sorted_gate || gate_up ? 0 : numel * N, unsorted ? 0 : numel * K) * 2);
  const int64_t o_c2 = room(mode == kFp8 ? 0 : numel * I * 2);
  const int64_t o_q2 = room(quant ? numel * I : 0), o_s2 = room(quant ? numel * s_cols2 * 4 : 0);
  const int64_t o_sorted = room((numel + E * (block - 1)) * 4), o_eid = room(blocks * 4), o_npp = room(4);
  const size_t sums = unsorted ? mi355q_moe_w4a16_unsorted_sum_bytes(numel, E, I, K) : 0;      // of the second GEMM's K ranges
  const int64_t o_sums = room(sums);
  const size_t need = std::max(mi355q_moe_gemm_workspace_bytes(mode, numel, block, blocks, E, K, N),
                               mi355q_moe_gemm_workspace_bytes(mode, numel, block, blocks, E, I, K));
  const OnDevice on(x);
  void* stream = on.stream();
  constexpr size_t kCounters = 1 << 20;      // the first MiB of the scratch holds arrival counters that stay zero
  Scratch ws{nullptr, 0};
  if (need) {
    ws = workspace(x, stream, need + kCounters);
    ws.p += kCounters, ws.bytes -= kCounters;
  }
  {
    const NoGil free_gil;
    const Tensor buf = empty({total}, at::kByte, x);
    char* b = static_cast<char*>(buf.data_ptr());
    const int code = dtype_code(dt), act = mode == kW4 ? code : MI355Q_F16;
    int32_t *sorted = reinterpret_cast<int32_t*>(b + o_sorted), *eid = reinterpret_cast<int32_t*>(b + o_eid),
            *npp = reinterpret_cast<int32_t*>(b + o_npp);
    float *s1 = reinterpret_cast<float*>(b + o_s1), *s2 = reinterpret_cast<float*>(b + o_s2);
    if (mode == kFp8)
      check(mi355q_moe_align_fp8_quant(reinterpret_cast<uint8_t*>(b + o_q1), s1, x.data_ptr(), M, K, code, ids.data_ptr(), ids64, numel, T, E, block,
                                       sorted, eid, npp, stream),
            "moe_align_fp8_quant");
    else if (mode == kInt8)
      check(mi355q_dynamic_int8_quant(reinterpret_cast<int8_t*>(b + o_q1), s1, x.data_ptr(), M, K, code, nullptr, stream),
            "dynamic_int8_quant");
    if (!unsorted && mode != kFp8)
      check(mi355q_moe_align_block_size(ids.data_ptr(), ids64, numel, T, nullptr, E, block, nullptr, sorted, eid, npp, stream), "moe_align_block_size");
    if (unsorted)
      check(mi355q_moe_w4a16_unsorted(b + (gate ? o_c2 : o_c1), x.data_ptr(), static_cast<const int32_t*>(w1.data_ptr()), s1p->data_ptr(), ptr(z1),
                                      z1.defined() ? MI355Q_ZP_PACKED : MI355Q_ZP_NONE, group, nullptr, ids.data_ptr(), ids64, numel, T, E, K, N,
                                      gate, code, stream),
            "moe_w4a16_unsorted");
    else if (gate_up)
      check(mi355q_moe_fp8_gate_up_quant(reinterpret_cast<uint8_t*>(b + o_q2), s2, b + o_q1, w1.data_ptr(), s1, static_cast<const float*>(s1p->data_ptr()),
                                         sorted, eid, npp, numel, T, block, blocks, E, K, N, code, 1, stream),
            "moe_fp8_gate_up_quant");
    else if (sorted_gate)
      check(mi355q_moe_w4a16_gate_up(b + o_c2, x.data_ptr(), static_cast<const int32_t*>(w1.data_ptr()), s1p->data_ptr(), ptr(z1),
                                     z1.defined() ? MI355Q_ZP_PACKED : MI355Q_ZP_NONE, group, sorted, eid, npp, numel, T, block, blocks, E, K, N, code,
                                     ws.p, ws.bytes, stream),
            "moe_w4a16_gate_up");
    else
      check(mi355q_moe_gemm(b + o_c1, quant ? static_cast<void*>(b + o_q1) : x.data_ptr(), w1.data_ptr(), quant ? s1 : nullptr,
                          s1p->data_ptr(), ptr(z1), z1.defined() ? MI355Q_ZP_PACKED : MI355Q_ZP_NONE, mode, group, nullptr, sorted, eid,
                          npp, numel, T, block, blocks, E, K, N, act, code, quant, ws.p, ws.bytes, stream),
          "moe_gemm");
    if (mode == kFp8 && !gate_up)
      check(mi355q_fp8_group_quant(reinterpret_cast<uint8_t*>(b + o_q2), s2, b + o_c1, numel, I, 128, 1, code, nullptr, 1, stream),
            "fp8_group_quant");
    else if (mode != kFp8 && !gate && !sorted_gate)
      check(mi355q_silu_and_mul(b + o_c2, b + o_c1, numel, I, code, nullptr, 1, stream), "silu_and_mul");
    if (mode == kInt8)
      check(mi355q_dynamic_int8_quant(reinterpret_cast<int8_t*>(b + o_q2), s2, b + o_c2, numel, I, code, nullptr, stream),
            "dynamic_int8_quant");
    if (unsorted) {
      check(mi355q_moe_w4a16_unsorted_sum(out.data_ptr(), b + o_c2, static_cast<const int32_t*>(w2.data_ptr()), s2p->data_ptr(), ptr(z2),
                                          z2.defined() ? MI355Q_ZP_PACKED : MI355Q_ZP_NONE, group, static_cast<const float*>(tw.data_ptr()),
                                          ids.data_ptr(), ids64, M, T, E, I, K, code, b + o_sums, sums, stream),
            "moe_w4a16_unsorted_sum");
    } else if (mode == kW4) {
      check(mi355q_moe_w4a16_down_sum_ids(out.data_ptr(), b + o_c1, b + o_c2, static_cast<const int32_t*>(w2.data_ptr()), s2p->data_ptr(), ptr(z2),
                                          z2.defined() ? MI355Q_ZP_PACKED : MI355Q_ZP_NONE, group, static_cast<const float*>(tw.data_ptr()),
                                          ids.data_ptr(), ids64, sorted, eid, npp, M, T, block, blocks, E, I, K, code, ws.p, ws.bytes, stream),
            "moe_w4a16_down_sum_ids");
    } else {
      check(mi355q_moe_gemm(b + o_c1, b + o_q2, w2.data_ptr(), s2, s2p->data_ptr(), nullptr, MI355Q_ZP_NONE, mode, group, static_cast<const float*>(tw.data_ptr()), sorted,
                           eid, npp, numel, 1, block, blocks, E, I, K, act, code, quant, ws.p, ws.bytes, stream),
            "moe_gemm");
      check(mi355q_moe_sum(out.data_ptr(), b + o_c1, M, T, K, code, code, nullptr, stream), "moe_sum");
    }
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

PyObject* py_register_activation_ops(PyObject*, PyObject*) {
  HANDLE_TH_ERRORS
  register_activation_ops();
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// ---- the workspace function of vllm_gcu_amd.kernels._runtime -------------------------------------------------
PyObject* g_workspace_fn = nullptr;

PyObject* py_set_workspace(PyObject*, PyObject* const* a, Py_ssize_t) {
  Py_INCREF(a[0]);
  Py_XSETREF(g_workspace_fn, a[0]);
  Py_RETURN_NONE;
}

#define MQ_FAST(NAME, FN) {NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(FN)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    MQ_FAST("w4a16", py_w4a16),
    MQ_FAST("w4a16_layer", py_w4a16_layer),
    MQ_FAST("w8a8_static_layer", py_w8a8_static_layer),
    MQ_FAST("int8_dynamic_layer", py_int8_dynamic_layer),
    MQ_FAST("int8_stream_rows", py_int8_stream_rows),
    MQ_FAST("fp8_block_layer", py_fp8_block_layer),
    MQ_FAST("fp8_scaled_layer", py_fp8_scaled_layer),
    MQ_FAST("fp8_tile_plan", py_fp8_tile_plan),
    MQ_FAST("q8_mid_plan", py_q8_mid_plan),
    MQ_FAST("fused_topk", py_fused_topk),
    MQ_FAST("grouped_topk", py_grouped_topk),
    MQ_FAST("fused_experts", py_fused_experts),
    MQ_FAST("kslab_register", py_kslab_register),
    MQ_FAST("kslab_unregister", py_kslab_unregister),
    MQ_FAST("is_kslab", py_is_kslab),
    MQ_FAST("set_workspace", py_set_workspace),
    {"register_activation_ops", py_register_activation_ops, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
#undef MQ_FAST

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_mi355q_host", "Native host path of vllm_gcu_amd.", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

bool is_kslab(const Tensor& w) {
  std::lock_guard<std::mutex> lk(g_kslab_mu);
  auto& m = kslab_map(w.get_device());
  auto it = m.find(reinterpret_cast<uintptr_t>(w.data_ptr()));
  return it != m.end() && it->second.bytes == static_cast<int64_t>(w.numel() * w.element_size());
}

Scratch workspace(const Tensor& like, void* stream, size_t bytes) {
  struct Entry {
    int dev;
    void* stream;
    Tensor buf;
  };
  // guarded by the GIL; a program has few streams.  Never destroyed: the runtime is gone by then
  static std::vector<Entry>& held = *new std::vector<Entry>;
  const int dev = like.get_device();
  Entry* e = nullptr;
  for (Entry& h : held)
    if (h.dev == dev && h.stream == stream) {
      e = &h;
      break;
    }
  if (!e || static_cast<size_t>(e->buf.numel()) < bytes) {
    TORCH_CHECK(g_workspace_fn, "mi355q: the workspace function is not set");
    const Ref d(THPDevice_New(like.device())), n(PyLong_FromSize_t(bytes));
    const Ref t(d.o && n.o ? PyObject_CallFunctionObjArgs(g_workspace_fn, d.o, n.o, nullptr) : nullptr);
    if (!t.o) throw python_error();
    const Tensor buf = THPVariable_Unpack(t.o);
    // (the call may have let other threads in: look again)
    e = nullptr;
    for (Entry& h : held)
      if (h.dev == dev && h.stream == stream) e = &h;
    if (e)
      e->buf = buf;
    else {
      held.push_back({dev, stream, buf});
      e = &held.back();
    }
  }
  return {static_cast<char*>(e->buf.data_ptr()), static_cast<size_t>(e->buf.numel())};
}

}  // namespace mi355q_host

PyMODINIT_FUNC PyInit__mi355q_host() {
  using namespace mi355q_host;
  auto attribute = [](const char* module, const char* name) -> PyObject* {
    const Ref m(PyImport_ImportModule(module));
    return m.o ? PyObject_GetAttrString(m.o, name) : nullptr;
  };
  g_disabled_torch_function = attribute("torch._C", "_disabled_torch_function_impl");
  g_device_context = attribute("torch.utils._device", "DeviceContext");
  if (!g_disabled_torch_function || !g_device_context) return nullptr;
  return PyModule_Create(&kModule);
}
