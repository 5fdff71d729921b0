// Native host side of eager calls: the module forwards' bound calls and the CUDA kernels of the operators that a
// worker's own modules call one after another. Everything here checks its tensors, allocates outputs and workspaces
// from torch's allocator and calls the C-ABI library's entry points on the current stream, with the arguments the
// Python bodies in ops.py pass, so results are theirs bit for bit. Whatever does not fit (a mode, a subclass, an
// operand the contract refuses) goes back to Python: a bound call returns None and the module takes its general
// path, an operator kernel calls the Python body, which raises the contract's own error.
//
// Why: below about 20 us of GPU work a call was bound by Python. Back to back, one token through a W4A4 3072 -> 18432
// layer 23.1 -> 16.1 us, through the AWQ layer of that shape 21.1 -> 11.8, 256 tokens through a W8A8 3072 -> 3072
// layer 20.6 -> 12.9, the quantize / GEMM operator pair at 1024 x 9216 x 3072 87.6 -> 67.1.
#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>
#include <torch/version.h>

#include <ATen/PythonTorchFunctionTLS.h>

#include <string>
#include <vector>

#include "gen_worker_amd.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// the C-ABI library's entry points (addresses from the library the Python binding loaded: one instance, one state)
struct Abi {
  decltype(&gwa_svdq_quant_int4) svdq_quant_int4;
  decltype(&gwa_svdq_pack_weight_fp6) svdq_pack_weight_fp6;
  decltype(&gwa_svdq_gemm_w4a4_fp6) svdq_gemm_w4a4_fp6;
  decltype(&gwa_svdq_w4a4_linear_fp6) svdq_w4a4_linear_fp6;
  decltype(&gwa_svdq_w4a4_linear_fp6_workspace) svdq_w4a4_linear_fp6_workspace;
  decltype(&gwa_svdq_w4a4_linear_gemv) svdq_w4a4_linear_gemv;
  decltype(&gwa_svdq_w4a4_linear_gemv_workspace) svdq_w4a4_linear_gemv_workspace;
  decltype(&gwa_w8a8_quant) w8a8_quant;
  decltype(&gwa_w8a8_gemm) w8a8_gemm;
  decltype(&gwa_awq_w4a16_mm) awq_w4a16_mm;
};
Abi g_abi;
bool g_bound = false;

// Python callables: an operator's Python body by name, and the fp6 record cache of reference-schema weights
PyObject* g_bodies = nullptr;
PyObject* g_ref_records = nullptr;

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor empty_like_device(at::IntArrayRef sizes, at::ScalarType dt, const Tensor& like) {
  return at::detail::empty_cuda(sizes, dt, like.device(), std::nullopt);
}

int dt_code(at::ScalarType dt) {
  return dt == at::kBFloat16 ? GWA_DT_BF16 : dt == at::kHalf ? GWA_DT_F16 : dt == at::kFloat ? GWA_DT_F32 : -1;
}

bool dense_on(const Tensor& t, at::ScalarType dt, const at::Device& dev) {
  return t.scalar_type() == dt && t.layout() == at::kStrided && t.device() == dev && t.is_contiguous();
}
bool absent_or_dense(const OptTensor& t, at::ScalarType dt, const at::Device& dev) {
  return !t.has_value() || dense_on(*t, dt, dev);
}
const void* ptr(const OptTensor& t) { return t.has_value() ? t->data_ptr() : nullptr; }
int64_t readable(const Tensor& t) {
  return (int64_t)t.storage().nbytes() - t.storage_offset() * (int64_t)t.element_size();
}

// ---------------------------------------------------------------------------
// bound module calls
// ---------------------------------------------------------------------------

enum Kind { kW4A4 = 0, kW8A8 = 1 };

// One attribute the binding was made from: where it lives in the module (its __dict__, _buffers or _parameters) and
// the object it was. One operand: the tensor, where its storage was, and for what derived buffers were computed
// from, its version. They only say whether the binding is still the module's; every call checks the operands again
// and takes their pointers anew.
struct Attr {
  int where;
  PyObject* key;
  PyObject* value;
};
struct Operand {
  Tensor t;
  const void* at = nullptr;
  bool versioned = false;
  int64_t version = 0;
  bool defined() const { return t.defined(); }
  template <class T>
  T* p() const {
    return t.defined() ? (T*)t.data_ptr() : nullptr;
  }
  // absent, or dense on dev with this dtype and shape
  bool fits(at::ScalarType dt, const at::Device& dev, at::IntArrayRef sizes) const {
    return !t.defined() || (dense_on(t, dt, dev) && t.sizes().equals(sizes));
  }
};

struct BoundCall {
  PyObject_HEAD
  Kind kind;
  std::vector<Attr>* attrs;
  std::vector<Operand>* ops;
  at::ScalarType out_dtype;
  int64_t k, n, rank, gemv_max_m, flags;
};

PyObject* g_names[2];  // "_buffers", "_parameters"

void bound_dealloc(PyObject* o) {
  BoundCall* b = (BoundCall*)o;
  if (b->attrs)
    for (Attr& a : *b->attrs) {
      Py_XDECREF(a.key);
      Py_XDECREF(a.value);
    }
  delete b->attrs;
  delete b->ops;
  Py_TYPE(o)->tp_free(o);
}

// BoundCall(kind, attrs [(where, name, value)], operands [tensor or None], versions [int or None per operand],
//           out_dtype, k, n, rank, gemv_max_m, flags)
int bound_init(PyObject* o, PyObject* args, PyObject*) {
  BoundCall* b = (BoundCall*)o;
  int kind;
  PyObject *attrs, *ops, *versions, *dtype;
  long long k, n, rank, gm, flags;
  if (!PyArg_ParseTuple(args, "iO!O!O!OLLLLL", &kind, &PyList_Type, &attrs, &PyList_Type, &ops, &PyList_Type, &versions,
                        &dtype, &k, &n, &rank, &gm, &flags))
    return -1;
  if (!THPDtype_Check(dtype) || PyList_GET_SIZE(ops) != PyList_GET_SIZE(versions) || b->attrs) {
    PyErr_SetString(PyExc_TypeError, "BoundCall: bad arguments");
    return -1;
  }
  b->kind = (Kind)kind;
  b->out_dtype = ((THPDtype*)dtype)->scalar_type;
  b->k = k, b->n = n, b->rank = rank, b->gemv_max_m = gm, b->flags = flags;
  b->attrs = new std::vector<Attr>();
  b->ops = new std::vector<Operand>();
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(attrs); ++i) {
    int where;
    PyObject *key, *value;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(attrs, i), "iOO", &where, &key, &value)) return -1;
    Py_INCREF(key);
    Py_INCREF(value);
    b->attrs->push_back({where, key, value});
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(ops); ++i) {
    Operand op;
    PyObject* t = PyList_GET_ITEM(ops, i);
    if (t != Py_None) {
      if (!THPVariable_Check(t)) {
        PyErr_SetString(PyExc_TypeError, "BoundCall: operands are tensors or None");
        return -1;
      }
      op.t = THPVariable_Unpack(t);
      op.at = op.t.data_ptr();
      PyObject* v = PyList_GET_ITEM(versions, i);
      if (v != Py_None) {
        op.versioned = true;
        op.version = PyLong_AsLongLong(v);
      }
    }
    b->ops->push_back(std::move(op));
  }
  return PyErr_Occurred() ? -1 : 0;
}

// Everything the binding was made from is still so: the same attribute objects, the same storages, no in-place
// update of what derived buffers were computed from.
bool still_bound(const BoundCall* b, PyObject* dict) {
  PyObject* where[3] = {dict, PyDict_GetItem(dict, g_names[0]), PyDict_GetItem(dict, g_names[1])};
  for (const Attr& a : *b->attrs) {
    PyObject* d = where[a.where];
    if (!d || !PyDict_Check(d) || PyDict_GetItem(d, a.key) != a.value) return false;
  }
  for (const Operand& op : *b->ops) {
    if (!op.t.defined()) continue;
    if (op.t.data_ptr() != op.at) return false;
    if (op.versioned && (op.t.is_inference() || op.t._version() != op.version)) return false;
  }
  return true;
}

// Keys under which the dispatcher does something to an operand ahead of an operator's CUDA kernel: a wrapper that hides
// its storage, or a lazy negation, whose storage holds the values before it
constexpr c10::DispatchKeySet kNotPlain({c10::DispatchKey::Python, c10::DispatchKey::Functionalize,
                                         c10::DispatchKey::Negative, c10::DispatchKey::Conjugate,
                                         c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                         c10::DispatchKey::ZeroTensor});
bool plain_tensor(const Tensor& t) {
  return !(t.requires_grad() && at::GradMode::is_enabled()) && !t.key_set().has_any(kNotPlain);
}

// A plain tensor in plain eager mode: what ops.eager_call_ok asks. A trace (which sets no mode) records operators: it
// would hold what is computed beside them as a constant.
bool plain_call(const Tensor& x) {
  return plain_tensor(x) && x.is_cuda() && x.layout() == at::kStrided && x.has_storage() &&
         c10::impl::TorchDispatchModeTLS::stack_len() == 0 && !at::impl::torch_function_mode_enabled() &&
         !torch::jit::tracer::isTracing();
}

// the output of a layer for x [..., k]: x's leading dimensions and n columns
Tensor layer_output(const Tensor& x, int64_t n, at::ScalarType dt) {
  c10::SmallVector<int64_t, 5> sizes(x.sizes().begin(), x.sizes().end());
  sizes[sizes.size() - 1] = n;
  return empty_like_device(sizes, dt, x);
}

// operands: weight_fp6, smooth, proj_down_op6, weight, weight_scale, second, proj_up, bias, proj_down (held only)
int run_w4a4(const BoundCall* b, const Tensor& x, int64_t m, Tensor& out) {
  const std::vector<Operand>& op = *b->ops;
  const at::Device dev = x.device();
  const int64_t k = b->k, n = b->n, r = b->rank, stages = (k + 127) / 128;
  const int odt = dt_code(b->out_dtype);
  if (op.size() != 9 || !op[0].defined() || !op[0].fits(at::kByte, dev, {stages, n, GWA_FP6_REC}) ||
      !op[1].fits(at::kBFloat16, dev, {k}) || !op[2].fits(at::kBFloat16, dev, {stages * 128, r}) ||
      !op[3].fits(at::kByte, dev, {n, k / 2}) || !op[4].fits(at::kHalf, dev, {n, k / 64}) || !op[3].defined() ||
      !op[4].defined() || !op[6].fits(at::kBFloat16, dev, {n, r}) || !op[7].fits(at::kBFloat16, dev, {n}) ||
      (r > 0) != op[2].defined() || (r > 0) != op[6].defined() ||
      (odt != GWA_DT_BF16 && odt != GWA_DT_F16))
    return -1;
  const int64_t sec_n = op[5].defined() ? op[5].t.numel() : 0;
  if (op[5].defined() && !dense_on(op[5].t, at::kFloat, dev)) return -1;
  out = layer_output(x, n, b->out_dtype);
  void* const s = stream_of(x);
  if (m <= b->gemv_max_m) {
    const int64_t wsn = std::max<int64_t>(g_abi.svdq_w4a4_linear_gemv_workspace(m, k, r), 256);
    const Tensor ws = empty_like_device({wsn}, at::kByte, x);
    return g_abi.svdq_w4a4_linear_gemv((const uint16_t*)x.data_ptr(), k, op[1].p<const uint16_t>(), nullptr,
                                       op[2].p<const uint16_t>(), r, op[3].p<const uint8_t>(), op[4].p<const uint16_t>(),
                                       op[5].p<const float>(), sec_n, op[6].p<const uint16_t>(),
                                       op[7].p<const uint16_t>(), out.data_ptr(), odt, (int)b->flags, m, n, k,
                                       (uint8_t*)ws.data_ptr(), wsn, s);
  }
  const int64_t wsn = g_abi.svdq_w4a4_linear_fp6_workspace(m, k, r);
  const Tensor ws = empty_like_device({wsn}, at::kByte, x);
  return g_abi.svdq_w4a4_linear_fp6((const uint16_t*)x.data_ptr(), k, op[1].p<const uint16_t>(), nullptr,
                                    op[2].p<const uint16_t>(), r, op[0].p<const uint8_t>(), readable(op[0].t),
                                    op[5].p<const float>(), sec_n, op[6].p<const uint16_t>(),
                                    op[7].p<const uint16_t>(), out.data_ptr(), odt, (int)b->flags, m, n, k,
                                    (uint8_t*)ws.data_ptr(), wsn, s);
}

// operands: weight, weight_scale, bias, input_scale; flags: pertensor
int run_w8a8(const BoundCall* b, const Tensor& x, int64_t m, Tensor& out) {
  const std::vector<Operand>& op = *b->ops;
  const at::Device dev = x.device();
  const int64_t k = b->k, n = b->n, scales = b->flags ? 1 : m;
  const int odt = dt_code(b->out_dtype);
  if (op.size() != 4 || !op[0].defined() || !op[0].fits(at::kChar, dev, {n, k}) || !op[1].defined() ||
      !op[1].fits(at::kFloat, dev, {n, 1}) ||
      (op[3].defined() && (!dense_on(op[3].t, at::kFloat, dev) || op[3].t.numel() != 1)) ||
      (odt != GWA_DT_BF16 && odt != GWA_DT_F16))
    return -1;
  int bdt = 0;
  if (op[2].defined()) {
    bdt = dt_code(op[2].t.scalar_type());
    if (bdt < 0 || !op[2].fits(op[2].t.scalar_type(), dev, {n})) return -1;
  }
  const Tensor q = empty_like_device({m, k}, at::kChar, x);
  const Tensor sa = empty_like_device({scales}, at::kFloat, x);
  Tensor ws;  // the per-tensor maximum's cell
  if (b->flags && !op[3].defined()) ws = empty_like_device({1}, at::kInt, x);
  out = layer_output(x, n, b->out_dtype);
  void* const s = stream_of(x);
  const int rc = g_abi.w8a8_quant((const uint16_t*)x.data_ptr(), k, (int8_t*)q.data_ptr(), (float*)sa.data_ptr(),
                                  op[3].p<const float>(), (int)b->flags,
                                  ws.defined() ? (uint32_t*)ws.data_ptr() : nullptr, m, k, s);
  if (rc != GWA_OK) return rc;
  return g_abi.w8a8_gemm((const int8_t*)q.data_ptr(), op[0].p<const int8_t>(), (const float*)sa.data_ptr(), scales,
                         op[1].p<const float>(), op[2].p<const void>(), bdt, out.data_ptr(), odt, m, n, k, s);
}

// rows of x [..., k] when it is a plain bf16 activation of this layer, else 0
int64_t plain_rows(const Tensor& x, int64_t k) {
  const int64_t d = x.dim();
  if (!plain_call(x) || x.scalar_type() != at::kBFloat16 || d < 1 || k <= 0 || x.size(d - 1) != k || !x.is_contiguous())
    return 0;
  return x.numel() / k;
}

// BoundCall.run(x, module.__dict__) -> the layer's output, or None where the general path has to decide (it meets a
// refusal of the library too, and raises it)
PyObject* bound_run(PyObject* o, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  BoundCall* b = (BoundCall*)o;
  if (nargs != 2 || !THPVariable_CheckExact(args[0]) || !PyDict_Check(args[1]) || !b->ops) Py_RETURN_NONE;
  const Tensor& x = THPVariable_Unpack(args[0]);
  const int64_t m = plain_rows(x, b->k);
  if (m == 0 || !still_bound(b, args[1])) Py_RETURN_NONE;
  Tensor out;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    rc = b->kind == kW4A4 ? run_w4a4(b, x, m, out) : run_w8a8(b, x, m, out);
  }
  if (rc != GWA_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

bool awq_fits(const Tensor& weight, const Tensor& wscales, const Tensor& wzeros, const OptTensor& bias,
              const at::Device& dev, int64_t k) {
  if (weight.dim() != 2) return false;
  const int64_t n = weight.size(0);
  return n % 16 == 0 && k % 128 == 0 && weight.size(1) * 2 == k && dense_on(weight, at::kByte, dev) &&
         dense_on(wscales, at::kBFloat16, dev) && wscales.sizes().equals({n, k / 64}) &&
         dense_on(wzeros, at::kBFloat16, dev) && wzeros.sizes().equals({n, k / 64}) &&
         absent_or_dense(bias, at::kBFloat16, dev) && (!bias.has_value() || bias->numel() == n);
}

// awq_forward(x, weight, wscales, wzeros, bias, max_rows) -> the AWQ layer's output for up to max_rows rows, or None
// where the operator has to decide
PyObject* awq_forward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 6 || !g_bound || !THPVariable_CheckExact(args[0])) Py_RETURN_NONE;
  for (int i = 1; i < 5; ++i)  // operands that a subclass, autograd or a transform has a say in are the operator's
    if (!(i == 4 && args[i] == Py_None) &&
        (!THPVariable_CheckExact(args[i]) || !plain_tensor(THPVariable_Unpack(args[i]))))
      Py_RETURN_NONE;
  const Tensor &x = THPVariable_Unpack(args[0]), &w = THPVariable_Unpack(args[1]), &sc = THPVariable_Unpack(args[2]),
               &z = THPVariable_Unpack(args[3]);
  OptTensor bias;
  if (args[4] != Py_None) bias = THPVariable_Unpack(args[4]);
  const int64_t k = w.dim() == 2 ? w.size(1) * 2 : 0, m = plain_rows(x, k);
  if (m == 0 || m > PyLong_AsLongLong(args[5]) || !awq_fits(w, sc, z, bias, x.device(), k)) Py_RETURN_NONE;
  Tensor out;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    out = layer_output(x, w.size(0), at::kBFloat16);
    rc = g_abi.awq_w4a16_mm((const uint16_t*)x.data_ptr(), k, (const uint8_t*)w.data_ptr(),
                            (const uint16_t*)sc.data_ptr(), (const uint16_t*)z.data_ptr(), (const uint16_t*)ptr(bias),
                            (uint16_t*)out.data_ptr(), m, w.size(0), k, stream_of(x));
  }
  if (rc != GWA_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

PyMethodDef bound_methods[] = {
    {"run", (PyCFunction)(void (*)(void))bound_run, METH_FASTCALL,
     "run(x, module.__dict__) -> the layer's output, or None where its general path has to decide"},
    {nullptr, nullptr, 0, nullptr}};

PyTypeObject BoundType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---------------------------------------------------------------------------
// operator kernels (CUDA dispatch key; the Python definitions keep the schemas, fake and autograd behaviour)
// ---------------------------------------------------------------------------

template <class R, class... A>
R python_body(const char* name, const A&... args) {
  pybind11::gil_scoped_acquire gil;
  pybind11::object body = pybind11::reinterpret_borrow<pybind11::dict>(g_bodies)[name];
  return body(args...).template cast<R>();
}

std::tuple<Tensor, Tensor> op_svdq_quant(const Tensor& x2, const OptTensor& smooth, const Tensor& s2, bool blocked) {
  const at::Device dev = x2.device();
  const int64_t k = x2.dim() == 2 ? x2.size(1) : 0;
  if (!blocked && k > 0 && k % 64 == 0 && dense_on(x2, at::kBFloat16, dev) &&
      absent_or_dense(smooth, at::kBFloat16, dev) && (!smooth.has_value() || smooth->numel() == k) &&
      dense_on(s2, at::kFloat, dev) && s2.numel() == 1) {
    const int64_t m = x2.size(0);
    Tensor q = empty_like_device({m, k / 2}, at::kByte, x2);
    Tensor sc = empty_like_device({m, k / 64}, at::kHalf, x2);
    if (g_abi.svdq_quant_int4((const uint16_t*)x2.data_ptr(), x2.stride(0), (const uint16_t*)ptr(smooth),
                              (const float*)s2.data_ptr(), nullptr, 0, GWA_QFMT_INT4, (uint8_t*)q.data_ptr(),
                              sc.data_ptr(), nullptr, m, k, stream_of(x2)) == GWA_OK)
      return {q, sc};
  }
  return python_body<std::tuple<Tensor, Tensor>>("svdq_quant", x2, smooth, s2, blocked);
}

Tensor op_svdq_gemm_w4a4_lora(const Tensor& qa, const Tensor& sa, const Tensor& wq_kn, const Tensor& ws,
                              const Tensor& s2, const Tensor& second, const Tensor& la, const Tensor& up,
                              const OptTensor& bias) {
  const at::Device dev = qa.device();
  if (qa.dim() == 2 && wq_kn.dim() == 2 && up.dim() == 2) {
    const int64_t m = qa.size(0), kh = wq_kn.size(0), n = wq_kn.size(1), k = 2 * kh, r = up.size(1);
    if (m > 0 && k > 0 && k % 64 == 0 && n % 16 == 0 && (r == 16 || r == 32 || r == 64 || r == 128) &&
        qa.size(1) == kh && dense_on(qa, at::kByte, dev) && dense_on(wq_kn, at::kByte, dev) &&
        dense_on(sa, at::kHalf, dev) && sa.sizes().equals({m, k / 64}) && dense_on(ws, at::kHalf, dev) &&
        ws.sizes().equals({n, k / 64}) && dense_on(s2, at::kFloat, dev) && s2.numel() == 1 &&
        dense_on(second, at::kFloat, dev) && dense_on(up, at::kBFloat16, dev) && up.size(0) == n &&
        dense_on(la, at::kBFloat16, dev) && la.sizes().equals({m, r}) &&
        absent_or_dense(bias, at::kBFloat16, dev) && (!bias.has_value() || bias->numel() == n)) {
      Tensor w6;
      {
        pybind11::gil_scoped_acquire gil;
        w6 = pybind11::reinterpret_borrow<pybind11::object>(g_ref_records)(wq_kn, ws).cast<Tensor>();
      }
      const int64_t stages = (k + 127) / 128, bytes = stages * m * GWA_FP6_REC + GWA_FP6_RECORD_SLACK;
      const Tensor q6 = empty_like_device({bytes}, at::kByte, qa);
      Tensor out = empty_like_device({m, n}, at::kBFloat16, qa);
      void* const s = stream_of(qa);
      int rc = g_abi.svdq_pack_weight_fp6((const uint8_t*)qa.data_ptr(), sa.data_ptr(), (uint8_t*)q6.data_ptr(), m, k,
                                          s);
      if (rc == GWA_OK)
        rc = g_abi.svdq_gemm_w4a4_fp6((const uint8_t*)q6.data_ptr(), bytes, (const uint8_t*)w6.data_ptr(), readable(w6),
                                      (const float*)s2.data_ptr(), (const float*)second.data_ptr(), second.numel(),
                                      la.data_ptr(), (const uint16_t*)up.data_ptr(), r, (const uint16_t*)ptr(bias),
                                      out.data_ptr(), GWA_DT_BF16, 0, m, n, stages * 128, s);
      if (rc == GWA_OK) return out;
    }
  }
  return python_body<Tensor>("svdq_gemm_w4a4_lora", qa, sa, wq_kn, ws, s2, second, la, up, bias);
}

// registered once the library is bound
void register_kernels() {
  static torch::Library lib(torch::Library::IMPL, "cozy_gen_worker", c10::DispatchKey::CUDA, __FILE__, __LINE__);
  lib.impl("svdq_quant", op_svdq_quant);
  lib.impl("svdq_gemm_w4a4_lora", op_svdq_gemm_w4a4_lora);
}

// bind(addresses {symbol: int}, bodies {operator: Python body}, ref_records callable)
PyObject* host_bind(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *addr, *bodies, *records;
  if (!PyArg_ParseTuple(args, "O!O!O", &PyDict_Type, &addr, &PyDict_Type, &bodies, &records)) return nullptr;
  Abi a{};
#define GWA_BIND(field)                                                        \
  do {                                                                         \
    PyObject* v = PyDict_GetItemString(addr, "gwa_" #field);                   \
    if (!v) {                                                                  \
      PyErr_SetString(PyExc_KeyError, "gwa_" #field);                          \
      return nullptr;                                                          \
    }                                                                          \
    a.field = (decltype(a.field))PyLong_AsVoidPtr(v);                          \
    if (PyErr_Occurred()) return nullptr;                                      \
  } while (0)
  GWA_BIND(svdq_quant_int4);
  GWA_BIND(svdq_pack_weight_fp6);
  GWA_BIND(svdq_gemm_w4a4_fp6);
  GWA_BIND(svdq_w4a4_linear_fp6);
  GWA_BIND(svdq_w4a4_linear_fp6_workspace);
  GWA_BIND(svdq_w4a4_linear_gemv);
  GWA_BIND(svdq_w4a4_linear_gemv_workspace);
  GWA_BIND(w8a8_quant);
  GWA_BIND(w8a8_gemm);
  GWA_BIND(awq_w4a16_mm);
#undef GWA_BIND
  Py_INCREF(bodies);
  Py_INCREF(records);
  Py_XDECREF(g_bodies);
  Py_XDECREF(g_ref_records);
  g_bodies = bodies;
  g_ref_records = records;
  g_abi = a;
  if (!g_bound) register_kernels();
  g_bound = true;
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef module_methods[] = {{"bind", host_bind, METH_VARARGS, "bind(addresses, bodies, ref_records)"},
                                {"awq_forward", (PyCFunction)(void (*)(void))awq_forward, METH_FASTCALL,
                                 "awq_forward(x, weight, wscales, wzeros, bias, max_rows) -> output or None"},
                                {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host_calls", "Native host side of eager calls.", -1, module_methods};

}  // namespace

PyMODINIT_FUNC PyInit__host_calls() {
  BoundType.tp_name = "gen_worker_amd._host_calls.BoundCall";
  BoundType.tp_basicsize = sizeof(BoundCall);
  BoundType.tp_flags = Py_TPFLAGS_DEFAULT;
  BoundType.tp_new = PyType_GenericNew;
  BoundType.tp_init = bound_init;
  BoundType.tp_dealloc = bound_dealloc;
  BoundType.tp_methods = bound_methods;
  BoundType.tp_doc = "A quantized layer's resident operands bound for eager calls.";
  if (PyType_Ready(&BoundType) < 0) return nullptr;
  g_names[0] = PyUnicode_InternFromString("_buffers");
  g_names[1] = PyUnicode_InternFromString("_parameters");
  PyObject* m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  Py_INCREF(&BoundType);
  if (PyModule_AddObject(m, "BoundCall", (PyObject*)&BoundType) < 0) return nullptr;
  // what this was compiled against: compared with the library's and torch's own before anything is bound
  if (PyModule_AddIntConstant(m, "GWA_VERSION", GWA_VERSION) < 0) return nullptr;
  if (PyModule_AddStringConstant(m, "TORCH_VERSION", TORCH_VERSION) < 0) return nullptr;
  return m;
}
