// Python module _native: whole calls of the package whose device work is short
// enough that the interpreter bounded them (one decode token through a
// projection: 17 us of kernels behind 32 us of argument checks, allocations
// and ctypes structs). Each function takes the plain case - exact tensors or
// parameters on the current device, in the layout the kernels read in place -
// checks it completely, allocates the outputs and calls the C ABI on the
// current stream; for anything else it returns None without having done
// anything, and the Python route (which converts, copies or raises) runs.
// Host time of a call, measured: a one-row projection 32 -> 10 us (the whole
// call 31.2 -> 14.7), a 64-row one with split K 36 -> 14, an attention 45 -> 11
// (16 heads x 353 x 1000 fp32: 45.8 -> 30.4), a modulated norm with 16
// segments 78 -> 25 (its labels came by a copy that waited for the stream).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <vector>

#include "w8a8.h"

namespace {

PyObject* g_error_class = nullptr;   // _abi.W8A8Error(function, status, message)

// The tensor of a plain torch.Tensor or Parameter on the current GPU, or null.
// Subclasses, functorch wrappers and dispatch modes take the Python route.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckTypeExact(Py_TYPE(o))) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.get_device() != c10::hip::current_device() || t.layout() != at::kStrided ||
      !t.has_storage() || t.is_neg() || t.is_conj())
    return nullptr;
  const auto keys = t.key_set();
  if (keys.has(c10::DispatchKey::Python) || keys.has(c10::DispatchKey::FuncTorchBatched) ||
      keys.has(c10::DispatchKey::FuncTorchGradWrapper) || keys.has(c10::DispatchKey::Functionalize))
    return nullptr;
  return &t;
}

bool modes_active() {
  return c10::impl::dispatch_mode_enabled() || at::impl::torch_function_mode_enabled();
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kHalf: return W8A8_F16;
    case at::kBFloat16: return W8A8_BF16;
    case at::kFloat: return W8A8_F32;
    default: return 0;
  }
}

void* stream_of(int device) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

template <typename T>
T* ptr(const at::Tensor& t) { return reinterpret_cast<T*>(t.data_ptr()); }

PyObject* fail(const char* fn, int rc) {
  PyObject* e = PyObject_CallFunction(g_error_class, "sis", fn, rc, w8a8_last_error());
  if (e) {
    PyErr_SetObject(g_error_class, e);
    Py_DECREF(e);
  }
  return nullptr;
}

// fn(&args) without the interpreter lock, as ctypes calls it.
template <typename Args>
int call(int (*fn)(const Args*), Args& a) {
  a.struct_size = sizeof(Args);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = fn(&a);
  Py_END_ALLOW_THREADS
  return rc;
}

// linear(x, weight, weight_scale, bias | None, epilogue, round_rotated,
// out_dtype): ConvRot256 and per-row INT8 of x [.., K], then the GEMM with the
// row- or column-order epilogue.
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7 || modes_active() || !THPDtype_Check(args[6])) Py_RETURN_NONE;
  const at::Tensor* x = plain(args[0]);
  const at::Tensor* w = plain(args[1]);
  const at::Tensor* ws = plain(args[2]);
  const at::Tensor* bias = args[3] == Py_None ? nullptr : plain(args[3]);
  if (!x || !w || !ws || (args[3] != Py_None && !bias)) Py_RETURN_NONE;
  const int dev = x->get_device();
  const long epilogue = PyLong_AsLong(args[4]), round_rotated = PyLong_AsLong(args[5]);
  const at::ScalarType out_type = reinterpret_cast<THPDtype*>(args[6])->scalar_type;
  const int xt = dtype_code(x->scalar_type()), ot = dtype_code(out_type);
  if (!xt || !ot || x->dim() < 1 || !x->is_contiguous() || w->dim() != 2 || w->scalar_type() != at::kChar ||
      !w->is_contiguous())
    Py_RETURN_NONE;
  const int64_t k = x->size(-1), nn = w->size(0);
  if (k <= 0 || k % 256 || w->size(1) != k || nn <= 0 || x->numel() == 0) Py_RETURN_NONE;
  const int64_t rows = x->numel() / k;
  if (ws->scalar_type() != at::kFloat || !ws->is_contiguous() || (ws->numel() != 1 && ws->numel() != nn))
    Py_RETURN_NONE;
  if (bias && ((bias->scalar_type() != at::kHalf && bias->scalar_type() != at::kFloat) || !bias->is_contiguous() ||
               bias->numel() != nn))
    Py_RETURN_NONE;
  const auto opt = at::TensorOptions().device(x->device());
  const at::Tensor q = at::empty({rows, k}, opt.dtype(at::kChar));
  const at::Tensor scale = at::empty({rows}, opt.dtype(at::kFloat));
  at::DimVector shape(x->sizes().begin(), x->sizes().end());
  shape.back() = nn;
  at::Tensor out = at::empty(shape, opt.dtype(out_type));
  void* const stream = stream_of(dev);

  W8A8QuantArgs qa{};
  qa.x_dtype = xt;
  qa.x = x->data_ptr();
  qa.ldx = k;
  qa.rows = rows;
  qa.cols = k;
  qa.convrot = 256;
  qa.round_rotated = round_rotated ? 1 : 0;
  qa.q = ptr<int8_t>(q);
  qa.ldq = k;
  qa.scale = ptr<float>(scale);
  qa.stream = stream;
  int rc = call(w8a8_quantize_rows, qa);
  if (rc != W8A8_OK) return fail("w8a8_quantize_rows", rc);

  W8A8GemmArgs ga{};
  ga.epilogue = (int32_t)epilogue;
  ga.a = qa.q;
  ga.lda = k;
  ga.b = ptr<int8_t>(*w);
  ga.ldb = k;
  ga.m = rows;
  ga.n = nn;
  ga.k = k;
  ga.row_scale = qa.scale;
  ga.col_scale = ptr<float>(*ws);
  ga.col_scale_stride = ws->numel() == 1 ? 0 : 1;
  if (bias) {
    ga.bias = bias->data_ptr();
    ga.bias_dtype = dtype_code(bias->scalar_type());
  }
  ga.out_dtype = ot;
  ga.out = out.data_ptr();
  ga.ldc = nn;
  at::Tensor workspace;
  ga.workspace_bytes = w8a8_gemm_workspace_size(rows, nn, k);
  if (ga.workspace_bytes > 0) {
    workspace = at::empty({ga.workspace_bytes}, opt.dtype(at::kByte));
    ga.workspace = workspace.data_ptr();
  }
  ga.stream = stream;
  rc = call(w8a8_gemm, ga);
  if (rc != W8A8_OK) return fail("w8a8_gemm", rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// Element strides {batch, head, token} of a [b, h, n, 128] tensor whose rows
// the kernels read in place; false: a copy is needed.
bool row_strides(const at::Tensor& t, int64_t (&st)[3]) {
  const int64_t es = t.element_size();
  if ((t.size(3) != 1 && t.stride(3) != 1) || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16) return false;
  for (int i = 0; i < 3; ++i) {
    st[i] = t.size(i) == 1 ? 0 : t.stride(i);
    if (st[i] < 0 || st[i] * es % 16) return false;
  }
  return true;
}

// int8_attention(q, k, v, sm_scale | None): the preparation and the attention
// of [b, h, n, 128] fp16 or fp32 tensors; the operands live in one buffer for
// the length of the call.
PyObject* int8_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4 || modes_active()) Py_RETURN_NONE;
  const at::Tensor* q = plain(args[0]);
  const at::Tensor* k = plain(args[1]);
  const at::Tensor* v = plain(args[2]);
  if (!q || !k || !v || q->dim() != 4 || k->dim() != 4 || v->dim() != 4) Py_RETURN_NONE;
  if (args[3] != Py_None && !PyFloat_CheckExact(args[3])) Py_RETURN_NONE;
  const at::ScalarType type = q->scalar_type();
  const int64_t b = q->size(0), h = q->size(1), nq = q->size(2), nk = k->size(2), d = 128;
  if ((type != at::kHalf && type != at::kFloat) || k->scalar_type() != type || v->scalar_type() != type ||
      q->size(3) != d || k->size(0) != b || k->size(1) != h || k->size(3) != d || v->sizes() != k->sizes() ||
      b * h == 0 || nq == 0 || nk == 0)
    Py_RETURN_NONE;
  W8A8AttnPrepareArgs pa{};
  if (!row_strides(*q, pa.q_strides) || !row_strides(*k, pa.k_strides) || !row_strides(*v, pa.v_strides)) Py_RETURN_NONE;
  const int64_t nblk = (nk + 127) / 128, nkp = 128 * nblk, bh = b * h;
  int64_t bytes = 0;
  auto take = [&](int64_t size) {
    const int64_t at = bytes;
    bytes += (size + 255) & ~int64_t(255);
    return at;
  };
  const int64_t wsb = w8a8_attention_workspace_size(b, h, nk);
  const int64_t o_q8 = take(bh * nq * d), o_qs = take(bh * nq * 4), o_k8 = take(bh * nkp * d), o_ks = take(bh * nblk * 16),
                o_vt = take(bh * nkp * d), o_vs = take(bh * d * 4), o_vsum = take(bh * nblk * d * 4), o_ws = take(wsb);
  const auto opt = at::TensorOptions().device(q->device());
  const at::Tensor buf = at::empty({bytes}, opt.dtype(at::kByte));
  at::Tensor out = at::empty({b, h, nq, d}, opt.dtype(type));
  char* const base = ptr<char>(buf);
  pa.in_dtype = dtype_code(type);
  pa.q = q->data_ptr();
  pa.k = k->data_ptr();
  pa.v = v->data_ptr();
  pa.b = b;
  pa.h = h;
  pa.nq = nq;
  pa.nk = nk;
  pa.d = (int32_t)d;
  pa.sm_scale = (float)(args[3] == Py_None ? std::pow((double)d, -0.5) : PyFloat_AS_DOUBLE(args[3]));
  pa.q8 = reinterpret_cast<int8_t*>(base + o_q8);
  pa.qs = reinterpret_cast<float*>(base + o_qs);
  pa.k8 = reinterpret_cast<int8_t*>(base + o_k8);
  pa.ks = reinterpret_cast<float*>(base + o_ks);
  pa.vt8 = reinterpret_cast<int8_t*>(base + o_vt);
  pa.vs = reinterpret_cast<float*>(base + o_vs);
  pa.vsum = reinterpret_cast<int32_t*>(base + o_vsum);
  pa.workspace = base + o_ws;
  pa.workspace_bytes = wsb;
  pa.stream = stream_of(q->get_device());
  int rc = call(w8a8_attention_prepare, pa);
  if (rc != W8A8_OK) return fail("w8a8_attention_prepare", rc);
  W8A8AttentionArgs aa{};
  aa.out_dtype = pa.in_dtype;
  aa.q8 = pa.q8;
  aa.qs = pa.qs;
  aa.k8 = pa.k8;
  aa.ks = pa.ks;
  aa.vt8 = pa.vt8;
  aa.vs = pa.vs;
  aa.vsum = pa.vsum;
  aa.b = b;
  aa.h = h;
  aa.nq = nq;
  aa.nk = nk;
  aa.d = (int32_t)d;
  aa.sm_scale = pa.sm_scale;
  aa.out = out.data_ptr();
  row_strides(out, aa.out_strides);
  aa.stream = pa.stream;
  rc = call(w8a8_attention, aa);
  if (rc != W8A8_OK) return fail("w8a8_attention", rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// segment_labels(rows, segments, table_rows, device_index): int32 [rows] with
// each row's table row, when the (a, b, row) segments tile [0, rows) exactly.
PyObject* segment_labels(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4 || modes_active() || !(PyList_CheckExact(args[1]) || PyTuple_CheckExact(args[1]))) Py_RETURN_NONE;
  const int64_t rows = PyLong_AsLongLong(args[0]), table_rows = PyLong_AsLongLong(args[2]);
  const long dev = PyLong_AsLong(args[3]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  if (rows <= 0 || rows >= (int64_t(1) << 31) || dev != c10::hip::current_device()) Py_RETURN_NONE;
  const Py_ssize_t count = PySequence_Fast_GET_SIZE(args[1]);
  std::vector<std::array<int64_t, 3>> segs((size_t)count);
  for (Py_ssize_t i = 0; i < count; ++i) {
    PyObject* s = PySequence_Fast_GET_ITEM(args[1], i);
    if (!(PyList_CheckExact(s) || PyTuple_CheckExact(s)) || PySequence_Fast_GET_SIZE(s) != 3) Py_RETURN_NONE;
    for (int j = 0; j < 3; ++j) {
      PyObject* v = PySequence_Fast_GET_ITEM(s, j);
      if (!PyLong_CheckExact(v)) Py_RETURN_NONE;
      int overflow = 0;
      segs[(size_t)i][(size_t)j] = PyLong_AsLongLongAndOverflow(v, &overflow);
      if (overflow) Py_RETURN_NONE;
    }
  }
  std::sort(segs.begin(), segs.end());
  std::vector<int32_t> ends, values;
  ends.reserve((size_t)count);
  values.reserve((size_t)count);
  int64_t cursor = 0;
  for (const auto& s : segs) {
    if (s[0] != cursor || s[1] <= s[0] || s[1] > rows || s[2] < 0 || s[2] >= table_rows || s[2] > INT32_MAX)
      Py_RETURN_NONE;
    cursor = s[1];
    ends.push_back((int32_t)s[1]);
    values.push_back((int32_t)s[2]);
  }
  if (cursor != rows) Py_RETURN_NONE;
  at::Tensor out = at::empty({rows}, at::TensorOptions().device(at::kCUDA, (c10::DeviceIndex)dev).dtype(at::kInt));
  void* const stream = stream_of((int)dev);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = w8a8_segment_labels(ends.data(), values.data(), (int64_t)ends.size(), ptr<int32_t>(out), rows, stream);
  Py_END_ALLOW_THREADS
  if (rc != W8A8_OK) return fail("w8a8_segment_labels", rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

PyObject* set_error_class(PyObject*, PyObject* cls) {
  Py_INCREF(cls);
  Py_XSETREF(g_error_class, cls);
  Py_RETURN_NONE;
}

template <typename F>
PyCFunction fast(F f) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }

}  // namespace

PyMODINIT_FUNC PyInit__native() {
  static PyMethodDef methods[] = {
      {"linear", fast(linear), METH_FASTCALL, nullptr},
      {"int8_attention", fast(int8_attention), METH_FASTCALL, nullptr},
      {"segment_labels", fast(segment_labels), METH_FASTCALL, nullptr},
      {"set_error_class", set_error_class, METH_O, nullptr},
      {nullptr, nullptr, 0, nullptr},
  };
  static PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};
  return PyModule_Create(&module);
}
