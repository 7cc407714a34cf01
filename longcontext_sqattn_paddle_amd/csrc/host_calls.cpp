// The short calls' way from Python to the C ABI: one native function per call that reads the tensors, allocates the
// output and the scratch and calls the library, in place of a dozen Python and ctypes steps.  Host side per call: decode over 1531 tokens
// 14.5 -> 8.2 us (of which two launches are 5), selection of 4096 tokens 10.7 -> 6.5, 777-token prefill 16.0 -> 9.3.
//
// Only plain arguments are taken (`plain`): torch tensors on a GPU, strided, not subclassed, wrapped, waiting for a gradient or
// carrying a forward-mode tangent, outside modes, transforms and traces, integers that are Python integers.  For anything else a
// function returns None before it has done anything, and the caller goes the general way (DLPack capsules, for `linear` torch's own),
// which accepts or refuses it as it always has.
// Returns the output (or a tuple), or the library's error code as an int.
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

#include "sqattn.h"

namespace {

// addresses in the loaded library (it is opened once, by _native.py)
struct Library {
  decltype(&sq_decode_num_splits) decode_num_splits;
  decltype(&sq_decode_workspace_bytes) decode_workspace_bytes;
  decltype(&sq_decode_fwd) decode_fwd;
  decltype(&sq_decode_selected_fwd) decode_selected_fwd;
  decltype(&sq_kmeans_workspace_bytes) kmeans_workspace_bytes;
  decltype(&sq_topk_select) topk_select;
  decltype(&sq_prefill_workspace_bytes_split) prefill_workspace_bytes_split;
  decltype(&sq_prefill_fwd) prefill_fwd;
  decltype(&sq_linear_preferred) linear_preferred;
  decltype(&sq_linear_workspace_bytes) linear_workspace_bytes;
  decltype(&sq_linear) linear;
} lib;

struct Arg : DLTensor {
  explicit Arg(const at::Tensor& t) {
    data = t.data_ptr();
    device.device_type = kDLROCM;
    device.device_id = t.device().index();
    ndim = (int32_t)t.dim();
    shape = const_cast<int64_t*>(t.sizes().data());
    strides = const_cast<int64_t*>(t.strides().data());
    byte_offset = 0;
    dtype.lanes = 1;
    dtype.bits = (uint8_t)(8 * t.element_size());
    switch (t.scalar_type()) {
      case at::kBFloat16: dtype.code = kDLBfloat; break;
      case at::kHalf: case at::kFloat: dtype.code = kDLFloat; break;
      case at::kByte: dtype.code = kDLUInt; break;
      default: dtype.code = kDLInt; break;   // `plain` lets no other type through
    }
  }
};

// a tensor that the general way would pass on as it is
bool plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.layout() != at::kStrided || !t.is_cuda() || t.requires_grad() || !t.has_storage()) return false;
  static const c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::Functionalize,
                                            c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                            c10::DispatchKey::Negative, c10::DispatchKey::Conjugate, c10::DispatchKey::ZeroTensor});
  if (t.key_set().has_any(wrapped)) return false;
  // a dual tensor shows neither in its type nor in its keys; without autograd metadata there is no tangent to ask for
  if (t.unsafeGetTensorImpl()->autograd_meta() && t._fw_grad(0).defined()) return false;
  switch (t.scalar_type()) {
    case at::kBFloat16: case at::kHalf: case at::kFloat: case at::kInt: case at::kByte: case at::kChar: return true;
    default: return false;
  }
}
bool plain_or_none(PyObject* o) { return o == Py_None || plain(o); }

// no mode and no recording trace that would want to see the allocations and the call
bool plain_context() {
  return !c10::impl::dispatch_mode_enabled() && !at::impl::torch_function_mode_enabled() &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Functionalize) && !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer);
}

bool is_int(PyObject* o) { return PyLong_CheckExact(o); }

// 4-dimensional rows of 128 contiguous elements
bool rows128(PyObject* o) {
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.dim() == 4 && t.size(3) == 128 && t.stride(3) == 1;
}

at::Tensor scratch(size_t bytes, c10::ScalarType type, const at::Tensor& like) {
  return at::empty({(int64_t)(bytes / c10::elementSize(type))}, like.options().dtype(type));
}

PyObject* result(const at::Tensor& o, const at::Tensor& lse) {
  if (!lse.defined()) return THPVariable_Wrap(o);
  PyObject* a = THPVariable_Wrap(o);
  PyObject* b = a ? THPVariable_Wrap(lse) : nullptr;
  PyObject* both = b ? PyTuple_Pack(2, a, b) : nullptr;
  Py_XDECREF(a);
  Py_XDECREF(b);
  return both;
}

// decode(q, k, v, token_ids, seqlens, layout, output_dtype, return_lse, p_quant, num_splits, workspace, out, stream)
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 13 || !plain_context()) Py_RETURN_NONE;
  if (!plain(a[0]) || !plain(a[1]) || !plain(a[2]) || !plain_or_none(a[3]) || !plain_or_none(a[4]) || !plain_or_none(a[10]) || !plain_or_none(a[11])) Py_RETURN_NONE;
  if (!rows128(a[0]) || !rows128(a[1]) || !rows128(a[2]) || !is_int(a[5]) || !THPDtype_Check(a[6]) || !PyBool_Check(a[7]) || !is_int(a[8]) || !is_int(a[9]) || !is_int(a[12])) Py_RETURN_NONE;
  const at::Tensor &q = THPVariable_Unpack(a[0]), &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]);
  const bool selected = a[3] != Py_None;
  if (selected && THPVariable_Unpack(a[3]).dim() != 2) Py_RETURN_NONE;
  const int hdim = PyLong_AsLong(a[5]) == SQ_LAYOUT_HND ? 1 : 2, ndim = 3 - hdim;
  const int64_t B = q.size(0), Hq = q.size(hdim), Hkv = k.size(hdim);
  const int64_t L = selected ? THPVariable_Unpack(a[3]).size(1) : k.size(ndim);
  const long named = PyLong_AsLong(a[9]);
  void* const stream = PyLong_AsVoidPtr(a[12]);
  sq_decode_params p = {};
  p.layout = (int32_t)PyLong_AsLong(a[5]);
  p.p_quant = (int32_t)PyLong_AsLong(a[8]);
  p.num_splits = named > 0 ? (int32_t)named : 0;
  p.head_dim_og = 128;
  if (PyErr_Occurred() || named > INT32_MAX) {   // a number of more than 32 bits: the general way says what it thinks of it
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  at::Tensor o, lse;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    at::Tensor ws = a[10] != Py_None ? THPVariable_Unpack(a[10])
                                     : scratch(lib.decode_workspace_bytes(B, Hq, 128, named > 0 ? (int32_t)named : lib.decode_num_splits(B, Hkv, L)), at::kFloat, q);
    o = a[11] != Py_None ? THPVariable_Unpack(a[11]) : at::empty(q.sizes(), q.options().dtype(reinterpret_cast<THPDtype*>(a[6])->scalar_type));
    if (a[7] == Py_True) lse = at::empty({B, Hq, 1}, q.options().dtype(at::kFloat));
    Arg dq(q), dk(k), dv(v), dout(o), dws(ws);
    c10::optional<Arg> ids, lens, dlse;
    if (selected) ids.emplace(THPVariable_Unpack(a[3]));
    if (a[4] != Py_None) lens.emplace(THPVariable_Unpack(a[4]));
    if (lse.defined()) dlse.emplace(lse);
    DLTensor *pl = lens ? &*lens : nullptr, *ps = dlse ? &*dlse : nullptr;
    rc = selected ? lib.decode_selected_fwd(&dq, &dk, &dv, &*ids, pl, &dout, ps, &dws, &p, stream) : lib.decode_fwd(&dq, &dk, &dv, pl, &dout, ps, &dws, &p, stream);
  }
  if (rc != SQ_OK) return PyLong_FromLong(rc);
  return result(o, lse);
  END_HANDLE_TH_ERRORS
}

// topk_select(query, centroids, clusters, cluster_size, k, num_kv_groups, out, workspace, stream)
PyObject* topk_select(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9 || !plain_context()) Py_RETURN_NONE;
  if (!plain(a[0]) || !plain(a[1]) || !plain(a[2]) || !plain(a[3]) || !is_int(a[4]) || !is_int(a[5]) || !plain_or_none(a[6]) || !plain_or_none(a[7]) || !is_int(a[8])) Py_RETURN_NONE;
  const at::Tensor &query = THPVariable_Unpack(a[0]), &cent = THPVariable_Unpack(a[1]);
  const long k = PyLong_AsLong(a[4]), groups = PyLong_AsLong(a[5]);
  void* const stream = PyLong_AsVoidPtr(a[8]);
  if (PyErr_Occurred() || k < 0 || groups < INT32_MIN || groups > INT32_MAX || cent.dim() != 3) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  at::Tensor o;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    o = a[6] != Py_None ? THPVariable_Unpack(a[6]) : at::empty({cent.size(0), (int64_t)k}, query.options().dtype(at::kInt));
    at::Tensor ws = a[7] != Py_None ? THPVariable_Unpack(a[7]) : scratch(lib.kmeans_workspace_bytes(cent.size(0), 1, cent.size(1), 128), at::kByte, query);
    Arg dq(query), dc(cent), dcl(THPVariable_Unpack(a[2])), dsz(THPVariable_Unpack(a[3])), dout(o), dws(ws);
    rc = lib.topk_select(&dq, &dc, &dcl, &dsz, &dout, &dws, (int32_t)groups, stream);
  }
  if (rc != SQ_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(o);
  END_HANDLE_TH_ERRORS
}

// prefill(q, k, v, layout, output_dtype, return_lse, p_quant, q_offset, workspace, out, stream): causal, no windows
PyObject* prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 11 || !plain_context()) Py_RETURN_NONE;
  if (!plain(a[0]) || !plain(a[1]) || !plain(a[2]) || !plain_or_none(a[8]) || !plain_or_none(a[9])) Py_RETURN_NONE;
  if (!rows128(a[0]) || !rows128(a[1]) || !rows128(a[2]) || !is_int(a[3]) || !THPDtype_Check(a[4]) || !PyBool_Check(a[5]) || !is_int(a[6]) || !is_int(a[7]) || !is_int(a[10])) Py_RETURN_NONE;
  const at::Tensor &q = THPVariable_Unpack(a[0]), &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]);
  sq_prefill_params p = {};
  const long layout = PyLong_AsLong(a[3]), p_quant = PyLong_AsLong(a[6]);
  p.layout = (int32_t)layout;
  p.p_quant = (int32_t)p_quant;
  p.head_dim_og = 128;
  p.q_offset = PyLong_AsLong(a[7]);
  p.window_mode = SQ_WINDOW_NONE;
  p.block_m = 128;
  void* const stream = PyLong_AsVoidPtr(a[10]);
  if (PyErr_Occurred() || p_quant < 0 || p_quant > INT32_MAX) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const int hdim = layout == SQ_LAYOUT_HND ? 1 : 2, ndim = 3 - hdim;
  const int64_t B = q.size(0), Hq = q.size(hdim), Nq = q.size(ndim), Hkv = k.size(hdim), Nk = k.size(ndim);
  at::Tensor o, lse;
  int rc;
  {
    pybind11::gil_scoped_release no_gil;
    o = a[9] != Py_None ? THPVariable_Unpack(a[9]) : at::empty(q.sizes(), q.options().dtype(reinterpret_cast<THPDtype*>(a[4])->scalar_type));
    if (a[5] == Py_True) lse = at::empty({B, Hq, Nq}, q.options().dtype(at::kFloat));
    at::Tensor ws = a[8] != Py_None ? THPVariable_Unpack(a[8]) : scratch(lib.prefill_workspace_bytes_split(B, Hq, Hkv, Nq, Nk, &p), at::kByte, q);
    Arg dq(q), dk(k), dv(v), dout(o), dws(ws);
    c10::optional<Arg> dlse;
    if (lse.defined()) dlse.emplace(lse);
    rc = lib.prefill_fwd(&dq, &dk, &dv, nullptr, nullptr, &dout, dlse ? &*dlse : nullptr, &dws, &p, stream);
  }
  if (rc != SQ_OK) return PyLong_FromLong(rc);
  return result(o, lse);
  END_HANDLE_TH_ERRORS
}

// linear(x, weight, bias, stream): None also where the BLAS library's product is the faster one, or the operands do not lie as
// sq_linear takes them
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4 || !plain_context() || !plain(a[0]) || !plain(a[1]) || !plain_or_none(a[2]) || !is_int(a[3])) Py_RETURN_NONE;
  const at::Tensor &x = THPVariable_Unpack(a[0]), &w = THPVariable_Unpack(a[1]);
  if (x.dim() < 1 || w.dim() != 2 || !x.is_contiguous() || !w.is_contiguous() || x.numel() == 0 || w.numel() == 0) Py_RETURN_NONE;
  const int64_t K = x.size(-1), M = x.numel() / K, N = w.size(0);
  const auto aligned = [](const at::Tensor& t) { return ((uintptr_t)t.data_ptr() & 15) == 0; };
  if (w.size(1) != K || !lib.linear_preferred(M, N, K) || !aligned(x) || !aligned(w) || x.device() != w.device() || x.scalar_type() != w.scalar_type() ||
      (x.scalar_type() != at::kBFloat16 && x.scalar_type() != at::kHalf) || x.numel() >= (int64_t)1 << 31 || w.numel() >= (int64_t)1 << 31)
    Py_RETURN_NONE;
  // torch's linear computes in the type autocast names
  if (at::autocast::is_autocast_enabled(at::kCUDA) && at::autocast::get_autocast_dtype(at::kCUDA) != x.scalar_type()) Py_RETURN_NONE;
  const bool biased = a[2] != Py_None;
  if (biased) {
    const at::Tensor& b = THPVariable_Unpack(a[2]);
    if (b.dim() != 1 || b.size(0) != N || !b.is_contiguous() || !aligned(b) || b.scalar_type() != x.scalar_type() || b.device() != x.device()) Py_RETURN_NONE;
  }
  void* const stream = PyLong_AsVoidPtr(a[3]);
  at::Tensor o;
  int rc;
  bool room = true;
  {
    pybind11::gil_scoped_release no_gil;
    std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = N;
    o = at::empty(shape, x.options());
    const size_t bytes = lib.linear_workspace_bytes(M, N, K);
    at::Tensor ws;
    try {
      if (bytes) ws = scratch(bytes, at::kByte, x);
    } catch (const c10::OutOfMemoryError&) {
      room = false;   // for the parts, which torch's linear does without
    }
    Arg dx(x), dw(w), dout(o);
    int64_t x_shape[2] = {M, K}, x_strides[2] = {K, 1}, o_shape[2] = {M, N}, o_strides[2] = {N, 1};
    dx.ndim = dout.ndim = 2;
    dx.shape = x_shape;
    dx.strides = x_strides;
    dout.shape = o_shape;
    dout.strides = o_strides;
    c10::optional<Arg> db, dws;
    if (biased) db.emplace(THPVariable_Unpack(a[2]));
    if (ws.defined()) dws.emplace(ws);
    rc = room ? lib.linear(&dx, &dw, db ? &*db : nullptr, &dout, dws ? &*dws : nullptr, stream) : SQ_OK;
  }
  if (!room) Py_RETURN_NONE;
  if (rc == SQ_EDEVICE) Py_RETURN_NONE;   // the operands' GPU is not the current one: refused before any launch, torch's linear changes over to it
  if (rc != SQ_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(o);
  END_HANDLE_TH_ERRORS
}

// bind(addresses): the library's functions, in the order of `Library`
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  constexpr Py_ssize_t kFunctions = sizeof(Library) / sizeof(void*);
  if (n != kFunctions) {
    PyErr_SetString(PyExc_TypeError, "bind takes one address per function");
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < n; ++i) {
    void* p = PyLong_AsVoidPtr(a[i]);
    if (!p) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null address");
      return nullptr;
    }
    memcpy((char*)&lib + i * sizeof(void*), &p, sizeof(void*));
  }
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
    {"decode", (PyCFunction)(void (*)(void))decode, METH_FASTCALL, nullptr},
    {"topk_select", (PyCFunction)(void (*)(void))topk_select, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void (*)(void))linear, METH_FASTCALL, nullptr},
    {"prefill", (PyCFunction)(void (*)(void))prefill, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// torch_version: of the headers this was compiled against; the layout of a tensor is that version's
PyMODINIT_FUNC PyInit__host_calls(void) {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", SQ_TORCH_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
