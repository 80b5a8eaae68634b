// The host side of the row and rotary ops in native code: the checks, the outputs and the launches of one call.
//
// What such a pass costs is the host's work: the rotary op forward and backward on 16 tokens took 135 us of Python, where the
// kernels of 14336 tokens take 58, and takes 70 to 83 this way; permute and unpermute of 14593 tokens forward and backward took
// 140 and take 100, which is what their kernels take.  Each function here takes the call as the op got it, and either makes it whole --
// allocates, launches, returns the outputs -- or returns None and has touched nothing: anything but plain CUDA tensors of one device
// with the shapes, types and strides that the kernels read in place (a subclass, a transform's wrapper, a tensor that would
// first be copied or moved, anything to be refused) is the general path's, in native.py, which warns, copies and raises.
// No state is kept between calls.  The library's entry points come in through bind(), from the library that _lib.py loaded.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstring>
#include <string>
#include <type_traits>

#include "wallx_mi355.h"

namespace {

struct Entry {
  decltype(&wx_last_error_string) last_error;
  decltype(&wx_mrope_apply) rope;
  decltype(&wx_mrope_apply_bwd) rope_bwd;
  decltype(&wx_mrope_apply_positions) rope_positions;
  decltype(&wx_mrope_apply_packed) rope_packed;
  decltype(&wx_mrope_table_width) table_width;
  decltype(&wx_partition_workspace_bytes) partition_bytes;
  decltype(&wx_partition_build) partition;
  decltype(&wx_permute_rows) permute;
  decltype(&wx_unpermute_rows) unpermute;
  decltype(&wx_unpermute_rows_bwd_clear) unpermute_bwd;
} entry;
const char* const kNames[] = {"wx_last_error_string", "wx_mrope_apply", "wx_mrope_apply_bwd", "wx_mrope_apply_positions",
                              "wx_mrope_apply_packed", "wx_mrope_table_width", "wx_partition_workspace_bytes", "wx_partition_build",
                              "wx_permute_rows", "wx_unpermute_rows", "wx_unpermute_rows_bwd_clear"};
constexpr int kEntries = sizeof(kNames) / sizeof(kNames[0]);
static_assert(sizeof(Entry) == kEntries * sizeof(void*), "a name per entry point");

// A tensor that is what it looks like: strided CUDA memory, no wrapper, no pending conjugation or negation -- and, as what is
// allocated inside a transform is a wrapper whatever the inputs are, outside of all transforms.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  for (const c10::DispatchKey transform : {c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::Functionalize})
    if (c10::impl::tls_is_dispatch_key_included(transform)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.is_conj() || t.is_neg()) return nullptr;
  constexpr c10::DispatchKeySet wrappers({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
                                          c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                          c10::DispatchKey::ZeroTensor, c10::DispatchKey::Batched});
  if (t.key_set().has_any(wrappers) || !t.has_storage()) return nullptr;
  return &t;
}

int dtype_code(at::ScalarType t) {
  return t == at::kFloat ? WX_F32 : t == at::kHalf ? WX_F16 : t == at::kBFloat16 ? WX_BF16 : -1;
}

void* ptr(const at::Tensor& t) { return t.numel() == 0 ? nullptr : t.data_ptr(); }

wx_stream_t stream_of(const at::Tensor& t) { return reinterpret_cast<wx_stream_t>(c10::hip::getCurrentHIPStream(t.get_device()).stream()); }

// Runs `f` without the interpreter lock (a launch waits where the queue is full) and with the device of `t` current; the
// library's statuses become Python errors here, C++ exceptions (an allocation that fails) in the functions' own frames.
template <typename F>
bool run(const at::Tensor& t, F f) {
  int rc = 0;
  std::string error;
  {
    const pybind11::gil_scoped_release no_gil;
    const c10::DeviceGuard guard(t.device());
    rc = f();
    if (rc != 0) error = entry.last_error();
  }
  if (rc != 0) PyErr_Format(PyExc_RuntimeError, "wallx_mi355: %s (status %d)", error.c_str(), rc);
  return rc == 0;
}

bool to_int(PyObject* o, int64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}

bool section_of(PyObject* o, int sec[3]) {
  if (!PyList_CheckExact(o) && !PyTuple_CheckExact(o)) return false;
  if (PySequence_Fast_GET_SIZE(o) != 3) return false;
  for (int i = 0; i < 3; ++i) {
    int64_t v;
    if (!to_int(PySequence_Fast_GET_ITEM(o, i), v) || v < 0 || v > 1024) return false;
    sec[i] = static_cast<int>(v);
  }
  return true;
}

bool layout_of(PyObject* o, int& layout) {
  if (!PyUnicode_CheckExact(o)) return false;
  if (PyUnicode_CompareWithASCIIString(o, "hf") == 0) layout = WX_MROPE_HF;
  else if (PyUnicode_CompareWithASCIIString(o, "csrc") == 0) layout = WX_MROPE_CSRC;
  else return false;
  return true;
}

PyObject* none() { Py_RETURN_NONE; }

PyObject* wrap(const at::Tensor& t) { return THPVariable_Wrap(t); }

PyObject* pair(const at::Tensor& a, const at::Tensor& b) {
  PyObject* const x = wrap(a);
  PyObject* const y = x ? wrap(b) : nullptr;
  PyObject* const r = y ? PyTuple_Pack(2, x, y) : nullptr;
  Py_XDECREF(x);
  Py_XDECREF(y);
  return r;
}

// rope(form, q, k, a, b, section, layout, backward) -> (q_out, k_out) or None.
// form 0: a, b = cos, sin [3, B, S, D]; 1: a, b = position_ids [3, B, S], inv_freq [D / 2]; 2: a = the packed table, b = None.
PyObject* rope(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t form, backward;
  int sec[3], layout;
  if (n != 8 || !entry.rope || !to_int(args[0], form) || !to_int(args[7], backward) || !section_of(args[5], sec) || !layout_of(args[6], layout)) return none();
  const at::Tensor *q = plain(args[1]), *k = plain(args[2]), *a = plain(args[3]), *b = form == 2 ? a : plain(args[4]);
  if (!q || !k || !a || !b || q->dim() != 4 || k->dim() != 4) return none();
  const int64_t B = q->size(0), Hq = q->size(1), S = q->size(2), D = q->size(3), Hk = k->size(1);
  if (k->size(0) != B || k->size(2) != S || k->size(3) != D || q->stride(3) != 1 || k->stride(3) != 1) return none();
  if (Hq > INT32_MAX || Hk > INT32_MAX || D > INT32_MAX) return none();
  const at::ScalarType dt = q->scalar_type();
  const int code = dtype_code(dt);
  if (code < 0 || k->scalar_type() != dt || k->device() != q->device() || a->device() != q->device() || b->device() != q->device()) return none();
  if (!a->is_contiguous() || !b->is_contiguous()) return none();
  if (form == 0) {
    for (const at::Tensor* t : {a, b})
      if (t->dim() != 4 || t->size(0) != 3 || t->size(1) != B || t->size(2) != S || t->size(3) != D || t->scalar_type() != dt) return none();
  } else if (form == 1) {
    if (a->dim() != 3 || a->size(0) != 3 || a->size(1) != B || a->size(2) != S || a->scalar_type() != at::kLong) return none();
    if (b->dim() != 1 || b->size(0) != D / 2 || b->scalar_type() != at::kFloat) return none();
  } else if (form == 2) {
    const int width = entry.table_width(static_cast<int>(D), sec, layout);
    if (width < 0 || a->dim() != 2 || a->size(0) != B * S || a->size(1) != width || a->scalar_type() != at::kInt || dt != at::kBFloat16) return none();
  } else {
    return none();
  }
  at::Tensor qo, ko;
  const bool ok = run(*q, [&] {
    qo = at::empty(q->sizes(), q->options());
    ko = at::empty(k->sizes(), k->options());
    const int64_t sq[3] = {q->stride(0), q->stride(1), q->stride(2)}, sk[3] = {k->stride(0), k->stride(1), k->stride(2)};
    const int64_t so[3] = {qo.stride(0), qo.stride(1), qo.stride(2)}, st[3] = {ko.stride(0), ko.stride(1), ko.stride(2)};
    const int hq = static_cast<int>(Hq), hk = static_cast<int>(Hk), d = static_cast<int>(D);
    const wx_stream_t stream = stream_of(*q);
    if (form == 0)
      return (backward ? entry.rope_bwd : entry.rope)(ptr(*q), ptr(*k), ptr(*a), ptr(*b), ptr(qo), ptr(ko), B, S, hq, hk, d, sq, sk, so, st, sec, layout, code, stream);
    if (form == 1)
      return entry.rope_positions(ptr(*q), ptr(*k), static_cast<const int64_t*>(ptr(*a)), static_cast<const float*>(ptr(*b)), ptr(qo), ptr(ko), B, S, hq, hk, d,
                                  sq, sk, so, st, sec, layout, code, backward != 0, stream);
    return entry.rope_packed(ptr(*q), ptr(*k), static_cast<const uint32_t*>(ptr(*a)), ptr(qo), ptr(ko), B, S, hq, hk, d, sq, sk, so, st, sec, layout, code,
                             backward != 0, stream);
  });
  return ok ? pair(qo, ko) : nullptr;
  END_HANDLE_TH_ERRORS
}

// permute(input [T, H], indices int32 [T, K], num_out_tokens, histograms, status, experts) -> (permuted, row_id_map) or None.
// The scratch is the caller's, and large enough (else the general path makes another), or with None this call's own; no status
// word with None.
PyObject* permute(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t num_out, experts;
  if (n != 6 || !entry.partition || !to_int(args[2], num_out) || !to_int(args[5], experts)) return none();
  const at::Tensor *x = plain(args[0]), *ids = plain(args[1]), *hist = args[3] == Py_None ? nullptr : plain(args[3]),
                   *status = args[4] == Py_None ? nullptr : plain(args[4]);
  if (!x || !ids || (args[3] != Py_None && !hist) || (args[4] != Py_None && !status)) return none();
  if (x->dim() != 2 || ids->dim() != 2 || !x->is_contiguous() || !ids->is_contiguous()) return none();
  const int64_t T = ids->size(0), K = ids->size(1), H = x->size(1);
  const int code = dtype_code(x->scalar_type());
  if (code < 0 || ids->scalar_type() != at::kInt || x->size(0) != T || T <= 0 || K <= 0 || K > 128 || H <= 0 || num_out < 0) return none();
  for (const at::Tensor* t : {ids, hist, status})
    if (t && t->device() != x->device()) return none();
  const int64_t need = static_cast<int64_t>(entry.partition_bytes(T * K));
  if ((hist && (!hist->is_contiguous() || hist->numel() * hist->element_size() < need)) || (status && status->numel() < 1)) return none();
  at::Tensor out, map;
  const bool ok = run(*x, [&] {
    const at::TensorOptions i32 = ids->options();
    map = at::empty({T * K}, i32);
    at::Tensor offsets = at::empty({experts + 1}, i32);
    out = at::empty({num_out > 0 ? num_out : T * K, H}, x->options());
    const at::Tensor scratch = hist ? *hist : at::empty({need}, x->options().dtype(at::kByte));
    const wx_stream_t stream = stream_of(*x);
    const int rc = entry.partition(ptr(*ids), WX_I32, T, static_cast<int>(K), static_cast<int>(experts), num_out, static_cast<int32_t*>(ptr(map)), nullptr,
                                   static_cast<int32_t*>(offsets.data_ptr()), status ? static_cast<int32_t*>(status->data_ptr()) : nullptr, ptr(scratch),
                                   static_cast<size_t>(scratch.numel()) * scratch.element_size(), stream);
    return rc != 0 ? rc : entry.permute(ptr(*x), ptr(out), static_cast<const int32_t*>(ptr(map)), T, static_cast<int>(K), H, code, stream);
  });
  return ok ? pair(out, map) : nullptr;
  END_HANDLE_TH_ERRORS
}

// unpermute(input, row_id_map int32, probs fp32 [T, K] or None, T, K) -> output [T, H] or None.
PyObject* unpermute(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t T, K;
  if (n != 5 || !entry.unpermute || !to_int(args[3], T) || !to_int(args[4], K)) return none();
  const at::Tensor *x = plain(args[0]), *map = plain(args[1]), *probs = args[2] == Py_None ? nullptr : plain(args[2]);
  if (!x || !map || (args[2] != Py_None && !probs) || x->dim() != 2 || !x->is_contiguous() || !map->is_contiguous()) return none();
  const int code = dtype_code(x->scalar_type());
  if (code < 0 || T <= 0 || K <= 0 || K > 128 || map->scalar_type() != at::kInt || map->numel() < T * K || map->device() != x->device()) return none();
  if (probs && (!probs->is_contiguous() || probs->scalar_type() != at::kFloat || probs->device() != x->device() || probs->numel() == 0)) return none();
  at::Tensor out;
  const bool ok = run(*x, [&] {
    out = at::empty({T, x->size(1)}, x->options());
    return entry.unpermute(ptr(*x), ptr(out), static_cast<const int32_t*>(ptr(*map)), probs && K > 1 ? static_cast<const float*>(ptr(*probs)) : nullptr, T,
                           static_cast<int>(K), x->size(1), code, stream_of(*x));
  });
  return ok ? wrap(out) : nullptr;
  END_HANDLE_TH_ERRORS
}

// unpermute_bwd(grad [T, H], input_fwd [R, H], row_id_map int32, probs fp32 [T, K] or None) -> act_grad [R, H], or with probs
// (act_grad, their gradient [T, K]), or None.  Without probs: one expert per token.  (A single weight per token, whose
// gradient is zeros, is the general path's.)
PyObject* unpermute_bwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4 || !entry.unpermute_bwd) return none();
  const at::Tensor *g = plain(args[0]), *x = plain(args[1]), *map = plain(args[2]), *probs = args[3] == Py_None ? nullptr : plain(args[3]);
  if (!g || !x || !map || (args[3] != Py_None && !probs) || g->dim() != 2 || x->dim() != 2 || !g->is_contiguous() || !x->is_contiguous() ||
      !map->is_contiguous())
    return none();
  const int64_t T = g->size(0), K = probs ? (probs->dim() == 2 ? probs->size(1) : 0) : 1;
  if (probs && (K < 2 || K > 128 || probs->size(0) != T || !probs->is_contiguous() || probs->scalar_type() != at::kFloat || probs->device() != g->device()))
    return none();
  const int code = dtype_code(g->scalar_type());
  if (code < 0 || x->scalar_type() != g->scalar_type() || map->scalar_type() != at::kInt || x->size(1) != g->size(1) || g->numel() == 0 || x->numel() == 0 ||
      map->numel() < T * K || x->device() != g->device() || map->device() != g->device())
    return none();
  at::Tensor out, prob_grad;
  const bool ok = run(*g, [&] {
    out = at::empty({x->size(0), g->size(1)}, g->options());
    if (probs) prob_grad = at::empty({T, K}, probs->options());
    return entry.unpermute_bwd(ptr(*g), ptr(*x), ptr(out), out.size(0), probs ? static_cast<float*>(ptr(prob_grad)) : nullptr,
                               static_cast<const int32_t*>(ptr(*map)), probs ? static_cast<const float*>(ptr(*probs)) : nullptr, T, static_cast<int>(K),
                               g->size(1), code, stream_of(*g));
  });
  return !ok ? nullptr : (probs ? pair(out, prob_grad) : wrap(out));
  END_HANDLE_TH_ERRORS
}

// names() -> the entry points in the order bind() takes their addresses in.
PyObject* names(PyObject*, PyObject*) {
  PyObject* const r = PyTuple_New(kEntries);
  for (int i = 0; r && i < kEntries; ++i) PyTuple_SET_ITEM(r, i, PyUnicode_FromString(kNames[i]));
  return r;
}

PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != kEntries) return PyErr_Format(PyExc_TypeError, "bind takes %d addresses", kEntries);
  void* at[kEntries];
  for (int i = 0; i < kEntries; ++i) {
    at[i] = PyLong_AsVoidPtr(args[i]);
    if (!at[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
      return nullptr;
    }
  }
  static_assert(std::is_trivially_copyable_v<Entry>);
  memcpy(&entry, at, sizeof(entry));
  return none();
}

#define WX_FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(f)), METH_FASTCALL
PyMethodDef methods[] = {{"rope", WX_FAST(rope), nullptr},
                         {"permute", WX_FAST(permute), nullptr},
                         {"unpermute", WX_FAST(unpermute), nullptr},
                         {"unpermute_bwd", WX_FAST(unpermute_bwd), nullptr},
                         {"bind", WX_FAST(bind), nullptr},
                         {"names", names, METH_NOARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_wallx_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__wallx_host() { return PyModule_Create(&module); }
