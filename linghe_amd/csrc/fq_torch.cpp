// The outputs and the launch of the row-wise quantisers in one native call.
//
// A decode step's kernels run 2.2-3.7 us each, and a Python wrapper that allocates its two to five outputs
// with torch.empty and calls the library through ctypes takes 12 us: what bounds a small call is the host.
// The wrappers keep their checks in Python and hand over here; allocation goes through the dispatcher as
// torch.empty does (same allocator, pools and modes) and the interpreter lock is released meanwhile.
// The kernel library is the one that _lib.py loaded: bind() takes its functions' addresses, there is no
// link-time dependency that could bring a second one into the process.
// RMSNorm + group + SwiGLU quantiser, three calls: 36.8 -> 21.7 us on 32 rows of 2048, 36.8 -> 23.9 on 3001 of 4096.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <pybind11/pybind11.h>

#include "../../include/fq_api.h"

namespace {

struct {
  decltype(&fq_rmsnorm_quant_fwd) rmsnorm_quant_fwd = nullptr;
  decltype(&fq_swiglu_quant_fwd) swiglu_quant_fwd = nullptr;
  decltype(&fq_group_quant) group_quant = nullptr;
  decltype(&fq_last_error) last_error = nullptr;
} lib;

at::ScalarType dtype_of(PyObject* o) {
  TORCH_CHECK(THPDtype_Check(o), "expected a torch.dtype");
  return reinterpret_cast<THPDtype*>(o)->scalar_type;
}

int64_t int_of(PyObject* o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}

void* stream_of(PyObject* o) { return reinterpret_cast<void*>(static_cast<intptr_t>(int_of(o))); }

// the tensor behind an argument; undefined for None
at::Tensor tensor_or_none(PyObject* o) {
  if (o == Py_None) return {};
  TORCH_CHECK(THPVariable_Check(o), "expected a tensor or None");
  return THPVariable_Unpack(o);
}

at::Tensor empty(const at::Tensor& like, at::ScalarType type, at::IntArrayRef sizes) {
  return at::empty(sizes, at::TensorOptions().dtype(type).device(like.device()));
}

void* data(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

void check(int rc) {
  TORCH_CHECK(rc == 0, "libfq_gfx950 error ", rc, ": ", lib.last_error());
}

void need_args(Py_ssize_t n, Py_ssize_t want) { TORCH_CHECK(n == want, "expected ", want, " arguments, got ", n); }

void need_lib() { TORCH_CHECK(lib.last_error, "bind() was not called"); }

template <typename F>
F function_at(PyObject* o) {
  const int64_t address = int_of(o);
  TORCH_CHECK(address != 0, "a function's address is 0");
  return reinterpret_cast<F>(static_cast<intptr_t>(address));
}

// (fq_rmsnorm_quant_fwd, fq_swiglu_quant_fwd, fq_group_quant, fq_last_error): addresses in the loaded library
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  need_args(n_args, 4);
  lib = {function_at<decltype(&fq_rmsnorm_quant_fwd)>(a[0]), function_at<decltype(&fq_swiglu_quant_fwd)>(a[1]),
         function_at<decltype(&fq_group_quant)>(a[2]), function_at<decltype(&fq_last_error)>(a[3])};
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// the outputs as a tuple, None for an undefined one
PyObject* wrap(const std::initializer_list<at::Tensor>& outs) {
  PyObject* tuple = PyTuple_New(static_cast<Py_ssize_t>(outs.size()));
  if (!tuple) throw python_error();
  Py_ssize_t i = 0;
  for (const at::Tensor& t : outs) {
    PyObject* item = t.defined() ? THPVariable_Wrap(t) : Py_NewRef(Py_None);
    if (!item) {
      Py_DECREF(tuple);
      throw python_error();
    }
    PyTuple_SET_ITEM(tuple, i++, item);
  }
  return tuple;
}

// (x, gamma, out, scale, rms, eps, round_scale, output_mode, fp8 dtype, kind, stream): out, scale and rms are
// allocated where None is given and the mode writes them
PyObject* rmsnorm_quant(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  need_args(n_args, 11);
  need_lib();
  const at::Tensor x = tensor_or_none(a[0]), gamma = tensor_or_none(a[1]);
  at::Tensor out = tensor_or_none(a[2]), scale = tensor_or_none(a[3]), rms = tensor_or_none(a[4]), qt, st;
  const double eps = PyFloat_AsDouble(a[5]);
  if (eps == -1.0 && PyErr_Occurred()) throw python_error();
  const int round = static_cast<int>(int_of(a[6])), mode = static_cast<int>(int_of(a[7]));
  const at::ScalarType fp8 = dtype_of(a[8]);
  const int kind = static_cast<int>(int_of(a[9]));
  void* stream = stream_of(a[10]);
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), n = x.size(1);
    if (mode != 1) {
      if (!out.defined()) out = empty(x, fp8, {M, n});
      if (!scale.defined()) scale = empty(x, at::kFloat, {n / 128, M});
    }
    qt = empty(x, fp8, {n, M});
    st = empty(x, at::kFloat, {(M + 127) / 128, n});
    if (!rms.defined()) rms = empty(x, at::kFloat, {M});
    if (M > 0)
      check(lib.rmsnorm_quant_fwd(data(x), data(gamma), mode != 1 ? data(out) : nullptr,
                                  static_cast<float*>(mode != 1 ? data(scale) : nullptr),
                                  static_cast<float*>(data(rms)), data(qt), static_cast<float*>(data(st)), M, n,
                                  static_cast<float>(eps), round, mode, kind, stream));
  }
  return wrap({out, scale, rms, qt, st});
  END_HANDLE_TH_ERRORS
}

// (x, out, scale, round_scale, output_mode, fp8 dtype, kind, stream)
PyObject* swiglu_quant(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  need_args(n_args, 8);
  need_lib();
  const at::Tensor x = tensor_or_none(a[0]);
  at::Tensor out = tensor_or_none(a[1]), scale = tensor_or_none(a[2]), qt, st;
  const int round = static_cast<int>(int_of(a[3])), mode = static_cast<int>(int_of(a[4]));
  const at::ScalarType fp8 = dtype_of(a[5]);
  const int kind = static_cast<int>(int_of(a[6]));
  void* stream = stream_of(a[7]);
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), n = x.size(1) / 2;
    if (!out.defined()) out = empty(x, fp8, {M, n});
    if (!scale.defined()) scale = empty(x, at::kFloat, {n / 128, M});
    qt = empty(x, fp8, {n, M});
    st = empty(x, at::kFloat, {(M + 127) / 128, n});
    if (M > 0)
      check(lib.swiglu_quant_fwd(data(x), data(out), static_cast<float*>(data(scale)), data(qt),
                                 static_cast<float*>(data(st)), M, n, round, mode, kind, stream));
  }
  return wrap({out, scale, qt, st});
  END_HANDLE_TH_ERRORS
}

// (x, round_scale, fp8 dtype, kind, stream)
PyObject* group_quant(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  need_args(n_args, 5);
  need_lib();
  const at::Tensor x = tensor_or_none(a[0]);
  at::Tensor q, s;
  const int round = static_cast<int>(int_of(a[1]));
  const at::ScalarType fp8 = dtype_of(a[2]);
  const int kind = static_cast<int>(int_of(a[3]));
  void* stream = stream_of(a[4]);
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), n = x.size(1);
    q = empty(x, fp8, {M, n});
    s = empty(x, at::kFloat, {M, n / 128});
    if (M > 0) check(lib.group_quant(data(x), data(q), static_cast<float*>(data(s)), M, n, round, kind, stream));
  }
  return wrap({q, s});
  END_HANDLE_TH_ERRORS
}

#define FQ_FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(f))
PyMethodDef methods[] = {{"bind", FQ_FAST(bind), METH_FASTCALL, nullptr},
                         {"rmsnorm_quant", FQ_FAST(rmsnorm_quant), METH_FASTCALL, nullptr},
                         {"swiglu_quant", FQ_FAST(swiglu_quant), METH_FASTCALL, nullptr},
                         {"group_quant", FQ_FAST(group_quant), METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fq_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" PyObject* PyInit__fq_torch() { return PyModule_Create(&module); }
