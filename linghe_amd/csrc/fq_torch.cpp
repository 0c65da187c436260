// The outputs and the launch of an entry point in one native call.
//
// A small call's kernels run 2-5 us each, and a Python wrapper that allocates its two to seven outputs with torch.empty
// and calls the library through ctypes takes 7-13 us (more where it adds up the tokens of 256 experts): what bounds a
// small call is the host. The wrappers keep their checks in Python and hand over here; the device is made current here, the outputs
// come from torch's allocator (Outputs) and the interpreter lock is released meanwhile.
// The kernel library is the one that _lib.py loaded: bind() takes its functions' addresses, there is no
// link-time dependency that could bring a second one into the process.
// us through ctypes / here with outputs through the dispatcher and the device guard in Python / now, back to back: RMSNorm + group +
// SwiGLU quantiser on 32 rows of 2048 36.8 / 19.4 / 15.5; activation 528 x 3456 and weight of a linear layer - / 12.4 / 9.8;
// RMSNorm + quant 624 x 1024 - / 10.7 / 8.7; row-wise and then transposed 384 x 1536 - / 14.2 / 11.2; bf16 RMSNorm and SwiGLU,
// forward and backward, 640 x 1024 / 768 - / 28.8 / 23.7; gather + pad + quant and per-expert quant, 486 tokens to 2 of 128
// experts, - / 18.7 / 16.8 (the kernels' time). One call: group quantiser 6.6 / 5.2, a tile plan of 64 experts 7.8 (ctypes) / 4.8.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <ATen/EmptyTensor.h>
#include <ATen/detail/CUDAHooksInterface.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <pybind11/pybind11.h>

#include <algorithm>
#include <iterator>
#include <vector>

#include "../../include/fq_api.h"

namespace {

// the library's functions that are called here
#define FQ_FUNCTIONS(F)                                                                                              \
  F(rmsnorm_fwd) F(rmsnorm_bwd) F(rmsnorm_bwd_num_partials) F(rmsnorm_quant_fwd) F(rmsnorm_router_quant_fwd)         \
  F(rmsnorm_router_quant_fwd_packed) F(rmsnorm_router_quant_fwd_folded) F(swiglu_fwd) F(swiglu_bwd)                  \
  F(rmsnorm_router_slices) F(rmsnorm_router_folds) F(rmsnorm_router_scratch_bytes)                                   \
  F(rmsnorm_router_folded_scratch_bytes)                                                                             \
  F(swiglu_quant_fwd) F(swiglu_quant_bwd)                                                                            \
  F(batched_swiglu_quant_fwd) F(batched_swiglu_quant_fwd_planned) F(batched_swiglu_quant_bwd)                        \
  F(batched_swiglu_quant_bwd_planned) F(group_quant) F(block_quant) F(blockwise_quant) F(batched_blockwise_quant)    \
  F(batched_blockwise_quant_planned) F(batched_pad_permute_quant) F(batched_pad_permute_quant_planned)               \
  F(expert_plan_shape) F(expert_plan_bytes) F(build_expert_plan) F(last_error)

struct {
#define FQ_MEMBER(name) decltype(&fq_##name) name = nullptr;
  FQ_FUNCTIONS(FQ_MEMBER)
#undef FQ_MEMBER
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

// the tensor behind an argument; undefined for None
at::Tensor tensor_or_none(PyObject* o) {
  if (o == Py_None) return {};
  TORCH_CHECK(THPVariable_Check(o), "expected a tensor or None");
  return THPVariable_Unpack(o);
}

// The device of a call's first tensor made the current one, and tensors on it. They are made as at::empty makes them behind
// the dispatcher (0.65 us of a call for each output, 0.25 without it), unless something could be listening there: a mode, a
// transform, a tracer, an observer of operators (a profiler), or the fill of new memory that deterministic algorithms ask for.
class Outputs {
 public:
  explicit Outputs(const at::Tensor& x)
      : on_(x.device()),
        device_(x.device()),
        plain_(x.is_cuda() && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
               (c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty() &&
               !at::hasCallbacks() && !at::globalContext().deterministicAlgorithms()) {}

  at::Tensor empty(const at::Tensor& like, at::ScalarType type, at::IntArrayRef sizes) const {
    if (!plain_ || like.device() != device_)
      return at::empty(sizes, at::TensorOptions().dtype(type).device(like.device()));
    return at::detail::empty_generic(sizes, at::detail::getCUDAHooks().getCUDADeviceAllocator(),
                                     c10::DispatchKeySet(c10::DispatchKey::CUDA), type, std::nullopt);
  }

  // of the type, sizes and strides of t
  at::Tensor empty_like(const at::Tensor& t) const {
    int64_t stride = 1;
    for (int64_t d = t.dim() - 1; d >= 0; --d) {  // (a contiguous tensor may have any stride where its size is 1)
      if (t.stride(d) != stride) return at::empty_like(t);
      stride *= std::max<int64_t>(t.size(d), 1);
    }
    return empty(t, t.scalar_type(), t.sizes());
  }

 private:
  c10::DeviceGuard on_;
  c10::Device device_;
  bool plain_;
};

void* data(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

void check(int rc) {
  TORCH_CHECK(rc == 0, "libfq_gfx950 error ", rc, ": ", lib.last_error());
}

float* floats(const at::Tensor& t) { return static_cast<float*>(data(t)); }

// the numbers of an iterable, each through int(); of a size that sums of a million of them cannot overflow
std::vector<int64_t> ints_of(PyObject* o) {
  const auto items = pybind11::reinterpret_steal<pybind11::object>(PySequence_Tuple(o));
  if (!items) throw python_error();
  std::vector<int64_t> values(static_cast<size_t>(PyTuple_GET_SIZE(items.ptr())));
  for (size_t i = 0; i < values.size(); ++i) {
    PyObject* item = PyTuple_GET_ITEM(items.ptr(), static_cast<Py_ssize_t>(i));
    if (PyLong_CheckExact(item)) {
      values[i] = int_of(item);
    } else {
      const auto number = pybind11::reinterpret_steal<pybind11::object>(PyNumber_Long(item));
      if (!number) throw python_error();
      values[i] = int_of(number.ptr());
    }
    constexpr int64_t kLimit = int64_t{1} << 40;
    TORCH_CHECK(-kLimit < values[i] && values[i] < kLimit, values[i], " rows of one expert");
  }
  return values;
}

// the arguments of a call, one after the other
class Args {
 public:
  Args(PyObject* const* a, Py_ssize_t n, Py_ssize_t want) : a_(a) {
    TORCH_CHECK(n == want, "expected ", want, " arguments, got ", n);
    TORCH_CHECK(lib.last_error, "bind() was not called");
  }
  at::Tensor tensor() { return tensor_or_none(*a_++); }
  int64_t integer() { return int_of(*a_++); }
  int flag() { return static_cast<int>(integer()); }
  std::vector<int64_t> integers() { return ints_of(*a_++); }
  void* address() { return reinterpret_cast<void*>(static_cast<intptr_t>(integer())); }
  at::ScalarType dtype() { return dtype_of(*a_++); }
  float real() {
    const double v = PyFloat_AsDouble(*a_++);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return static_cast<float>(v);
  }

 private:
  PyObject* const* a_;
};

template <typename F>
void set_function(F& f, PyObject* o) {
  const int64_t address = int_of(o);
  TORCH_CHECK(address != 0, "a function's address is 0");
  f = reinterpret_cast<F>(static_cast<intptr_t>(address));
}

// the addresses in the loaded library of the functions that FUNCTIONS names, in its order
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  decltype(lib) bound;
  Py_ssize_t i = 0;
#define FQ_SET(name)                                             \
  TORCH_CHECK(i < n_args, "bind() misses the address of fq_" #name); \
  set_function(bound.name, a[i++]);
  FQ_FUNCTIONS(FQ_SET)
#undef FQ_SET
  TORCH_CHECK(i == n_args, "bind() expected ", i, " addresses, got ", n_args);
  lib = bound;
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

// (x, gamma, out, rms, M, n, eps, reuse rms, stream): out and rms are allocated where None is given
PyObject* rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 9);
  const at::Tensor x = in.tensor(), gamma = in.tensor();
  at::Tensor out = in.tensor(), rms = in.tensor();
  const int64_t M = in.integer(), n = in.integer();
  const float eps = in.real();
  const int reuse = in.flag();
  void* stream = in.address();
  const Outputs outputs(x);
  {
    pybind11::gil_scoped_release no_gil;
    if (!out.defined()) out = outputs.empty_like(x);
    if (!rms.defined()) rms = outputs.empty(x, at::kFloat, {M});
    if (M > 0) check(lib.rmsnorm_fwd(data(x), data(gamma), data(out), floats(rms), M, n, eps, reuse, stream));
  }
  return wrap({out, rms});
  END_HANDLE_TH_ERRORS
}

// (dy, x, gamma, rms, dx, M, n, eps, stream): dx is allocated where None is given
PyObject* rmsnorm_bwd(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 9);
  const at::Tensor dy = in.tensor(), x = in.tensor(), gamma = in.tensor(), rms = in.tensor();
  at::Tensor dx = in.tensor(), dgamma;
  const int64_t M = in.integer(), n = in.integer();
  const float eps = in.real();
  void* stream = in.address();
  const Outputs outputs(x);
  {
    pybind11::gil_scoped_release no_gil;
    if (!dx.defined()) dx = outputs.empty_like(x);
    dgamma = outputs.empty(gamma, at::kFloat, {n});
    const int64_t n_partials = lib.rmsnorm_bwd_num_partials(M, n);
    const at::Tensor partials = outputs.empty(gamma, at::kFloat, {n_partials, n});
    check(lib.rmsnorm_bwd(data(dy), data(x), data(gamma), floats(rms), data(dx), floats(dgamma), floats(partials),
                          n_partials, M, n, eps, stream));
  }
  return wrap({dx, dgamma});
  END_HANDLE_TH_ERRORS
}

// (x, gamma, out, scale, rms, eps, round_scale, output_mode, fp8 dtype, kind, stream): out, scale and rms are
// allocated where None is given and the mode writes them
PyObject* rmsnorm_quant(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 11);
  const at::Tensor x = in.tensor(), gamma = in.tensor();
  at::Tensor out = in.tensor(), scale = in.tensor(), rms = in.tensor(), qt, st;
  const float eps = in.real();
  const int round = in.flag(), mode = in.flag();
  const at::ScalarType fp8 = in.dtype();
  const int kind = in.flag();
  void* stream = in.address();
  const Outputs outputs(x);
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), n = x.size(1);
    if (mode != 1) {
      if (!out.defined()) out = outputs.empty(x, fp8, {M, n});
      if (!scale.defined()) scale = outputs.empty(x, at::kFloat, {n / 128, M});
    }
    qt = outputs.empty(x, fp8, {n, M});
    st = outputs.empty(x, at::kFloat, {(M + 127) / 128, n});
    if (!rms.defined()) rms = outputs.empty(x, at::kFloat, {M});
    if (M > 0)
      check(lib.rmsnorm_quant_fwd(data(x), data(gamma), mode != 1 ? data(out) : nullptr,
                                  mode != 1 ? floats(scale) : nullptr, floats(rms), data(qt), floats(st), M, n, eps,
                                  round, mode, kind, stream));
  }
  return wrap({out, scale, rms, qt, st});
  END_HANDLE_TH_ERRORS
}

// (M, K, N, weight is fp32) -> (slices of K, gamma is folded into the weight, bytes of the re-ordered weight, bytes of
// scratch where it is folded): what a call is to know of its sizes, in 0.2 us (ctypes takes 0.55 for each of the four)
PyObject* router_sizes(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 4);
  const int64_t M = in.integer(), K = in.integer(), N = in.integer();
  const int fp32 = in.flag();
  const int slices = lib.rmsnorm_router_slices(M, K, N, fp32);
  PyObject* sizes = Py_BuildValue("(iiLL)", slices, slices ? 0 : lib.rmsnorm_router_folds(M, K, N, fp32),
                                  static_cast<long long>(lib.rmsnorm_router_scratch_bytes(K, N, fp32)),
                                  static_cast<long long>(lib.rmsnorm_router_folded_scratch_bytes(K, N)));
  if (!sizes) throw python_error();
  return sizes;
  END_HANDLE_TH_ERRORS
}

// (x, gamma, weight, logits, its form, weight is fp32, scratch bytes, rms, output_mode, eps, round_scale, stream): rms is
// allocated where None is given; weight: 0 as it is, 1 re-ordered ahead, 2 as it is and gamma is folded into it
PyObject* rmsnorm_router_quant(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 12);
  const at::Tensor x = in.tensor(), gamma = in.tensor(), weight = in.tensor();
  const int64_t N = in.integer();
  const int form = in.flag(), fp32 = in.flag();
  const int64_t scratch_bytes = in.integer();
  at::Tensor rms = in.tensor(), y, logits, q, s, qt, st;
  const int mode = in.flag();
  const float eps = in.real();
  const int round = in.flag();
  void* stream = in.address();
  const Outputs outputs(x);
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), K = x.size(1);
    y = outputs.empty(x, x.scalar_type(), {M, K});
    if (!rms.defined()) rms = outputs.empty(x, at::kFloat, {M});
    logits = outputs.empty(x, at::kFloat, {M, N});
    q = outputs.empty(x, at::kFloat8_e4m3fn, {M, K});
    s = outputs.empty(x, at::kFloat, {K / 128, M});
    qt = outputs.empty(x, at::kFloat8_e4m3fn, {K, M});
    st = outputs.empty(x, at::kFloat, {M / 128, K});
    if (M > 0 && mode == 1) {
      check(lib.rmsnorm_quant_fwd(data(x), data(gamma), nullptr, nullptr, floats(rms), data(qt), floats(st), M, K, eps,
                                  round, 1, FQ_E4M3, stream));
    } else if (M > 0 && form == 1) {
      check(lib.rmsnorm_router_quant_fwd_packed(data(x), data(gamma), data(weight), fp32, data(y), floats(rms),
                                                floats(logits), data(q), floats(s), M, K, N, eps, round, FQ_E4M3,
                                                stream));
    } else if (M > 0 && form == 2) {
      // the two planes of gamma * weight, which every call makes
      const at::Tensor scratch = outputs.empty(x, at::kByte, {scratch_bytes});
      check(lib.rmsnorm_router_quant_fwd_folded(data(x), data(gamma), data(weight), data(scratch), data(y), floats(rms),
                                                floats(logits), data(q), floats(s), M, K, N, eps, round, FQ_E4M3,
                                                stream));
    } else if (M > 0) {
      // the weight re-ordered for the matrix cores (an fp32 weight as two bf16 planes)
      const at::Tensor scratch = outputs.empty(x, at::kByte, {scratch_bytes});
      check(lib.rmsnorm_router_quant_fwd(data(x), data(gamma), data(weight), fp32, data(scratch), data(y), floats(rms),
                                         floats(logits), data(q), floats(s), M, K, N, eps, round, FQ_E4M3, stream));
    }
  }
  return wrap({y, rms, logits, q, s, qt, st});
  END_HANDLE_TH_ERRORS
}

// (x, weight or None, weight is bf16, out, stream): out is allocated where None is given
PyObject* swiglu(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 5);
  const at::Tensor x = in.tensor(), weight = in.tensor();
  const int wbf16 = in.flag();
  at::Tensor out = in.tensor();
  void* stream = in.address();
  const Outputs outputs(x);
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), n = x.size(1) / 2;
    if (!out.defined()) out = outputs.empty(x, x.scalar_type(), {M, n});
    check(lib.swiglu_fwd(data(x), data(weight), wbf16, data(out), M, n, stream));
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// (g, x, weight or None, weight is bf16, stream)
PyObject* swiglu_bwd(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 5);
  const at::Tensor g = in.tensor(), x = in.tensor(), weight = in.tensor();
  const int wbf16 = in.flag();
  void* stream = in.address();
  const Outputs outputs(x);
  at::Tensor dx, dw;
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), N = x.size(1);
    if (weight.defined()) dw = outputs.empty(x, weight.scalar_type(), weight.sizes());
    dx = outputs.empty(x, x.scalar_type(), {M, N});
    check(lib.swiglu_bwd(data(g), data(x), data(weight), wbf16, data(dx), data(dw), M, N / 2, stream));
  }
  return wrap({dx, dw});
  END_HANDLE_TH_ERRORS
}

// (x, out, scale, round_scale, output_mode, fp8 dtype, kind, stream)
PyObject* swiglu_quant(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 8);
  const at::Tensor x = in.tensor();
  at::Tensor out = in.tensor(), scale = in.tensor(), qt, st;
  const int round = in.flag(), mode = in.flag();
  const at::ScalarType fp8 = in.dtype();
  const int kind = in.flag();
  void* stream = in.address();
  const Outputs outputs(x);
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), n = x.size(1) / 2;
    if (!out.defined()) out = outputs.empty(x, fp8, {M, n});
    if (!scale.defined()) scale = outputs.empty(x, at::kFloat, {n / 128, M});
    qt = outputs.empty(x, fp8, {n, M});
    st = outputs.empty(x, at::kFloat, {(M + 127) / 128, n});
    if (M > 0)
      check(lib.swiglu_quant_fwd(data(x), data(out), floats(scale), data(qt), floats(st), M, n, round, mode, kind,
                                 stream));
  }
  return wrap({out, scale, qt, st});
  END_HANDLE_TH_ERRORS
}

// (g, x, round_scale, fp8 dtype, kind, stream)
PyObject* swiglu_quant_bwd(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 6);
  const at::Tensor g = in.tensor(), x = in.tensor();
  const int round = in.flag();
  const at::ScalarType fp8 = in.dtype();
  const int kind = in.flag();
  void* stream = in.address();
  const Outputs outputs(x);
  at::Tensor q, s, qt, st;
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), N = x.size(1);
    q = outputs.empty(x, fp8, {M, N});
    s = outputs.empty(x, at::kFloat, {N / 128, M});
    qt = outputs.empty(x, fp8, {N, M});
    st = outputs.empty(x, at::kFloat, {(M + 127) / 128, N});
    if (M > 0)
      check(lib.swiglu_quant_bwd(data(g), data(x), data(q), floats(s), data(qt), floats(st), M, N / 2, round, kind,
                                 stream));
  }
  return wrap({q, s, qt, st});
  END_HANDLE_TH_ERRORS
}

// (x, weight, weight is bf16, counts, counts are int64, plan's table or None, plan's shape, blocks, out, scale,
// round_scale, output_mode, fp8 dtype, kind, stream): out and scale are allocated where None is given
PyObject* batched_swiglu_quant(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 15);
  const at::Tensor x = in.tensor(), weight = in.tensor();
  const int wbf16 = in.flag();
  const at::Tensor counts = in.tensor();
  const int i64 = in.flag();
  const at::Tensor plan = in.tensor();
  const int64_t* shape = static_cast<const int64_t*>(in.address());
  const int64_t blocks = in.integer();
  at::Tensor out = in.tensor(), scale = in.tensor(), qt, st;
  const int round = in.flag(), mode = in.flag();
  const at::ScalarType fp8 = in.dtype();
  const int kind = in.flag();
  void* stream = in.address();
  const Outputs outputs(x);
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), n = x.size(1) / 2;
    if (!out.defined()) out = outputs.empty(x, fp8, {M, n});
    if (!scale.defined()) scale = outputs.empty(x, at::kFloat, {M, n / 128});
    qt = outputs.empty(x, fp8, {M, n});
    st = outputs.empty(x, at::kFloat, {blocks, n});
    if (M > 0 && plan.defined())
      check(lib.batched_swiglu_quant_fwd_planned(data(x), data(weight), wbf16, data(plan), shape, data(out),
                                                 floats(scale), data(qt), floats(st), M, n, round, mode, kind, stream));
    else if (M > 0)
      check(lib.batched_swiglu_quant_fwd(data(x), data(weight), wbf16, data(counts), i64,
                                         static_cast<int>(counts.size(0)), blocks, data(out), floats(scale), data(qt),
                                         floats(st), M, n, round, mode, kind, stream));
  }
  return wrap({out, scale, qt, st});
  END_HANDLE_TH_ERRORS
}

// (g, x, weight, weight is bf16, dw, counts, counts are int64, plan's table or None, plan's shape, blocks, round_scale,
// fp8 dtype, kind, stream): dw is allocated where None is given
PyObject* batched_swiglu_quant_bwd(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 14);
  const at::Tensor g = in.tensor(), x = in.tensor(), weight = in.tensor();
  const int wbf16 = in.flag();
  at::Tensor dw = in.tensor(), q, s, qt, st;
  const at::Tensor counts = in.tensor();
  const int i64 = in.flag();
  const at::Tensor plan = in.tensor();
  const int64_t* shape = static_cast<const int64_t*>(in.address());
  const int64_t blocks = in.integer();
  const int round = in.flag();
  const at::ScalarType fp8 = in.dtype();
  const int kind = in.flag();
  void* stream = in.address();
  const Outputs outputs(x);
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), N = x.size(1), n = N / 2;
    q = outputs.empty(x, fp8, {M, N});
    s = outputs.empty(x, at::kFloat, {M, N / 128});
    qt = outputs.empty(x, fp8, {M, N});
    st = outputs.empty(x, at::kFloat, {blocks, N});
    if (!dw.defined()) dw = outputs.empty_like(weight);
    if (blocks != 0) {
      const at::Tensor partials = outputs.empty(x, at::kFloat, {M, n / 128});
      if (plan.defined())
        check(lib.batched_swiglu_quant_bwd_planned(data(g), data(x), data(weight), wbf16, data(plan), shape, data(q),
                                                   floats(s), data(dw), data(qt), floats(st), floats(partials), M, n,
                                                   round, kind, stream));
      else
        check(lib.batched_swiglu_quant_bwd(data(g), data(x), data(weight), wbf16, data(counts), i64,
                                           static_cast<int>(counts.size(0)), blocks, data(q), floats(s), data(dw),
                                           data(qt), floats(st), floats(partials), M, n, round, kind, stream));
    }
  }
  return wrap({q, s, dw, qt, st});
  END_HANDLE_TH_ERRORS
}

// (x, round_scale, fp8 dtype, kind, stream)
PyObject* group_quant(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 5);
  const at::Tensor x = in.tensor();
  at::Tensor q, s;
  const int round = in.flag();
  const at::ScalarType fp8 = in.dtype();
  const int kind = in.flag();
  void* stream = in.address();
  const Outputs outputs(x);
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), n = x.size(1);
    q = outputs.empty(x, fp8, {M, n});
    s = outputs.empty(x, at::kFloat, {M, n / 128});
    if (M > 0) check(lib.group_quant(data(x), data(q), floats(s), M, n, round, kind, stream));
  }
  return wrap({q, s});
  END_HANDLE_TH_ERRORS
}

// (x, round_scale, fp8 dtype, kind, stream)
PyObject* block_quant(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 5);
  const at::Tensor x = in.tensor();
  at::Tensor q, s;
  const int round = in.flag();
  const at::ScalarType fp8 = in.dtype();
  const int kind = in.flag();
  void* stream = in.address();
  const Outputs outputs(x);
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), n = x.size(1);
    q = outputs.empty(x, fp8, {M, n});
    s = outputs.empty(x, at::kFloat, {M / 128, n / 128});
    check(lib.block_quant(data(x), data(q), floats(s), M, n, round, kind, stream));
  }
  return wrap({q, s});
  END_HANDLE_TH_ERRORS
}

// (x, round_scale, output_mode, fp8 dtype, kind, stream)
PyObject* blockwise_quant(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 6);
  const at::Tensor x = in.tensor();
  at::Tensor q, s, qt, st;
  const int round = in.flag(), mode = in.flag();
  const at::ScalarType fp8 = in.dtype();
  const int kind = in.flag();
  void* stream = in.address();
  const Outputs outputs(x);
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), n = x.size(1);
    q = outputs.empty(x, fp8, {M, n});
    s = outputs.empty(x, at::kFloat, {n / 128, M});
    qt = outputs.empty(x, fp8, {n, M});
    st = outputs.empty(x, at::kFloat, {(M + 127) / 128, n});
    if (M > 0)
      check(lib.blockwise_quant(data(x), data(q), floats(s), data(qt), floats(st), M, n, round, mode, kind, stream));
  }
  return wrap({q, s, qt, st});
  END_HANDLE_TH_ERRORS
}

// (x, counts, counts are int64, plan's table or None, plan's shape, blocks, round_scale, fp8 dtype, kind, stream)
PyObject* batched_blockwise_quant(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 10);
  const at::Tensor x = in.tensor(), counts = in.tensor();
  const int i64 = in.flag();
  const at::Tensor plan = in.tensor();
  const int64_t* shape = static_cast<const int64_t*>(in.address());
  const int64_t blocks = in.integer();
  const int round = in.flag();
  const at::ScalarType fp8 = in.dtype();
  const int kind = in.flag();
  void* stream = in.address();
  const Outputs outputs(x);
  at::Tensor q, s, qt, st;
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t M = x.size(0), n = x.size(1);
    q = outputs.empty(x, fp8, {M, n});
    s = outputs.empty(x, at::kFloat, {M * n / 128});
    qt = outputs.empty(x, fp8, {M * n});
    st = outputs.empty(x, at::kFloat, {blocks * n});
    if (M > 0 && plan.defined())
      check(lib.batched_blockwise_quant_planned(data(x), data(plan), shape, data(q), floats(s), data(qt), floats(st), M,
                                                n, round, kind, stream));
    else if (M > 0)
      check(lib.batched_blockwise_quant(data(x), data(counts), i64, static_cast<int>(counts.size(0)), blocks, data(q),
                                        floats(s), data(qt), floats(st), M, n, round, kind, stream));
  }
  return wrap({q, s, qt, st});
  END_HANDLE_TH_ERRORS
}

// (x, counts, counts are int64, plan's table or None, plan's shape, blocks, indices, probs or None, probs are bf16,
// launch, round_scale, fp8 dtype, kind, stream); launch 0: the outputs alone
PyObject* batched_pad_permute_quant(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 14);
  const at::Tensor x = in.tensor(), counts = in.tensor();
  const int i64 = in.flag();
  const at::Tensor plan = in.tensor();
  const int64_t* shape = static_cast<const int64_t*>(in.address());
  const int64_t blocks = in.integer();
  const at::Tensor indices = in.tensor(), probs = in.tensor();
  const int pbf16 = in.flag(), launch = in.flag(), round = in.flag();
  const at::ScalarType fp8 = in.dtype();
  const int kind = in.flag();
  void* stream = in.address();
  const Outputs outputs(x);
  at::Tensor q, s, qt, st, prob_out;
  {
    pybind11::gil_scoped_release no_gil;
    const int64_t m = x.size(0), n = x.size(1), M = indices.size(0);
    const int experts = static_cast<int>(counts.size(0));
    q = outputs.empty(x, fp8, {M, n});
    s = outputs.empty(x, at::kFloat, {M, n / 128});
    qt = outputs.empty(x, fp8, {M, n});
    st = outputs.empty(x, at::kFloat, {blocks, n});
    if (probs.defined()) prob_out = outputs.empty(x, probs.scalar_type(), {M});
    if (launch && plan.defined())
      check(lib.batched_pad_permute_quant_planned(data(x), data(plan), shape, experts, data(indices), data(probs),
                                                  pbf16, data(prob_out), data(q), floats(s), data(qt), floats(st), m, M,
                                                  n, round, kind, stream));
    else if (launch)
      check(lib.batched_pad_permute_quant(data(x), data(counts), i64, experts, blocks, data(indices), data(probs),
                                          pbf16, data(prob_out), data(q), floats(s), data(qt), floats(st), m, M, n,
                                          round, kind, stream));
  }
  return wrap({q, s, qt, st, prob_out});
  END_HANDLE_TH_ERRORS
}

// (tokens per expert) -> (128-row blocks, rows with every expert's rounded up to 16)
PyObject* expert_blocks(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n_args == 1, "expected 1 argument, got ", n_args);
  int64_t blocks = 0, padded = 0;
  for (const int64_t c : ints_of(a[0])) {
    blocks += (c + 127) >> 7;  // (below zero rounded as Python's // does)
    padded += ((c + 15) >> 4) * 16;
  }
  PyObject* pair = Py_BuildValue("(LL)", static_cast<long long>(blocks), static_cast<long long>(padded));
  if (!pair) throw python_error();
  return pair;
  END_HANDLE_TH_ERRORS
}

// (counts, counts are int64 (-1: of another type), tokens per expert, pad, address of the plan's shape, stream) -> the plan's
// table, None where there are rows and the counts are of another type
PyObject* expert_plan(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  Args in(a, n_args, 6);
  const at::Tensor counts = in.tensor();
  const int i64 = in.flag();
  const std::vector<int64_t> tokens = in.integers();
  const int pad = in.flag();
  int64_t* shape = static_cast<int64_t*>(in.address());
  void* stream = in.address();
  const int64_t none = 0;
  check(lib.expert_plan_shape(tokens.empty() ? &none : tokens.data(), static_cast<int>(tokens.size()), pad, shape));
  const int64_t bytes = std::max<int64_t>(lib.expert_plan_bytes(shape), 16);
  if (shape[0] == 0)
    return THPVariable_Wrap(at::empty({bytes}, at::TensorOptions().dtype(at::kByte).device(counts.device())));
  if (i64 < 0) Py_RETURN_NONE;
  TORCH_CHECK_VALUE(counts.is_cuda(), "Expected a cuda device, but got: ", counts.device());
  const Outputs outputs(counts);
  at::Tensor table;
  {
    pybind11::gil_scoped_release no_gil;
    table = outputs.empty(counts, at::kByte, {bytes});
    check(lib.build_expert_plan(data(counts), i64, static_cast<int>(counts.size(0)), shape, data(table), stream));
  }
  return THPVariable_Wrap(table);
  END_HANDLE_TH_ERRORS
}

#define FQ_METHOD(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FQ_METHOD(bind),
                         FQ_METHOD(rmsnorm),
                         FQ_METHOD(rmsnorm_bwd),
                         FQ_METHOD(rmsnorm_quant),
                         FQ_METHOD(router_sizes),
                         FQ_METHOD(rmsnorm_router_quant),
                         FQ_METHOD(swiglu),
                         FQ_METHOD(swiglu_bwd),
                         FQ_METHOD(swiglu_quant),
                         FQ_METHOD(swiglu_quant_bwd),
                         FQ_METHOD(batched_swiglu_quant),
                         FQ_METHOD(batched_swiglu_quant_bwd),
                         FQ_METHOD(group_quant),
                         FQ_METHOD(block_quant),
                         FQ_METHOD(blockwise_quant),
                         FQ_METHOD(batched_blockwise_quant),
                         FQ_METHOD(batched_pad_permute_quant),
                         FQ_METHOD(expert_blocks),
                         FQ_METHOD(expert_plan),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fq_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" PyObject* PyInit__fq_torch() {
  PyObject* m = PyModule_Create(&module);
#define FQ_NAME(name) "fq_" #name,
  const char* const names[] = {FQ_FUNCTIONS(FQ_NAME)};
#undef FQ_NAME
  PyObject* functions = m ? PyTuple_New(static_cast<Py_ssize_t>(std::size(names))) : nullptr;
  for (Py_ssize_t i = 0; functions && i < static_cast<Py_ssize_t>(std::size(names)); ++i) {
    PyObject* name = PyUnicode_FromString(names[i]);
    if (!name) Py_CLEAR(functions);
    else PyTuple_SET_ITEM(functions, i, name);
  }
  if (!functions || PyModule_AddObject(m, "FUNCTIONS", functions) < 0) {
    Py_XDECREF(functions);
    Py_CLEAR(m);
  }
  return m;
}
