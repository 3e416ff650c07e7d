// One native call per Python API function: the argument checks, the output
// allocations and the launch, without the interpreter in between. Included by
// native.cpp only.
//
// Each function takes its Python function's arguments by position and returns
// its outputs, or None when the call is not the ordinary one (plain contiguous
// unnamed torch.Tensors of the supported dtypes on one GPU, consistent shapes,
// some work to do, and no torch function or dispatch mode, no functorch
// transform active; a default device, set for the process or by `with
// torch.device(...)`, is such a function mode): the Python function then goes the
// long way, through torch.empty and the validating *_fwd functions, which raise
// the errors. So the checks here only have to be at least as strict as theirs.
//
// Outputs come from at::empty or at::empty_strided, the allocator, stream and
// device of torch.empty. What bounds a small call is this host path. Host time of a call
// on [8, 4096] bf16, back to back, median of three processes each (which differ by
// up to 10 %), the long way vs this: RMSNorm 6.1 vs 5.5 us, with per-token FP8 10.8
// vs 6.3, SwiGLU + FP8 9.5 vs 5.6, per-token FP8 7.2 vs 5.6, RoPE 6.3 vs 5.9, the
// permutation 6.9 vs 5.2, the router 7.5 vs 5.2; torch's own x.add_(0) takes 4.9, a
// launch through the *_fwd functions alone 4.0. Of this, 0.1 to 0.3 us look at the
// inputs again after the allocations and give the outputs the inputs' strides.
#pragma once

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/util/DimVector.h>
#include <torch/csrc/Exceptions.h>

namespace {
namespace calls {

using PyArgs = PyObject* const*;

// No mode or transform that would see the allocations or wrap the tensors.
inline bool ordinary_state() {
  constexpr c10::DispatchKeySet kWrappers({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                           c10::DispatchKey::Functionalize,
                                           c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                           c10::DispatchKey::FuncTorchDynamicLayerBackMode});
  return !at::impl::torch_function_mode_enabled() &&
         !c10::impl::tls_local_dispatch_key_set().included_.has_any(kWrappers);
}

// A plain (exactly torch.Tensor or Parameter), contiguous, non-empty, unnamed GPU tensor, or nullptr.
inline const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.device().type() != c10::DeviceType::CUDA || t.layout() != c10::kStrided) return nullptr;
  if (t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::Functionalize,
                                               c10::DispatchKey::FuncTorchBatched,
                                               c10::DispatchKey::FuncTorchGradWrapper}))) {
    return nullptr;
  }
  return t.is_contiguous() && t.numel() > 0 && !t.has_names() ? &t : nullptr;
}

// A plain input as the checks saw it: what they compare and the outputs are
// sized by is this copy, since another Python thread may set the tensor's data
// whenever the interpreter lock is not held. (Operators that change a tensor
// without the lock, as set_ and resize_, race with any reader of it.)
class Input {
 public:
  explicit Input(PyObject* o) : object_(o), t_(plain(o)) {
    if (t_ == nullptr) return;
    sizes_ = t_->sizes();
    strides_ = t_->strides();
    type_ = t_->scalar_type();
    device_ = t_->device();
  }
  explicit operator bool() const { return t_ != nullptr; }
  // The tensor still is what the checks saw.
  bool unchanged() const {
    return plain(object_) == t_ && t_->sizes() == sizes() && t_->strides() == strides() &&
           t_->scalar_type() == type_ && t_->device() == device_;
  }
  const at::Tensor& tensor() const { return *t_; }
  // For the launch, in the hold of the lock of the last look at the tensor.
  void* data() const { return t_->data_ptr(); }
  c10::IntArrayRef sizes() const { return sizes_; }
  c10::IntArrayRef strides() const { return strides_; }
  int64_t dim() const { return (int64_t)sizes_.size(); }
  int64_t size(int64_t i) const { return sizes_[i < 0 ? i + sizes_.size() : i]; }
  int64_t numel() const { return c10::multiply_integers(sizes_); }
  c10::ScalarType type() const { return type_; }
  c10::Device device() const { return device_; }

 private:
  PyObject* object_;
  const at::Tensor* t_;
  c10::DimVector sizes_, strides_;
  c10::ScalarType type_ = c10::ScalarType::Undefined;
  c10::Device device_ = c10::kCPU;
};

template <class... In>
inline bool unchanged(const In&... in) {
  return (in.unchanged() && ...);
}

// The tag of a float32 / float16 / bfloat16 tensor, -1 otherwise.
inline int32_t float_tag(const Input& t) {
  const int32_t tag = tag_of(t.type());
  return tag == F32 || tag == F16 || tag == BF16 ? tag : -1;
}

// The FP8 tag of a format name, -1 for anything else.
inline int32_t fmt_tag(PyObject* o) {
  if (!PyUnicode_CheckExact(o)) return -1;
  if (PyUnicode_CompareWithASCIIString(o, "e4m3") == 0) return F8E4M3;
  return PyUnicode_CompareWithASCIIString(o, "e5m2") == 0 ? F8E5M2 : -1;
}

inline c10::ScalarType fp8_type(int32_t fmt) {
  return fmt == F8E4M3 ? c10::ScalarType::Float8_e4m3fn : c10::ScalarType::Float8_e5m2;
}

// None (dynamic) or a float (static); false for anything else.
inline bool scale_arg(PyObject* o, bool* is_static, float* value) {
  *is_static = o != Py_None;
  if (!*is_static) return true;
  if (!PyFloat_CheckExact(o)) return false;
  *value = (float)PyFloat_AS_DOUBLE(o);
  return true;
}

// A positive Python int of at most `most`, or -1.
inline int64_t int_arg(PyObject* o, int64_t most) {
  if (!PyLong_CheckExact(o)) return -1;
  int overflow = 0;
  const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0 && v >= 1 && v <= most ? (int64_t)v : -1;
}

// An output: dense in row-major order or, as empty_like, with the strides of
// an input (they differ from those in dimensions of size 1 only).
struct Output {
  c10::IntArrayRef sizes;
  c10::ScalarType type;
  c10::IntArrayRef strides = {};
};
inline Output like(const Input& t) { return {t.sizes(), t.type(), t.strides()}; }

// Without the interpreter lock, as torch.empty: an allocation may have to wait
// for the GPU, whose work may wait for another Python thread. Sizes and strides
// are the caller's copies. The inputs must be looked at again afterwards.
template <size_t N>
inline void allocate(c10::Device device, const Output (&wanted)[N], at::Tensor (&out)[N]) {
  const py::gil_scoped_release unlocked;
  for (size_t i = 0; i < N; ++i) {
    const auto options = at::TensorOptions().dtype(wanted[i].type).device(device);
    out[i] = wanted[i].strides.size() != wanted[i].sizes.size()
                 ? at::empty(wanted[i].sizes, options)
                 : at::empty_strided(wanted[i].sizes, wanted[i].strides, options);
  }
}

inline bool same(const Input& a, const Input& b) {
  return a.type() == b.type() && a.device() == b.device() && a.sizes() == b.sizes();
}

template <class... T>
inline PyObject* result(T... t) {
  if constexpr (sizeof...(T) == 1) {
    return THPVariable_Wrap(std::move(t)...);
  } else {
    py::tuple out(sizeof...(T));
    Py_ssize_t i = 0;
    (PyTuple_SET_ITEM(out.ptr(), i++, THPVariable_Wrap(std::move(t))), ...);
    return out.release().ptr();
  }
}

// (x, residual, weight, eps)
inline PyObject* rmsnorm_residual(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4 || !PyFloat_CheckExact(a[3]) || !ordinary_state()) Py_RETURN_NONE;
  const Input x(a[0]), r(a[1]), w(a[2]);
  if (!x || !r || !w || float_tag(x) < 0 || !same(x, r) || x.dim() < 1) Py_RETURN_NONE;
  const int64_t cols = x.size(-1);
  if (w.dim() != 1 || w.size(0) != cols || w.type() != x.type() || w.device() != x.device()) Py_RETURN_NONE;
  const Launch launch(x.device().index());
  at::Tensor out[2];
  allocate(x.device(), {like(x), like(x)}, out);
  if (!unchanged(x, r, w)) Py_RETURN_NONE;
  check_launch("launch_rmsnorm_residual_fwd",
               launch_rmsnorm_residual_fwd(x.data(), r.data(), w.data(), out[0].data_ptr(), out[1].data_ptr(),
                                           x.numel() / cols, cols, (float)PyFloat_AS_DOUBLE(a[3]), float_tag(x),
                                           launch.st));
  return result(std::move(out[0]), std::move(out[1]));
  END_HANDLE_TH_ERRORS
}

// The scale tensor of the fused FP8 calls: one scale a row of x, or one.
constexpr int64_t kOne[1] = {1};
inline Output scales_of(const Input& x, bool is_static) {
  return {is_static ? c10::IntArrayRef(kOne) : x.sizes().slice(0, x.dim() - 1), c10::ScalarType::Float};
}

// (x, residual, weight, eps, fp8_format, scale)
inline PyObject* rmsnorm_residual_fp8(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  bool is_static = false;
  float value = 0.0f;
  if (n != 6 || !PyFloat_CheckExact(a[3]) || !scale_arg(a[5], &is_static, &value) || !ordinary_state()) {
    Py_RETURN_NONE;
  }
  const int32_t fmt = fmt_tag(a[4]);
  const Input x(a[0]), r(a[1]), w(a[2]);
  if (fmt < 0 || !x || !r || !w || float_tag(x) < 0 || !same(x, r) || x.dim() < 1) Py_RETURN_NONE;
  const int64_t cols = x.size(-1);
  if (w.dim() != 1 || w.size(0) != cols || w.type() != x.type() || w.device() != x.device()) Py_RETURN_NONE;
  const Launch launch(x.device().index());
  at::Tensor out[3];
  allocate(x.device(), {{x.sizes(), fp8_type(fmt)}, scales_of(x, is_static), like(x)}, out);
  if (!unchanged(x, r, w)) Py_RETURN_NONE;
  check_launch("launch_rmsnorm_residual_fp8_fwd",
               launch_rmsnorm_residual_fp8_fwd(x.data(), r.data(), w.data(), (uint8_t*)out[0].data_ptr(),
                                               (float*)out[1].data_ptr(), out[2].data_ptr(), x.numel() / cols, cols,
                                               (float)PyFloat_AS_DOUBLE(a[3]), value,
                                               is_static ? CCK_SCALE_STATIC : CCK_SCALE_TOKEN, float_tag(x), fmt,
                                               launch.st));
  return result(std::move(out[0]), std::move(out[1]), std::move(out[2]));
  END_HANDLE_TH_ERRORS
}

// (gate, up)
inline PyObject* swiglu(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !ordinary_state()) Py_RETURN_NONE;
  const Input g(a[0]), u(a[1]);
  if (!g || !u || float_tag(g) < 0 || !same(g, u)) Py_RETURN_NONE;
  const Launch launch(g.device().index());
  at::Tensor out[1];
  allocate(g.device(), {like(g)}, out);
  if (!unchanged(g, u)) Py_RETURN_NONE;
  check_launch("launch_swiglu_fwd",
               launch_swiglu_fwd(g.data(), u.data(), out[0].data_ptr(), g.numel(), float_tag(g), launch.st));
  return result(std::move(out[0]));
  END_HANDLE_TH_ERRORS
}

// (gate, up, fp8_format, scale)
inline PyObject* swiglu_fp8(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  bool is_static = false;
  float value = 0.0f;
  if (n != 4 || !scale_arg(a[3], &is_static, &value) || !ordinary_state()) Py_RETURN_NONE;
  const int32_t fmt = fmt_tag(a[2]);
  const Input g(a[0]), u(a[1]);
  if (fmt < 0 || !g || !u || float_tag(g) < 0 || !same(g, u) || g.dim() < 1) Py_RETURN_NONE;
  const int64_t cols = g.size(-1);
  const Launch launch(g.device().index());
  at::Tensor out[2];
  allocate(g.device(), {{g.sizes(), fp8_type(fmt)}, scales_of(g, is_static)}, out);
  if (!unchanged(g, u)) Py_RETURN_NONE;
  check_launch("launch_swiglu_fp8_fwd",
               launch_swiglu_fp8_fwd(g.data(), u.data(), (uint8_t*)out[0].data_ptr(), (float*)out[1].data_ptr(),
                                     g.numel() / cols, cols, value, is_static ? CCK_SCALE_STATIC : CCK_SCALE_TOKEN,
                                     float_tag(g), fmt, launch.st));
  return result(std::move(out[0]), std::move(out[1]));
  END_HANDLE_TH_ERRORS
}

// (q, k, cos, sin, inplace)
inline PyObject* rope(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5 || (a[4] != Py_True && a[4] != Py_False) || !ordinary_state()) Py_RETURN_NONE;
  const Input q(a[0]), k(a[1]), c(a[2]), s(a[3]);
  if (!q || !k || !c || !s || float_tag(q) < 0 || q.dim() != 4 || k.dim() != 4) Py_RETURN_NONE;
  const int64_t b = q.size(0), len = q.size(1), d = q.size(3);
  if (k.type() != q.type() || k.device() != q.device() || k.size(0) != b || k.size(1) != len || k.size(3) != d ||
      d % 2 != 0 || c.type() != c10::ScalarType::Float || !same(c, s) || c.device() != q.device() || c.dim() != 2 ||
      c.size(0) != len || c.size(1) != d / 2) {
    Py_RETURN_NONE;
  }
  const Launch launch(q.device().index());
  at::Tensor out[2];
  if (a[4] == Py_True) {
    out[0] = q.tensor();
    out[1] = k.tensor();
  } else {
    allocate(q.device(), {like(q), like(k)}, out);
    if (!unchanged(q, k, c, s)) Py_RETURN_NONE;
  }
  check_launch("launch_rope_fwd",
               launch_rope_fwd(q.data(), k.data(), c.data(), s.data(), out[0].data_ptr(), out[1].data_ptr(), b, len,
                               q.size(2), k.size(2), d, float_tag(q), launch.st));
  return result(std::move(out[0]), std::move(out[1]));
  END_HANDLE_TH_ERRORS
}

// (x, fp8_format, granularity, scale)
inline PyObject* fp8_quant(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  bool is_static = false;
  float value = 0.0f;
  if (n != 4 || !PyUnicode_CheckExact(a[2]) || !scale_arg(a[3], &is_static, &value) || !ordinary_state()) {
    Py_RETURN_NONE;
  }
  const int32_t fmt = fmt_tag(a[1]);
  const Input x(a[0]);
  const bool block = PyUnicode_CompareWithASCIIString(a[2], "block") == 0;
  const bool token = !block && PyUnicode_CompareWithASCIIString(a[2], "token") == 0;
  const bool tensor = !block && !token && PyUnicode_CompareWithASCIIString(a[2], "tensor") == 0;
  if (fmt < 0 || !x || float_tag(x) < 0 || x.dim() != 2 || !(block || token || tensor) || (is_static && !tensor)) {
    Py_RETURN_NONE;
  }
  const int64_t m = x.size(0), cols = x.size(1);
  const int32_t dt = float_tag(x);
  const int64_t tiles[2] = {(m + 127) / 128, (cols + 127) / 128};
  const c10::IntArrayRef scales = block ? c10::IntArrayRef(tiles) : token ? x.sizes().slice(0, 1) : c10::IntArrayRef(kOne);
  const Launch launch(x.device().index());
  at::Tensor out[2];
  allocate(x.device(), {{x.sizes(), fp8_type(fmt)}, {scales, c10::ScalarType::Float}}, out);
  if (!unchanged(x)) Py_RETURN_NONE;
  const void* xp = x.data();
  uint8_t* qp = (uint8_t*)out[0].data_ptr();
  float* sp = (float*)out[1].data_ptr();
  if (is_static) {
    check_launch("launch_fp8_quant_static_fwd",
                 launch_fp8_quant_static_fwd(xp, qp, value, sp, m, cols, dt, fmt, launch.st));
  } else if (block) {
    check_launch("launch_fp8_quant_block_fwd", launch_fp8_quant_block_fwd(xp, qp, sp, m, cols, dt, fmt, launch.st));
  } else if (token) {
    check_launch("launch_fp8_quant_token_fwd", launch_fp8_quant_token_fwd(xp, qp, sp, m, cols, dt, fmt, launch.st));
  } else {
    check_launch("launch_fp8_quant_tensor_fwd",
                 launch_fp8_quant_tensor_fwd(xp, qp, sp, nullptr, m, cols, dt, fmt, launch.st));
  }
  return result(std::move(out[0]), std::move(out[1]));
  END_HANDLE_TH_ERRORS
}

// (src, indices)
inline PyObject* token_gather(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !ordinary_state()) Py_RETURN_NONE;
  const Input src(a[0]), idx(a[1]);
  if (!src || !idx || tag_of(src.type()) < 0 || src.dim() != 2 || idx.dim() != 1 ||
      idx.type() != c10::ScalarType::Long || idx.device() != src.device()) {
    Py_RETURN_NONE;
  }
  const int64_t sizes[2] = {idx.size(0), src.size(1)};
  const Launch launch(src.device().index());
  at::Tensor out[1];
  allocate(src.device(), {{sizes, src.type()}}, out);
  if (!unchanged(src, idx)) Py_RETURN_NONE;
  check_launch("launch_token_gather_fwd",
               launch_token_gather_checked_fwd(src.data(), (const int64_t*)idx.data(), out[0].data_ptr(), src.size(0),
                                               sizes[0], sizes[1], tag_of(src.type()), launch.st));
  return result(std::move(out[0]));
  END_HANDLE_TH_ERRORS
}

// (expert_output, unpermute_index, weights)
inline PyObject* token_combine(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3 || !ordinary_state()) Py_RETURN_NONE;
  const Input eo(a[0]), idx(a[1]), w(a[2]);
  if (!eo || !idx || !w || float_tag(eo) < 0 || eo.dim() != 2 || idx.dim() != 2 ||
      idx.type() != c10::ScalarType::Long || w.type() != c10::ScalarType::Float || w.sizes() != idx.sizes() ||
      idx.device() != eo.device() || w.device() != eo.device()) {
    Py_RETURN_NONE;
  }
  const int64_t sizes[2] = {idx.size(0), eo.size(1)};
  const Launch launch(eo.device().index());
  at::Tensor out[1];
  allocate(eo.device(), {{sizes, eo.type()}}, out);
  if (!unchanged(eo, idx, w)) Py_RETURN_NONE;
  check_launch("launch_token_combine_fwd",
               launch_token_combine_checked_fwd(eo.data(), (const int64_t*)idx.data(), (const float*)w.data(),
                                                out[0].data_ptr(), eo.size(0), sizes[0], idx.size(1), sizes[1],
                                                float_tag(eo), launch.st));
  return result(std::move(out[0]));
  END_HANDLE_TH_ERRORS
}

// (topk_indices, num_experts)
inline PyObject* compute_permutation(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !ordinary_state()) Py_RETURN_NONE;
  const Input ids(a[0]);
  const int64_t experts = int_arg(a[1], 256);
  if (!ids || experts < 0 || ids.dim() != 2 || ids.type() != c10::ScalarType::Long) Py_RETURN_NONE;
  const int64_t flat[1] = {ids.numel()};
  const Launch launch(ids.device().index());
  at::Tensor out[2];
  allocate(ids.device(), {{flat, c10::ScalarType::Long}, {ids.sizes(), c10::ScalarType::Long}}, out);
  if (!unchanged(ids)) Py_RETURN_NONE;
  check_launch("launch_moe_permutation_fwd",
               launch_moe_permutation_fwd((const int64_t*)ids.data(), (int64_t*)out[0].data_ptr(),
                                          (int64_t*)out[1].data_ptr(), ids.size(0), ids.size(1), experts, launch.st));
  return result(std::move(out[0]), std::move(out[1]));
  END_HANDLE_TH_ERRORS
}

// (logits, k, renormalize)
inline PyObject* moe_router(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3 || (a[2] != Py_True && a[2] != Py_False) || !ordinary_state()) Py_RETURN_NONE;
  const Input logits(a[0]);
  if (!logits || float_tag(logits) < 0 || logits.dim() != 2 || logits.size(1) > 256) Py_RETURN_NONE;
  const int64_t experts = logits.size(1), k = int_arg(a[1], experts);
  if (k < 0) Py_RETURN_NONE;
  const int64_t sizes[2] = {logits.size(0), k};
  const Launch launch(logits.device().index());
  at::Tensor out[2];
  allocate(logits.device(), {{sizes, c10::ScalarType::Float}, {sizes, c10::ScalarType::Long}}, out);
  if (!unchanged(logits)) Py_RETURN_NONE;
  check_launch("launch_moe_router_fwd",
               launch_moe_router_fwd(logits.data(), (float*)out[0].data_ptr(), (int64_t*)out[1].data_ptr(), sizes[0],
                                     experts, k, float_tag(logits), a[2] == Py_True ? 1 : 0, launch.st));
  return result(std::move(out[0]), std::move(out[1]));
  END_HANDLE_TH_ERRORS
}

using FastCall = PyObject* (*)(PyObject*, PyArgs, Py_ssize_t);
template <FastCall F>
PyCFunction as_method() {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(F));
}

inline PyMethodDef kMethods[] = {
    {"rmsnorm_residual_call", as_method<rmsnorm_residual>(), METH_FASTCALL, nullptr},
    {"rmsnorm_residual_fp8_call", as_method<rmsnorm_residual_fp8>(), METH_FASTCALL, nullptr},
    {"swiglu_call", as_method<swiglu>(), METH_FASTCALL, nullptr},
    {"swiglu_fp8_call", as_method<swiglu_fp8>(), METH_FASTCALL, nullptr},
    {"rope_call", as_method<rope>(), METH_FASTCALL, nullptr},
    {"fp8_quant_call", as_method<fp8_quant>(), METH_FASTCALL, nullptr},
    {"token_gather_call", as_method<token_gather>(), METH_FASTCALL, nullptr},
    {"token_combine_call", as_method<token_combine>(), METH_FASTCALL, nullptr},
    {"compute_permutation_call", as_method<compute_permutation>(), METH_FASTCALL, nullptr},
    {"moe_router_call", as_method<moe_router>(), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

}  // namespace calls
}  // namespace
