// One native call per Python API function: the argument checks, the output
// allocations and the launch, without the interpreter in between. Included by
// native.cpp only.
//
// Each function takes its Python function's arguments by position and returns
// its outputs, or None when the call is not the ordinary one (plain contiguous
// torch.Tensors of the supported dtypes on one GPU, consistent shapes, some
// work to do, and no torch function or dispatch mode, no functorch transform
// active): the Python function then goes the long way, through torch.empty and
// the validating *_fwd functions, which raise the errors. So the checks here
// only have to be at least as strict as theirs.
//
// Outputs come from at::empty, the allocator, stream and device of
// torch.empty. What bounds a small call is this host path. Host time of a call
// on [8, 4096] bf16, back to back, the long way vs this: RMSNorm 7.0 vs 5.5 us,
// with per-token FP8 11.5 vs 6.4, SwiGLU + FP8 9.5 vs 5.5, per-token FP8 7.1 vs
// 5.4, per-tensor (two launches) 10.5 vs 9.0, RoPE 6.5 vs 5.7; torch's own x.add_(0)
// takes 4.9, a launch through the *_fwd functions alone 4.0.
#pragma once

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
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

// A plain (exactly torch.Tensor or Parameter), contiguous, non-empty GPU tensor, or nullptr.
inline const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.device().type() != c10::DeviceType::CUDA || t.layout() != c10::kStrided) return nullptr;
  if (t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::Functionalize,
                                               c10::DispatchKey::FuncTorchBatched,
                                               c10::DispatchKey::FuncTorchGradWrapper}))) {
    return nullptr;
  }
  return t.is_contiguous() && t.numel() > 0 ? &t : nullptr;
}

// The tag of a float32 / float16 / bfloat16 tensor, -1 otherwise.
inline int32_t float_tag(const at::Tensor& t) {
  const int32_t tag = tag_of(t.scalar_type());
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

// Without the interpreter lock, as torch.empty: an allocation may have to wait
// for the GPU, whose work may wait for another Python thread.
inline at::Tensor empty(c10::IntArrayRef sizes, c10::ScalarType type, const at::Tensor& like) {
  const auto options = at::TensorOptions().dtype(type).device(like.device());
  const py::gil_scoped_release unlocked;
  return at::empty(sizes, options);
}

inline bool same(const at::Tensor& a, const at::Tensor& b) {
  return a.scalar_type() == b.scalar_type() && a.device() == b.device() && a.sizes() == b.sizes();
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
  const at::Tensor *x = plain(a[0]), *r = plain(a[1]), *w = plain(a[2]);
  if (!x || !r || !w || float_tag(*x) < 0 || !same(*x, *r) || x->dim() < 1) Py_RETURN_NONE;
  const int64_t cols = x->size(-1);
  if (w->dim() != 1 || w->size(0) != cols || w->scalar_type() != x->scalar_type() || w->device() != x->device()) {
    Py_RETURN_NONE;
  }
  const Launch launch(x->device().index());
  at::Tensor y = empty(x->sizes(), x->scalar_type(), *x), ro = empty(x->sizes(), x->scalar_type(), *x);
  check_launch("launch_rmsnorm_residual_fwd",
               launch_rmsnorm_residual_fwd(x->data_ptr(), r->data_ptr(), w->data_ptr(), y.data_ptr(), ro.data_ptr(),
                                           x->numel() / cols, cols, (float)PyFloat_AS_DOUBLE(a[3]), float_tag(*x),
                                           launch.st));
  return result(std::move(y), std::move(ro));
  END_HANDLE_TH_ERRORS
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
  const at::Tensor *x = plain(a[0]), *r = plain(a[1]), *w = plain(a[2]);
  if (fmt < 0 || !x || !r || !w || float_tag(*x) < 0 || !same(*x, *r) || x->dim() < 1) Py_RETURN_NONE;
  const int64_t cols = x->size(-1), rows = x->numel() / cols;
  if (w->dim() != 1 || w->size(0) != cols || w->scalar_type() != x->scalar_type() || w->device() != x->device()) {
    Py_RETURN_NONE;
  }
  const Launch launch(x->device().index());
  at::Tensor q = empty(x->sizes(), fp8_type(fmt), *x), ro = empty(x->sizes(), x->scalar_type(), *x);
  at::Tensor s = is_static ? empty({1}, c10::ScalarType::Float, *x)
                           : empty(x->sizes().slice(0, x->dim() - 1), c10::ScalarType::Float, *x);
  check_launch("launch_rmsnorm_residual_fp8_fwd",
               launch_rmsnorm_residual_fp8_fwd(x->data_ptr(), r->data_ptr(), w->data_ptr(), (uint8_t*)q.data_ptr(),
                                               (float*)s.data_ptr(), ro.data_ptr(), rows, cols,
                                               (float)PyFloat_AS_DOUBLE(a[3]), value,
                                               is_static ? CCK_SCALE_STATIC : CCK_SCALE_TOKEN, float_tag(*x), fmt,
                                               launch.st));
  return result(std::move(q), std::move(s), std::move(ro));
  END_HANDLE_TH_ERRORS
}

// (gate, up)
inline PyObject* swiglu(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !ordinary_state()) Py_RETURN_NONE;
  const at::Tensor *g = plain(a[0]), *u = plain(a[1]);
  if (!g || !u || float_tag(*g) < 0 || !same(*g, *u)) Py_RETURN_NONE;
  const Launch launch(g->device().index());
  at::Tensor y = empty(g->sizes(), g->scalar_type(), *g);
  check_launch("launch_swiglu_fwd", launch_swiglu_fwd(g->data_ptr(), u->data_ptr(), y.data_ptr(), g->numel(),
                                                      float_tag(*g), launch.st));
  return result(std::move(y));
  END_HANDLE_TH_ERRORS
}

// (gate, up, fp8_format, scale)
inline PyObject* swiglu_fp8(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  bool is_static = false;
  float value = 0.0f;
  if (n != 4 || !scale_arg(a[3], &is_static, &value) || !ordinary_state()) Py_RETURN_NONE;
  const int32_t fmt = fmt_tag(a[2]);
  const at::Tensor *g = plain(a[0]), *u = plain(a[1]);
  if (fmt < 0 || !g || !u || float_tag(*g) < 0 || !same(*g, *u) || g->dim() < 1) Py_RETURN_NONE;
  const int64_t cols = g->size(-1);
  const Launch launch(g->device().index());
  at::Tensor q = empty(g->sizes(), fp8_type(fmt), *g);
  at::Tensor s = is_static ? empty({1}, c10::ScalarType::Float, *g)
                           : empty(g->sizes().slice(0, g->dim() - 1), c10::ScalarType::Float, *g);
  check_launch("launch_swiglu_fp8_fwd",
               launch_swiglu_fp8_fwd(g->data_ptr(), u->data_ptr(), (uint8_t*)q.data_ptr(), (float*)s.data_ptr(),
                                     g->numel() / cols, cols, value, is_static ? CCK_SCALE_STATIC : CCK_SCALE_TOKEN,
                                     float_tag(*g), fmt, launch.st));
  return result(std::move(q), std::move(s));
  END_HANDLE_TH_ERRORS
}

// (q, k, cos, sin, inplace)
inline PyObject* rope(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5 || (a[4] != Py_True && a[4] != Py_False) || !ordinary_state()) Py_RETURN_NONE;
  const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *c = plain(a[2]), *s = plain(a[3]);
  if (!q || !k || !c || !s || float_tag(*q) < 0 || q->dim() != 4 || k->dim() != 4) Py_RETURN_NONE;
  const int64_t b = q->size(0), len = q->size(1), d = q->size(3);
  if (k->scalar_type() != q->scalar_type() || k->device() != q->device() || k->size(0) != b || k->size(1) != len ||
      k->size(3) != d || d % 2 != 0 || c->scalar_type() != c10::ScalarType::Float || !same(*c, *s) ||
      c->device() != q->device() || c->dim() != 2 || c->size(0) != len || c->size(1) != d / 2) {
    Py_RETURN_NONE;
  }
  const Launch launch(q->device().index());
  const bool inplace = a[4] == Py_True;
  at::Tensor qo = inplace ? *q : empty(q->sizes(), q->scalar_type(), *q);
  at::Tensor ko = inplace ? *k : empty(k->sizes(), k->scalar_type(), *k);
  check_launch("launch_rope_fwd",
               launch_rope_fwd(q->data_ptr(), k->data_ptr(), c->data_ptr(), s->data_ptr(), qo.data_ptr(),
                               ko.data_ptr(), b, len, q->size(2), k->size(2), d, float_tag(*q), launch.st));
  return result(std::move(qo), std::move(ko));
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
  const at::Tensor* x = plain(a[0]);
  const bool block = PyUnicode_CompareWithASCIIString(a[2], "block") == 0;
  const bool token = !block && PyUnicode_CompareWithASCIIString(a[2], "token") == 0;
  const bool tensor = !block && !token && PyUnicode_CompareWithASCIIString(a[2], "tensor") == 0;
  if (fmt < 0 || !x || float_tag(*x) < 0 || x->dim() != 2 || !(block || token || tensor) || (is_static && !tensor)) {
    Py_RETURN_NONE;
  }
  const int64_t m = x->size(0), cols = x->size(1);
  const int32_t dt = float_tag(*x);
  const Launch launch(x->device().index());
  at::Tensor q = empty({m, cols}, fp8_type(fmt), *x);
  at::Tensor s = block   ? empty({(m + 127) / 128, (cols + 127) / 128}, c10::ScalarType::Float, *x)
                 : token ? empty({m}, c10::ScalarType::Float, *x)
                         : empty({1}, c10::ScalarType::Float, *x);
  const void* xp = x->data_ptr();
  uint8_t* qp = (uint8_t*)q.data_ptr();
  float* sp = (float*)s.data_ptr();
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
  return result(std::move(q), std::move(s));
  END_HANDLE_TH_ERRORS
}

// (src, indices)
inline PyObject* token_gather(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !ordinary_state()) Py_RETURN_NONE;
  const at::Tensor *src = plain(a[0]), *idx = plain(a[1]);
  if (!src || !idx || tag_of(src->scalar_type()) < 0 || src->dim() != 2 || idx->dim() != 1 ||
      idx->scalar_type() != c10::ScalarType::Long || idx->device() != src->device()) {
    Py_RETURN_NONE;
  }
  const Launch launch(src->device().index());
  at::Tensor dst = empty({idx->size(0), src->size(1)}, src->scalar_type(), *src);
  check_launch("launch_token_gather_fwd",
               launch_token_gather_checked_fwd(src->data_ptr(), (const int64_t*)idx->data_ptr(), dst.data_ptr(),
                                               src->size(0), idx->size(0), src->size(1), tag_of(src->scalar_type()),
                                               launch.st));
  return result(std::move(dst));
  END_HANDLE_TH_ERRORS
}

// (expert_output, unpermute_index, weights)
inline PyObject* token_combine(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3 || !ordinary_state()) Py_RETURN_NONE;
  const at::Tensor *eo = plain(a[0]), *idx = plain(a[1]), *w = plain(a[2]);
  if (!eo || !idx || !w || float_tag(*eo) < 0 || eo->dim() != 2 || idx->dim() != 2 ||
      idx->scalar_type() != c10::ScalarType::Long || w->scalar_type() != c10::ScalarType::Float ||
      w->sizes() != idx->sizes() || idx->device() != eo->device() || w->device() != eo->device()) {
    Py_RETURN_NONE;
  }
  const Launch launch(eo->device().index());
  at::Tensor out = empty({idx->size(0), eo->size(1)}, eo->scalar_type(), *eo);
  check_launch("launch_token_combine_fwd",
               launch_token_combine_checked_fwd(eo->data_ptr(), (const int64_t*)idx->data_ptr(),
                                                (const float*)w->data_ptr(), out.data_ptr(), eo->size(0),
                                                idx->size(0), idx->size(1), eo->size(1), float_tag(*eo), launch.st));
  return result(std::move(out));
  END_HANDLE_TH_ERRORS
}

// (topk_indices, num_experts)
inline PyObject* compute_permutation(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !ordinary_state()) Py_RETURN_NONE;
  const at::Tensor* ids = plain(a[0]);
  const int64_t experts = int_arg(a[1], 256);
  if (!ids || experts < 0 || ids->dim() != 2 || ids->scalar_type() != c10::ScalarType::Long) Py_RETURN_NONE;
  const int64_t t = ids->size(0), k = ids->size(1);
  const Launch launch(ids->device().index());
  at::Tensor permute = empty({t * k}, c10::ScalarType::Long, *ids);
  at::Tensor unpermute = empty({t, k}, c10::ScalarType::Long, *ids);
  check_launch("launch_moe_permutation_fwd",
               launch_moe_permutation_fwd((const int64_t*)ids->data_ptr(), (int64_t*)permute.data_ptr(),
                                          (int64_t*)unpermute.data_ptr(), t, k, experts, launch.st));
  return result(std::move(permute), std::move(unpermute));
  END_HANDLE_TH_ERRORS
}

// (logits, k, renormalize)
inline PyObject* moe_router(PyObject*, PyArgs a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3 || (a[2] != Py_True && a[2] != Py_False) || !ordinary_state()) Py_RETURN_NONE;
  const at::Tensor* logits = plain(a[0]);
  if (!logits || float_tag(*logits) < 0 || logits->dim() != 2 || logits->size(1) > 256) Py_RETURN_NONE;
  const int64_t t = logits->size(0), experts = logits->size(1), k = int_arg(a[1], experts);
  if (k < 0) Py_RETURN_NONE;
  const Launch launch(logits->device().index());
  at::Tensor w = empty({t, k}, c10::ScalarType::Float, *logits), ids = empty({t, k}, c10::ScalarType::Long, *logits);
  check_launch("launch_moe_router_fwd",
               launch_moe_router_fwd(logits->data_ptr(), (float*)w.data_ptr(), (int64_t*)ids.data_ptr(), t, experts,
                                     k, float_tag(*logits), a[2] == Py_True ? 1 : 0, launch.st));
  return result(std::move(w), std::move(ids));
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
