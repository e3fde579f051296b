// What the host-side modules share: tensors of the plain kind, status codes, streams, and the launch of the bidirectional op.
#pragma once
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <ATen/TracerMode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <cmath>
#include <optional>

#include "../../include/vig_gla.h"

namespace vig_host {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

inline void check_rc(int rc, const char* what) {
  TORCH_CHECK(rc == VIG_OK, what, " failed: ", vig_gla_strerror(rc), " (code ", rc, ")");
}
inline void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

inline int dtype_code(const Tensor& t) {
  const auto s = t.scalar_type();
  return s == at::kBFloat16 ? VIG_BF16 : (s == at::kFloat ? VIG_F32 : -1);
}
// Whether somebody records the operators of this call (a trace, a FLOP counter or another dispatch mode): kernels launched
// outside of the dispatcher would be missing from the record, a trace would keep their uninitialised outputs.
inline bool observed() { return at::tracer::impl::is_dispatch_enabled() || c10::impl::dispatch_mode_enabled(); }

// (a tensor subclass that dispatches to Python has no data of its own)
inline bool plain(const Tensor& t, const c10::Device& dev) {
  return t.defined() && !t.unsafeGetTensorImpl()->is_python_dispatch() && t.layout() == at::kStrided && t.device() == dev && t.is_contiguous() &&
         reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

struct Call {
  int B, H, L, Dk, Dv, io, gd;
  float scale, out_scale;
};

// Whether the arguments are of the plain kind the kernels take as they are; fills `c`.  `packed`: gf holds both
// directions' gates, [2B, H, L, Dk].
inline bool plain_call(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& gf, const Tensor& gb, bool packed, Call& c) {
  if (!q.defined() || !q.is_cuda() || q.dim() != 4 || v.dim() != 4 || gf.dim() != 4) return false;
  const auto dev = q.device();
  if (!plain(q, dev) || !plain(k, dev) || !plain(v, dev) || !plain(gf, dev)) return false;
  if (k.sizes() != q.sizes() || v.sizes().slice(0, 3) != q.sizes().slice(0, 3)) return false;
  if (gf.size(0) != q.size(0) * (packed ? 2 : 1) || gf.sizes().slice(1) != q.sizes().slice(1)) return false;
  if (k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
  c.io = dtype_code(q), c.gd = dtype_code(gf);
  if (c.io < 0 || c.gd < 0) return false;
  if (gb.defined() && (packed || !plain(gb, dev) || gb.sizes() != gf.sizes() || gb.scalar_type() != gf.scalar_type())) return false;
  for (int i = 0; i < 4; ++i)
    if (q.size(i) <= 0 || q.size(i) > (1 << 30)) return false;
  c.B = (int)q.size(0), c.H = (int)q.size(1), c.L = (int)q.size(2), c.Dk = (int)q.size(3), c.Dv = (int)v.size(3);
  return (c.Dk == 16 || c.Dk == 32 || c.Dk == 64 || c.Dk == 128) && (c.Dv == 32 || c.Dv == 64 || c.Dv == 128);
}

inline const void* reverse_gates(const Tensor& gf, const Tensor& gb, bool packed) {
  if (packed) return static_cast<const char*>(gf.data_ptr()) + gf.numel() / 2 * gf.element_size();
  return gb.defined() ? gb.data_ptr() : nullptr;
}

inline Tensor bytes_like(size_t n, const Tensor& like) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte)); }

enum Mode { kDefault = 0, kWide = 1, kExact = 2 };

// The launch alone; the status code goes back to the caller (a refusal comes before any launch).
inline int run_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& gf, const Tensor& gb, bool packed, int mode,
                const Call& c, Tensor& o) {
  const c10::DeviceGuard guard(q.device());
  const void* rev = reverse_gates(gf, gb, packed);
  o = at::empty({c.B, c.H, c.L, c.Dv}, q.options());
  const size_t need = mode == kExact ? (rev && c.io != VIG_F32 ? (size_t)c.B * c.H * c.L * c.Dv * 4 : 0)
                                     : vig_gla_bidir_fwd_workspace_for(c.B, c.H, c.L, c.Dk, c.Dv, c.io, c.gd, rev != nullptr);
  Tensor ws;
  if (need) ws = bytes_like(need, q);
  auto fn = mode == kExact ? vig_gla_bidir_fwd_exact : (mode == kWide ? vig_gla_bidir_fwd_wide : vig_gla_bidir_fwd);
  return fn(q.data_ptr(), k.data_ptr(), v.data_ptr(), gf.data_ptr(), rev, o.data_ptr(), need ? ws.data_ptr() : nullptr, need,
            c.B, c.H, c.L, c.Dk, c.Dv, c.scale, c.out_scale, c.io, c.gd, stream_of(q));
}

inline Tensor tensor_arg(PyObject* o) {
  if (o == Py_None) return Tensor();
  return THPVariable_Check(o) ? THPVariable_Unpack(o) : Tensor();
}
inline bool is_tensor(PyObject* o) { return THPVariable_Check(o); }

// the methods of train_block.cpp
PyObject* block_mix(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* block_mlp(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* stem_conv(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* stem_norm(PyObject*, PyObject* const* a, Py_ssize_t n);

// the methods of model_forward.cpp
PyObject* make_plan(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* plan_describes(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* run_plan(PyObject*, PyObject* const* a, Py_ssize_t n);

}  // namespace vig_host
