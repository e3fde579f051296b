// CPython extension module `vig_host`: the op-level calls of vig_amd/ops.py as one native call each, over the C ABI of
// libvig_gla.so (include/vig_gla.h).  Host code only.
//
// What bounds a small call is the host: through ctypes, the argument checks, two context managers and a dozen pointer
// conversions in Python took 22 us per call at one image's layer (B 1, H 3, L 196), whose kernel takes 8 us.  Here the
// checks, the output's and the workspace's allocation and the launch are one METH_FASTCALL function without a
// dispatcher or a signature parser in between (7.5 us per call, the kernel's own time).  A call that is not of the plain kind (not contiguous, not on the GPU, a
// shape or dtype the kernels do not take, mismatched arguments) returns None before anything has happened, and
// vig_amd/ops.py takes its general path, which also words the errors.
//
// The recorded form is a C++ autograd node: no GIL in the backward pass, and the packed gates of the bidirectional op
// ([2B, H, L, Dk], both directions' one after the other) stay one tensor both ways.  Sliced in Python, the two halves'
// gradients came back as two zero-filled tensors of full size, two copies into them and a sum: 47 of 187 us of device
// time at B 128, H 6, L 196, D 64.
#include "host_calls.h"

namespace {

using namespace vig_host;

// Autograd node of the op (the reference's FusedChunkGLAFunction, chunk_fuse.py:315-518).
struct Gla : torch::autograd::Function<Gla> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& gf,
                        const std::optional<Tensor>& rev, bool packed, int64_t mode, double scale, double out_scale) {
    const Tensor gb = rev ? *rev : Tensor();
    Call c;
    TORCH_CHECK(plain_call(q, k, v, gf, gb, packed, c), "vig_amd: not a plain call");
    c.scale = (float)scale, c.out_scale = (float)out_scale;
    Tensor o;
    check_rc(run_forward(q, k, v, gf, gb, packed, (int)mode, c, o), "vig_gla_bidir_fwd");
    ctx->save_for_backward({q, k, v, gf, gb});
    ctx->saved_data["packed"] = packed;
    ctx->saved_data["exact"] = mode == kExact;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["out_scale"] = out_scale;
    return o;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &gf = saved[3], &gb = saved[4];
    const bool packed = ctx->saved_data["packed"].toBool(), exact = ctx->saved_data["exact"].toBool();
    Call c;
    TORCH_CHECK(plain_call(q, k, v, gf, gb, packed, c), "vig_amd: saved tensors changed");
    Tensor d_o = grads[0].contiguous();
    TORCH_CHECK(d_o.sizes() == v.sizes() && d_o.scalar_type() == q.scalar_type(),
                "d_o must match the output in shape and dtype");
    if (reinterpret_cast<uintptr_t>(d_o.data_ptr()) % 16) d_o = d_o.clone();
    const c10::DeviceGuard guard(q.device());
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v), dgf = at::empty_like(gf), dgb;
    if (gb.defined()) dgb = at::empty_like(gb);
    const void* rev = reverse_gates(gf, gb, packed);
    void* drev = const_cast<void*>(reverse_gates(dgf, dgb, packed));
    const size_t need = exact ? vig_gla_bidir_bwd_workspace(c.B, c.H, c.L, c.Dk, c.Dv, rev != nullptr)
                              : vig_gla_bidir_bwd_workspace_for(c.B, c.H, c.L, c.Dk, c.Dv, c.io, c.gd, rev != nullptr);
    TORCH_CHECK(need > 0, "vig_gla_bidir_bwd: shape Dk=", c.Dk, ", Dv=", c.Dv, " is not built");
    Tensor ws = bytes_like(need, q);
    auto fn = exact ? vig_gla_bidir_bwd_exact : vig_gla_bidir_bwd;
    check_rc(fn(q.data_ptr(), k.data_ptr(), v.data_ptr(), gf.data_ptr(), rev, d_o.data_ptr(), dq.data_ptr(), dk.data_ptr(),
                dv.data_ptr(), dgf.data_ptr(), drev, ws.data_ptr(), need, c.B, c.H, c.L, c.Dk, c.Dv,
                (float)ctx->saved_data["scale"].toDouble(), (float)ctx->saved_data["out_scale"].toDouble(), c.io, c.gd,
                stream_of(q)),
             "vig_gla_bidir_bwd");
    return {dq, dk, dv, dgf, dgb, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// scale None or -1: Dk^-0.5
bool scale_arg(PyObject* o, double& x) {
  x = -1.0;
  if (o != Py_None) x = PyFloat_AsDouble(o);
  return !PyErr_Occurred();
}

PyObject* gla_call(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& gf, const Tensor& gb, bool packed, int mode,
                   double scale, double out_scale) {
  Call c;
  if (!plain_call(q, k, v, gf, gb, packed, c)) Py_RETURN_NONE;
  if (scale == -1.0) scale = std::pow((double)c.Dk, -0.5);
  c.scale = (float)scale, c.out_scale = (float)out_scale;
  if (at::GradMode::is_enabled() &&
      (q.requires_grad() || k.requires_grad() || v.requires_grad() || gf.requires_grad() || (gb.defined() && gb.requires_grad()))) {
    if (c.Dk > 64 || c.Dv > 64 || mode == kWide) Py_RETURN_NONE;  // (wide heads: block by block, ops.py)
    const auto rev = gb.defined() ? std::optional<Tensor>(gb) : std::nullopt;
    return THPVariable_Wrap(Gla::apply(q, k, v, gf, rev, packed, (int64_t)mode, scale, out_scale));
  }
  Tensor o;
  if (run_forward(q, k, v, gf, gb, packed, mode, c, o) != VIG_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(o));
}

// bid_gla(q, k, v, g, scale, out_scale): g [2B, H, L, Dk] = both directions' gates
PyObject* bid_gla(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 6, "bid_gla takes 6 arguments");
  for (int i = 0; i < 4; ++i)
    if (!is_tensor(a[i])) Py_RETURN_NONE;
  double scale;
  if (!scale_arg(a[4], scale)) return nullptr;
  const double out_scale = PyFloat_AsDouble(a[5]);
  return gla_call(THPVariable_Unpack(a[0]), THPVariable_Unpack(a[1]), THPVariable_Unpack(a[2]), THPVariable_Unpack(a[3]),
                  Tensor(), true, kDefault, scale, out_scale);
  END_HANDLE_TH_ERRORS
}

// gla(q, k, v, g_fwd, g_bwd or None, scale, out_scale, mode)
PyObject* gla(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 8, "gla takes 8 arguments");
  for (int i = 0; i < 4; ++i)
    if (!is_tensor(a[i])) Py_RETURN_NONE;
  if (a[4] != Py_None && !is_tensor(a[4])) Py_RETURN_NONE;
  double scale;
  if (!scale_arg(a[5], scale)) return nullptr;
  const double out_scale = PyFloat_AsDouble(a[6]);
  return gla_call(THPVariable_Unpack(a[0]), THPVariable_Unpack(a[1]), THPVariable_Unpack(a[2]), THPVariable_Unpack(a[3]),
                  tensor_arg(a[4]), false, (int)PyLong_AsLong(a[7]), scale, out_scale);
  END_HANDLE_TH_ERRORS
}

// gla_gate(q, k, v, g_fwd, g_bwd or None, weight, h, w, scale, out_scale): the op with the locality gate in its kernel, or
// as a second kernel behind it where the library refuses the one-kernel form
PyObject* gla_gate(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 10, "gla_gate takes 10 arguments");
  for (int i = 0; i < 6; ++i)
    if (!is_tensor(a[i]) && !(i == 4 && a[i] == Py_None)) Py_RETURN_NONE;
  const Tensor &q = THPVariable_Unpack(a[0]), &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]);
  const Tensor &gf = THPVariable_Unpack(a[3]), &weight = THPVariable_Unpack(a[5]);
  const Tensor gb = tensor_arg(a[4]);
  const long h = PyLong_AsLong(a[6]), w = PyLong_AsLong(a[7]);
  double scale;
  if (PyErr_Occurred() || !scale_arg(a[8], scale)) return nullptr;
  const double out_scale = PyFloat_AsDouble(a[9]);
  Call c;
  if (!plain_call(q, k, v, gf, gb, false, c) || h <= 0 || w <= 0 || (int64_t)h * w != c.L) Py_RETURN_NONE;
  if (!plain(weight, q.device()) || weight.scalar_type() != at::kFloat || weight.numel() != (int64_t)c.H * c.Dv * 9)
    Py_RETURN_NONE;
  c.scale = scale == -1.0 ? (float)std::pow((double)c.Dk, -0.5) : (float)scale, c.out_scale = (float)out_scale;
  const c10::DeviceGuard guard(q.device());
  Tensor y = at::empty({c.B, c.H, c.L, c.Dv}, q.options());
  const float* wt = static_cast<const float*>(weight.data_ptr());
  int rc = gb.defined() ? vig_gla_bidir_locgate_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), gf.data_ptr(), gb.data_ptr(), wt,
                                                    y.data_ptr(), c.B, c.H, c.L, c.Dk, c.Dv, (int)h, (int)w, c.scale,
                                                    c.out_scale, c.io, c.gd, stream_of(q))
                        : VIG_ENOTSUP;
  if (rc == VIG_ENOTSUP && gb.defined() && c.L > 256)
    rc = vig_gla_slab_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), gf.data_ptr(), gb.data_ptr(), wt, y.data_ptr(), c.B, c.H, c.L,
                          c.Dk, c.Dv, nullptr, nullptr, nullptr, (int)h, (int)w, c.scale, c.out_scale, c.io, c.gd, stream_of(q));
  if (rc == VIG_ENOTSUP) {
    Tensor o;
    rc = run_forward(q, k, v, gf, gb, false, kDefault, c, o);
    if (rc == VIG_OK)
      rc = vig_locality_gate_fwd(o.data_ptr(), wt, y.data_ptr(), c.B, c.H, (int)h, (int)w, c.Dv, c.io, stream_of(q));
  }
  if (rc != VIG_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"bid_gla", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(bid_gla)), METH_FASTCALL, nullptr},
    {"gla", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(gla)), METH_FASTCALL, nullptr},
    {"gla_gate", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(gla_gate)), METH_FASTCALL, nullptr},
    {"block_mix", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(block_mix)), METH_FASTCALL, nullptr},
    {"block_mlp", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(block_mlp)), METH_FASTCALL, nullptr},
    {"stem_conv", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(stem_conv)), METH_FASTCALL, nullptr},
    {"stem_norm", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(stem_norm)), METH_FASTCALL, nullptr},
    {"make_plan", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(make_plan)), METH_FASTCALL, nullptr},
    {"plan_describes", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(plan_describes)), METH_FASTCALL, nullptr},
    {"run_plan", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(run_plan)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "vig_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit_vig_host() { return PyModule_Create(&kModule); }
