// The evaluation forward of a whole ViG (classification/models/vig.py:880-912) in bf16 as one native call over the C ABI:
// stem, blocks in the carried form, closing norm with the mean over tokens, classifier.
//
// At small batches the model is bound by the host: 117 launches through Python modules, operator dispatch and the BLAS
// library's own front end took 1.45 ms for one 224 px image whose kernels need 0.85.  Here a forward is a walk over a plan (raw
// pointers of the parameters and of their packed copies, laid out once) with one allocation for all activations.
//
// A plan describes the model as it was when the plan was made.  Each call first checks that it still is: the entries of
// the modules' own dictionaries (submodules, parameters, settings, absent overrides, empty hook tables) by identity, and every
// parameter's storage address, version counter and type.  About 500 lookups, 12 us, while the GPU still works on the call before.
// ViG-T, one 224 px image: 1.49 -> 0.47 ms; ViG-T, 8 x 1024 px: 2.49 -> 2.07 ms (the stem's and the row kernels' share included).
#include <ATen/autocast_mode.h>

#include <algorithm>

#include "host_calls.h"

namespace vig_host {

namespace {

struct Ref {  // an owned Python object
  PyObject* o = nullptr;
  explicit Ref(PyObject* p) : o(p) { Py_XINCREF(o); }
  Ref(Ref&& r) noexcept : o(r.o) { r.o = nullptr; }
  Ref(const Ref&) = delete;
  ~Ref() { Py_XDECREF(o); }
};

struct Entry {
  Ref dict, key, value;  // value NULL: the key has to be absent
};
struct Watched {
  Tensor t;
  c10::Storage storage;  // kept, so that nothing else can come to lie at ptr
  void* ptr;
  uint32_t version;
  at::ScalarType type;
};

struct Stem {
  Tensor w1, b1, ln1w, ln1b, w2, b2, ln2w, ln2b, pos;
  double eps1, eps2;
  int KH, KW, gh, gw;
};
struct Block {
  Tensor norm1, conv_w, conv_b, w_in, b_in, w_up, b_up, gn, ln, w_o, norm2, w_gate, w_down;
  double eps1, eps, eps2, inv_norm, clamp;
  int H, Dk, Dv, act, out_act;
};
struct Plan {
  std::vector<Entry> entries;
  std::vector<Ref> empty;
  std::vector<Watched> watched;
  std::vector<PyObject*> modules;  // sorted; the model itself, and children that `entries` keep alive
  Stem stem;
  std::vector<Block> blocks;
  Tensor norm, head_w, head_b;
  double norm_eps;
};

constexpr const char* kPlanName = "vig_amd.plan";
void free_plan(PyObject* cap) { delete static_cast<Plan*>(PyCapsule_GetPointer(cap, kPlanName)); }

bool still_valid(const Plan& p) {
  for (const auto& e : p.entries) {
    PyObject* v = PyDict_GetItemWithError(e.dict.o, e.key.o);
    if (v != e.value.o) {
      PyErr_Clear();
      return false;
    }
  }
  for (const auto& d : p.empty)
    if (!d.o || PyDict_Size(d.o) != 0) return false;
  for (const auto& w : p.watched)
    if (w.t.data_ptr() != w.ptr || w.t._version() != (int64_t)w.version || w.t.scalar_type() != w.type) return false;
  return true;
}

// ---- reading the plan's description ----
struct Reader {
  PyObject* tuple;
  Py_ssize_t i = 0;
  PyObject* next() {
    PyObject* o = PyTuple_GetItem(tuple, i++);
    if (!o) throw python_error();
    return o;
  }
  Tensor tensor() { return tensor_arg(next()); }
  double real() {
    PyObject* o = next();
    const double v = o == Py_None ? std::nan("") : PyFloat_AsDouble(o);
    if (PyErr_Occurred()) throw python_error();
    return v;
  }
  int integer() {
    const long v = PyLong_AsLong(next());
    if (PyErr_Occurred()) throw python_error();
    return (int)v;
  }
};

// ---- the walk ----
struct Walk {
  Tensor space;  // every activation of the call, bf16 elements
  void* stream;
  int64_t used = 0;
  int64_t take(int64_t n) {
    const int64_t at = used;
    used += (n + 127) / 128 * 128;
    return at;
  }
  void* at(int64_t off) const { return static_cast<char*>(space.data_ptr()) + 2 * off; }
  Tensor rows(int64_t off, int64_t M, int64_t N) const { return space.as_strided({M, N}, {N, 1}, off); }
  void linear(int64_t x, const Tensor& w, const Tensor& b, int64_t y, int64_t M) const {
    const int64_t N = w.size(0), K = w.size(1);
    if (vig_linear_preferred(M, (int)N, (int)K)) {
      check_rc(vig_linear_fwd(at(x), K, w.data_ptr(), b.defined() ? b.data_ptr() : nullptr, at(y), N, M, (int)N, (int)K, stream),
               "vig_linear_fwd");
      return;
    }
    Tensor out = rows(y, M, N);
    if (b.defined()) at::addmm_out(out, b, rows(x, M, K), w.t());
    else at::mm_out(out, rows(x, M, K), w.t());
  }
  void norm(int64_t x, int64_t residual, const Tensor& w, double eps, bool round_sum, int64_t y, int64_t sum, int64_t M) const {
    check_rc(vig_rmsnorm_fwd(at(x), residual < 0 ? nullptr : at(residual), static_cast<const float*>(w.data_ptr()), at(y),
                             sum < 0 ? nullptr : at(sum), M, (int)w.numel(), (float)eps, round_sum, VIG_BF16, stream),
             "vig_rmsnorm_fwd");
  }
};
const float* f32(const Tensor& t) { return t.defined() ? static_cast<const float*>(t.data_ptr()) : nullptr; }

Tensor run(const Plan& p, const Tensor& images) {
  const int64_t B = images.size(0), S = images.size(2), W = images.size(3);
  const Stem& st = p.stem;
  const int64_t half = st.w1.size(0), C = st.w2.size(0), cin = images.size(1);
  const int64_t oh1 = (S + 2 - st.KH) / 8 + 1, ow1 = (W + 2 - st.KW) / 8 + 1;
  const int64_t L = (int64_t)st.gh * st.gw, T = B * L, n1 = B * oh1 * ow1;
  const int64_t classes = p.head_w.size(0);
  int64_t nz = 0, I = 0, K2 = 0;
  bool swiglu_kernel = C == 384 || C == 192;  // in every block
  for (const auto& b : p.blocks) {
    nz = std::max(nz, b.w_in.size(0)), I = std::max(I, b.w_down.size(1)), K2 = std::max<int64_t>(K2, 2 * b.H * b.Dk);
    swiglu_kernel = swiglu_kernel && b.w_down.size(1) % 32 == 0;
  }
  // q, k, v are read in place from the projection's rows, with the gates made in the same kernels or by one of their own, or split into heads
  const auto lowrank = [&](const Block& b) { return b.Dk == 32 && b.Dv == 64 && b.w_up.size(1) == 16; };
  const auto whole = [&](const Block& b) { return L <= vig_gla_slab_tokens(b.Dk); };
  bool all_lowrank = true, all_in_place = true;
  size_t gla_ws = 0;
  for (const auto& b : p.blocks) {
    all_lowrank = all_lowrank && lowrank(b), all_in_place = all_in_place && (lowrank(b) || whole(b));
    const size_t need = lowrank(b) ? vig_gla_lowrank_fwd_workspace((int)B, b.H, (int)L, b.Dk, b.Dv)
                        : whole(b) ? 0
                                   : vig_gla_bidir_fwd_workspace_for((int)B, b.H, (int)L, b.Dk, b.Dv, VIG_BF16, VIG_BF16, 1);
    gla_ws = std::max(gla_ws, need);
  }
  Walk k;
  k.stream = stream_of(images);
  // branch and residual alternate between two places each; the mixer's and the MLP's intermediates share one region
  const int64_t branch0 = k.take(T * C), branch1 = k.take(T * C), res0 = k.take(T * C), res1 = k.take(T * C), y = k.take(T * C),
                xs = k.take(T * C), o = k.take(T * C);
  const int64_t region = k.used;
  const int64_t z = k.take(T * nz), gates = all_lowrank ? 0 : k.take(T * K2), ws = k.take((int64_t)(gla_ws + 1) / 2);
  int64_t q = 0, kk = 0, v = 0;
  if (!all_in_place) q = k.take(T * K2 / 2), kk = k.take(T * K2 / 2), v = k.take(T * C);
  int64_t most = k.used;
  k.used = region;
  int64_t mid = k.take(T * I);
  const int64_t wide = swiglu_kernel ? 0 : k.take(T * 2 * I);
  most = std::max(most, k.used);
  const auto one_middle = [&](const Block& b) { return b.Dv == 64 && vig_locality_blend_swiglu_preferred(T, (int)C, (int)b.w_down.size(1)); };
  if (std::any_of(p.blocks.begin(), p.blocks.end(), one_middle)) {  // (reads z while it writes mid)
    k.used = most;
    mid = k.take(T * I);
    most = k.used;
  }
  k.used = region;
  const int64_t c1 = k.take(n1 * half), c1n = half > 256 ? k.take(n1 * half) : c1;  // (beyond: two kernels)
  most = std::max(most, k.used);
  k.used = region;
  const size_t pool_ws = vig_rmsnorm_pool_workspace((int)B, (int)L, (int)C);
  const int64_t part = k.take((int64_t)(pool_ws + 1) / 2), pooled = k.take(B * C);
  most = std::max(most, k.used);
  k.space = at::empty({most}, images.options());

  // ---- stem: convolution, norm + SiLU, convolution, norm + position table (each convolution's bias rides in the norm behind) ----
  int64_t stem = c1;
  int rc = vig_patch_conv_norm_fwd(images.data_ptr(), st.w1.data_ptr(), f32(st.ln1w), f32(st.ln1b), f32(st.b1), k.at(c1), (int)B, (int)cin, (int)S, (int)W,
                                   st.KH, st.KW, 8, 1, (int)half, (float)st.eps1, 1, k.stream);
  if (rc == VIG_ENOTSUP) {
    check_rc(vig_patch_conv_fwd(images.data_ptr(), st.w1.data_ptr(), k.at(c1), (int)B, (int)cin, (int)S, (int)W, st.KH, st.KW, 8, 1,
                                (int)half, VIG_BF16, k.stream),
             "vig_patch_conv_fwd");
    stem = c1n;
    rc = vig_layernorm_fwd(k.at(c1), f32(st.ln1w), f32(st.ln1b), k.at(c1n), n1, (int)half, (float)st.eps1, 1, f32(st.b1), nullptr, 0, VIG_BF16,
                           k.stream);
  }
  check_rc(rc, "the stem's first norm");
  check_rc(vig_conv3x3s2_fwd(k.at(stem), st.w2.data_ptr(), k.at(y), (int)B, (int)oh1, (int)ow1, (int)half, (int)C, k.stream),
           "vig_conv3x3s2_fwd");
  check_rc(vig_layernorm_fwd(k.at(y), f32(st.ln2w), f32(st.ln2b), k.at(branch0), T, (int)C, (float)st.eps2, 0, f32(st.b2),
                             st.pos.data_ptr(), (int)L, VIG_BF16, k.stream),
           "vig_layernorm_fwd");

  int64_t residual = -1;
  bool normed = false;  // the block before left its sum and this block's norm of it
  for (size_t i = 0; i < p.blocks.size(); ++i) {
    const Block& b = p.blocks[i];
    const int64_t n0 = (int64_t)b.H * (2 * b.Dk + b.Dv), n1c = n0 + (int64_t)b.H * b.Dv, ld = b.w_in.size(0);
    int64_t hidden = branch0;
    // the explicit add of the reference stores a rounded sum and attn_norm normalises that (vig.py:598,606)
    const bool sums = !normed && residual >= 0;
    if (normed) hidden = residual;
    else if (sums) hidden = residual == res0 ? res1 : res0;
    if (!normed && vig_norm_dwconv3x3_linear_preferred((int)B, st.gh, st.gw, (int)C, (int)ld)) {
      check_rc(vig_norm_dwconv3x3_linear_fwd(k.at(branch0), sums ? k.at(residual) : nullptr, f32(b.norm1), f32(b.conv_w), f32(b.conv_b),
                                             b.w_in.data_ptr(), b.b_in.data_ptr(), sums ? k.at(hidden) : nullptr, k.at(xs), k.at(z), (int)B,
                                             st.gh, st.gw, (int)C, (int)ld, (float)b.eps1, b.act, k.stream),
               "vig_norm_dwconv3x3_linear_fwd");
    } else {
      if (!normed && vig_norm_dwconv3x3_preferred((int)B, st.gh, st.gw, (int)C)) {
        check_rc(vig_norm_dwconv3x3_fwd(k.at(branch0), sums ? k.at(residual) : nullptr, f32(b.norm1), f32(b.conv_w), f32(b.conv_b),
                                        sums ? k.at(hidden) : nullptr, k.at(xs), (int)B, st.gh, st.gw, (int)C, (float)b.eps1, b.act, k.stream),
                 "vig_norm_dwconv3x3_fwd");
      } else {
        if (!normed) k.norm(branch0, sums ? residual : -1, b.norm1, b.eps1, sums, y, sums ? hidden : -1, T);
        check_rc(vig_dwconv3x3_fwd(k.at(y), f32(b.conv_w), f32(b.conv_b), k.at(xs), (int)B, st.gh, st.gw, (int)C, b.act, VIG_BF16, k.stream),
                 "vig_dwconv3x3_fwd");
      }
      k.linear(xs, b.w_in, b.b_in, z, T);
    }
    const float scale = 1.0f / std::sqrt((float)b.Dk);
    const long long sqk[3] = {(long long)(L * ld), b.Dk, ld}, sv[3] = {(long long)(L * ld), b.Dv, ld};
    if (lowrank(b)) {
      check_rc(vig_gla_lowrank_fwd(k.at(z), k.at(z + b.H * b.Dk), k.at(z + 2 * b.H * b.Dk), k.at(z + n1c), ld, b.w_up.data_ptr(),
                                   b.b_up.data_ptr(), k.at(o), gla_ws ? k.at(ws) : nullptr, gla_ws, (int)B, b.H, (int)L, b.Dk, b.Dv, sqk,
                                   sqk, sv, (float)b.inv_norm, (float)b.clamp, scale, 0.25f, VIG_BF16, k.stream),
               "vig_gla_lowrank_fwd");
    } else {
      check_rc(vig_dirgate_lowrank_fwd(k.at(z + n1c), ld, b.w_up.data_ptr(), b.b_up.data_ptr(), k.at(gates), (int)B, (int)L, b.H, b.Dk,
                                       (int)b.w_up.size(1), (float)b.inv_norm, (float)b.clamp, VIG_BF16, VIG_BF16, k.stream),
               "vig_dirgate_lowrank_fwd");
      const int64_t gb = gates + T * b.H * b.Dk;
      if (whole(b)) {
        check_rc(vig_gla_slab_fwd(k.at(z), k.at(z + b.H * b.Dk), k.at(z + 2 * b.H * b.Dk), k.at(gates), k.at(gb), nullptr, k.at(o), (int)B,
                                  b.H, (int)L, b.Dk, b.Dv, sqk, sqk, sv, 0, 0, scale, 0.25f, VIG_BF16, VIG_BF16, k.stream),
                 "vig_gla_slab_fwd");
      } else {
        check_rc(vig_split_heads_fwd(k.at(z), k.at(q), k.at(kk), k.at(v), (int)B, (int)L, b.H, b.Dk, b.Dv, ld, VIG_BF16, k.stream),
                 "vig_split_heads_fwd");
        check_rc(vig_gla_bidir_fwd(k.at(q), k.at(kk), k.at(v), k.at(gates), k.at(gb), k.at(o), k.at(ws), gla_ws, (int)B, b.H, (int)L, b.Dk,
                                   b.Dv, scale, 0.25f, VIG_BF16, VIG_BF16, k.stream),
                 "vig_gla_bidir_fwd");
      }
    }
    const int64_t next = hidden == res0 ? res1 : res0;
    residual = next;
    const int64_t width = b.w_down.size(1);
    if (one_middle(b)) {
      check_rc(vig_locality_blend_swiglu_fwd(k.at(o), k.at(xs), k.at(z + n0), f32(b.gn), f32(b.ln), b.w_o.data_ptr(), k.at(hidden), f32(b.norm2),
                                             b.w_gate.data_ptr(), k.at(next), k.at(mid), (int)B, b.H, (int)L, b.Dv, (int)C, (int)width, ld,
                                             (float)b.eps, b.out_act, (float)b.eps2, k.stream),
               "vig_locality_blend_swiglu_fwd");
    } else {
      if (b.Dv == 64 && (C == 384 || C == 192)) {
        check_rc(vig_locality_blend_linear_fwd(k.at(o), k.at(xs), k.at(z + n0), f32(b.gn), f32(b.ln), b.w_o.data_ptr(), k.at(branch1), (int)B,
                                               b.H, (int)L, b.Dv, (int)C, ld, (float)b.eps, b.out_act, VIG_BF16, k.stream),
                 "vig_locality_blend_linear_fwd");
      } else {
        check_rc(vig_locality_blend_fwd(k.at(o), k.at(xs), k.at(z + n0), f32(b.gn), f32(b.ln), k.at(y), (int)B, b.H, (int)L, b.Dv, ld,
                                        (float)b.eps, b.out_act, VIG_BF16, k.stream),
                 "vig_locality_blend_fwd");
        k.linear(y, b.w_o, Tensor(), branch1, T);
      }
      const bool with_norm = swiglu_kernel && vig_norm_swiglu_preferred(T, (int)C, (int)width);
      if (!with_norm) k.norm(branch1, hidden, b.norm2, b.eps2, false, y, next, T);
      if (with_norm) {
        check_rc(vig_norm_swiglu_fwd(k.at(branch1), k.at(hidden), f32(b.norm2), b.w_gate.data_ptr(), k.at(next), k.at(mid), T, (int)C, (int)width,
                                     (float)b.eps2, k.stream),
                 "vig_norm_swiglu_fwd");
      } else if (swiglu_kernel) {
        check_rc(vig_linear_swiglu_fwd(k.at(y), b.w_gate.data_ptr(), k.at(mid), T, (int)C, (int)width, VIG_BF16, k.stream),
                 "vig_linear_swiglu_fwd");
      } else {
        k.linear(y, b.w_gate, Tensor(), wide, T);
        check_rc(vig_swiglu_fwd(k.at(wide), k.at(mid), T, (int)width, VIG_BF16, k.stream), "vig_swiglu_fwd");
      }
    }
    normed = i + 1 < p.blocks.size() && vig_linear_norm_preferred(T, (int)C, (int)width);
    if (normed) {
      const Block& after = p.blocks[i + 1];
      const int64_t sum = residual == res0 ? res1 : res0;
      check_rc(vig_linear_norm_fwd(k.at(mid), b.w_down.data_ptr(), k.at(residual), f32(after.norm1), k.at(y), k.at(sum), T, (int)C, (int)width,
                                   (float)after.eps1, k.stream),
               "vig_linear_norm_fwd");
      residual = sum;
    } else {
      k.linear(mid, b.w_down, Tensor(), branch0, T);
    }
  }
  check_rc(vig_rmsnorm_pool_fwd(k.at(branch0), k.at(residual), f32(p.norm), k.at(pooled), k.at(part), pool_ws, (int)B, (int)L, (int)C,
                                (float)p.norm_eps, k.stream),
           "vig_rmsnorm_pool_fwd");
  Tensor logits = at::empty({B, classes}, images.options());
  if (classes % 8 == 0 && vig_linear_preferred(B, (int)classes, (int)C)) {
    check_rc(vig_linear_fwd(k.at(pooled), C, p.head_w.data_ptr(), p.head_b.defined() ? p.head_b.data_ptr() : nullptr, logits.data_ptr(),
                            classes, B, (int)classes, (int)C, k.stream),
             "vig_linear_fwd");
  } else if (p.head_b.defined()) {
    at::addmm_out(logits, p.head_b, k.rows(pooled, B, C), p.head_w.t());
  } else {
    at::mm_out(logits, k.rows(pooled, B, C), p.head_w.t());
  }
  return logits;
}

bool usable(const Tensor& t, const c10::Device& dev, at::ScalarType type) {
  return !t.defined() || (plain(t, dev) && t.scalar_type() == type);
}

}  // namespace

// Adds what has to stay as it is of a module and its children: their places in the tree, every parameter, and the entries of the
// module's own dictionary that `settings` (type or module -> names) lists; false where a name of `absent` (type -> name) is there.
bool collect(Plan& p, PyObject* module, PyObject* settings, PyObject* absent, std::vector<PyObject*>& seen) {
  if (std::find(seen.begin(), seen.end(), module) != seen.end()) return true;
  seen.push_back(module);
  PyObject* own = PyObject_GenericGetDict(module, nullptr);
  if (!own) throw python_error();
  const Ref hold(own);
  Py_DECREF(own);
  PyObject *children = PyDict_GetItemString(own, "_modules"), *params = PyDict_GetItemString(own, "_parameters");
  if (!children || !params || !PyDict_Check(children) || !PyDict_Check(params)) return false;
  PyObject *key, *value, *type = reinterpret_cast<PyObject*>(Py_TYPE(module));
  PyObject* names = PyDict_GetItemWithError(settings, type);
  if (!names) names = PyDict_GetItemWithError(settings, module);
  if (names)
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(names); ++i) {
      PyObject* v = PyDict_GetItemWithError(own, PyTuple_GET_ITEM(names, i));
      p.entries.push_back({Ref(own), Ref(PyTuple_GET_ITEM(names, i)), Ref(v)});
    }
  if (PyObject* name = PyDict_GetItemWithError(absent, type)) {
    if (PyDict_GetItemWithError(own, name)) return false;
    p.entries.push_back({Ref(own), Ref(name), Ref(nullptr)});
  }
  for (Py_ssize_t at = 0; PyDict_Next(params, &at, &key, &value);) {
    p.entries.push_back({Ref(params), Ref(key), Ref(value)});
    if (value == Py_None) continue;
    const Tensor t = tensor_arg(value);
    if (!t.defined() || t.unsafeGetTensorImpl()->is_python_dispatch() || t.scalar_type() != at::kBFloat16) return false;
    p.watched.push_back({t, t.storage(), t.data_ptr(), (uint32_t)t._version(), t.scalar_type()});
  }
  for (Py_ssize_t at = 0; PyDict_Next(children, &at, &key, &value);) {
    p.entries.push_back({Ref(children), Ref(key), Ref(value)});
    if (value != Py_None && !collect(p, value, settings, absent, seen)) return false;
  }
  return true;
}

// make_plan(model, settings, absent, called, stem, blocks [tuple], tail) -> capsule, or None where a tensor is not what the kernels take.
// called: the modules that are called as modules, and tables; a hook on one of them (or an entry in a table, or an overridden
// forward) sends the call through the modules
PyObject* make_plan(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 7, "make_plan takes 7 arguments");
  auto p = std::make_unique<Plan>();
  if (!collect(*p, a[0], a[1], a[2], p->modules)) Py_RETURN_NONE;
  std::sort(p->modules.begin(), p->modules.end());
  const Ref forward(PyUnicode_InternFromString("forward")), compiled(PyUnicode_InternFromString("_compiled_call_impl"));
  Py_DECREF(forward.o), Py_DECREF(compiled.o);
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[3]); ++i) {
    PyObject* m = PyList_GET_ITEM(a[3], i);
    if (PyDict_Check(m)) {
      p->empty.emplace_back(m);
      continue;
    }
    PyObject* own = PyObject_GenericGetDict(m, nullptr);
    if (!own) throw python_error();
    const Ref hold(own);
    Py_DECREF(own);
    for (const char* table : {"_forward_hooks", "_forward_pre_hooks"}) p->empty.emplace_back(PyDict_GetItemString(own, table));
    for (PyObject* name : {forward.o, compiled.o}) p->entries.push_back({Ref(own), Ref(name), Ref(nullptr)});
  }
  if (!still_valid(*p)) Py_RETURN_NONE;
  a += 1;
  Reader s{a[3]};
  Stem& st = p->stem;
  st.w1 = s.tensor(), st.b1 = s.tensor(), st.ln1w = s.tensor(), st.ln1b = s.tensor(), st.eps1 = s.real(), st.w2 = s.tensor(),
  st.b2 = s.tensor(), st.ln2w = s.tensor(), st.ln2b = s.tensor(), st.eps2 = s.real(), st.pos = s.tensor(), st.KH = s.integer(),
  st.KW = s.integer(), st.gh = s.integer(), st.gw = s.integer();
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[4]); ++i) {
    Reader r{PyList_GET_ITEM(a[4], i)};
    Block b;
    b.norm1 = r.tensor(), b.eps1 = r.real(), b.conv_w = r.tensor(), b.conv_b = r.tensor(), b.act = r.integer(), b.w_in = r.tensor(),
    b.b_in = r.tensor(), b.H = r.integer(), b.Dk = r.integer(), b.Dv = r.integer(), b.w_up = r.tensor(), b.b_up = r.tensor(),
    b.inv_norm = 1.0 / r.real(), b.clamp = r.real(), b.gn = r.tensor(), b.ln = r.tensor(), b.eps = r.real(), b.out_act = r.integer(),
    b.w_o = r.tensor(), b.norm2 = r.tensor(), b.eps2 = r.real(), b.w_gate = r.tensor(), b.w_down = r.tensor();
    p->blocks.push_back(std::move(b));
  }
  Reader t{a[5]};
  p->norm = t.tensor(), p->norm_eps = t.real(), p->head_w = t.tensor(), p->head_b = t.tensor();
  if (!st.w1.defined() || !st.w1.is_cuda() || p->blocks.empty()) Py_RETURN_NONE;
  const auto dev = st.w1.device();
  bool ok = true;
  for (const Tensor* x : {&st.w1, &st.w2, &st.pos, &p->head_w, &p->head_b}) ok = ok && usable(*x, dev, at::kBFloat16);
  for (const Tensor* x : {&st.b1, &st.ln1w, &st.ln1b, &st.b2, &st.ln2w, &st.ln2b, &p->norm}) ok = ok && usable(*x, dev, at::kFloat);
  for (const auto& b : p->blocks) {
    for (const Tensor* x : {&b.w_in, &b.b_in, &b.w_up, &b.b_up, &b.w_o, &b.w_gate, &b.w_down}) ok = ok && usable(*x, dev, at::kBFloat16);
    for (const Tensor* x : {&b.norm1, &b.conv_w, &b.conv_b, &b.gn, &b.ln, &b.norm2}) ok = ok && usable(*x, dev, at::kFloat);
  }
  // shapes: the walk lays its buffers out by the stem's width and each block's heads, and the kernels take sizes on trust
  const auto is = [](const Tensor& t, std::initializer_list<int64_t> shape) { return t.defined() && t.sizes() == at::IntArrayRef(shape); };
  const auto has = [](const Tensor& t, int64_t n) { return t.defined() && t.numel() == n; };
  const auto fits = [&](const Tensor& t, int64_t n) { return !t.defined() || t.numel() == n; };
  const int64_t half = st.w1.size(0), C = st.w2.defined() ? st.w2.size(0) : 0;
  ok = ok && is(st.w2, {C, 3, 3, half}) && fits(st.b1, half) && has(st.ln1w, half) && has(st.ln1b, half) && fits(st.b2, C) &&
       has(st.ln2w, C) && has(st.ln2b, C) && is(st.pos, {1, (int64_t)st.gh * st.gw, C}) && has(p->norm, C) && p->head_w.defined() &&
       p->head_w.dim() == 2 && is(p->head_w, {p->head_w.size(0), C}) && fits(p->head_b, p->head_w.size(0));
  for (const auto& b : p->blocks) {
    const int64_t K = (int64_t)b.H * b.Dk, V = (int64_t)b.H * b.Dv, n = 2 * K + 2 * V + 16, nz = (n + 127) / 128 * 128;
    const int64_t I = b.w_down.defined() && b.w_down.dim() == 2 ? b.w_down.size(1) : 0;
    ok = ok && V == C && I > 0 && I % 8 == 0 && has(b.norm1, C) && has(b.conv_w, C * 9) && fits(b.conv_b, C) && is(b.w_in, {nz, C}) &&
         has(b.b_in, nz) && is(b.w_up, {2 * K, 16}) && has(b.b_up, 2 * K) && has(b.gn, b.Dv) && has(b.ln, b.Dv) && is(b.w_o, {C, V}) &&
         has(b.norm2, C) && is(b.w_gate, {2 * I, C}) && is(b.w_down, {C, I});
  }
  if (!ok) Py_RETURN_NONE;
  return PyCapsule_New(p.release(), kPlanName, [](PyObject* cap) { free_plan(cap); });
  END_HANDLE_TH_ERRORS
}

// plan_describes(plan, modules [list]) -> whether one of them is the plan's model or part of it
PyObject* plan_describes(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 2 && PyList_Check(a[1]), "plan_describes takes a plan and a list");
  const auto* p = static_cast<const Plan*>(PyCapsule_GetPointer(a[0], kPlanName));
  if (!p) return nullptr;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[1]); ++i)
    if (std::binary_search(p->modules.begin(), p->modules.end(), PyList_GET_ITEM(a[1], i))) Py_RETURN_TRUE;
  Py_RETURN_FALSE;
  END_HANDLE_TH_ERRORS
}

// run_plan(plan, images) -> logits; None for images the plan does not take, False when the model has changed since
PyObject* run_plan(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 2, "run_plan takes 2 arguments");
  const auto* p = static_cast<const Plan*>(PyCapsule_GetPointer(a[0], kPlanName));
  if (!p) return nullptr;
  if (!is_tensor(a[1])) Py_RETURN_NONE;
  const Tensor images = THPVariable_Unpack(a[1]);
  const Stem& st = p->stem;
  if (images.dim() != 4 || !plain(images, st.w1.device()) || images.scalar_type() != at::kBFloat16 || images.numel() == 0) Py_RETURN_NONE;
  if (at::autocast::is_autocast_enabled(at::kCUDA) || observed()) Py_RETURN_NONE;
  const int64_t B = images.size(0), S = images.size(2), W = images.size(3), half = st.w1.size(0);
  const int64_t oh1 = (S + 2 - st.KH) / 8 + 1, ow1 = (W + 2 - st.KW) / 8 + 1;
  // the stem's shape, and the grid the position table is for
  if (B > 65535 || images.size(1) * st.KH != 27 || st.KW > 16 || (W > 248 && st.KW > 9) || S + 2 < st.KH || W % 8 || W + 2 < st.KW || half % 32 || half < 64 || (half > 256 && half != 384) ||
      (oh1 + 1) / 2 != st.gh || (ow1 + 1) / 2 != st.gw || B * oh1 * ow1 > 0x7fffffff - 8192)
    Py_RETURN_NONE;
  if (!still_valid(*p)) Py_RETURN_FALSE;
  const at::NoGradGuard no_grad;
  const c10::DeviceGuard guard(images.device());
  return THPVariable_Wrap(run(*p, images));
  END_HANDLE_TH_ERRORS
}

}  // namespace vig_host
