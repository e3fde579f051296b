// The recorded (training) forward of a ViG block as two autograd nodes over the C ABI: the token mixer with the norm in front
// of it, and the SwiGLU MLP with its own (classification/models/vig.py:530-618; training branch :354-426).  Two, because
// stochastic depth acts on each branch between them.
//
// As separate modules the block was bound by what lay between its products: under autocast the fp32 residual stream was cast
// and re-cast around every norm, the four projections of the same rows ran as four products forward and their input gradients
// as four products and three additions, each weight gradient was rounded to bf16 and cast back, and bias gradients were
// reductions of their own.  Here
//   - the norms read and write the stream in its type and the branch in the products' type (vig_rmsnorm_mixed_fwd / _bwd);
//   - q/k/v, gate and low-rank projection are one product over stacked weights (rows padded to a multiple of 128: 35 instead of
//     62 us at 25088 x 384), their gradients gather into one matrix whose rows the kernels write in place, and one product
//     returns the input gradient, added to the local branch's in fp32 before it is rounded;
//   - weight and bias gradients leave vig_linear_bwd_weight_many as fp32, a node's layers together;
//   - the up-projection of the gates and its input gradient run inside the gate kernels (bf16), and the depthwise
//     convolution's three gradients are one kernel.
// ViG-S, B 128 at 224 px under bf16 autocast, forward and backward on one MI355X: 23.7 -> 9.9 ms.
#include <ATen/autocast_mode.h>

#include <torch/csrc/autograd/autograd.h>

#include "host_calls.h"

namespace vig_host {

namespace {

constexpr int64_t kRank = 16;  // the low-rank width the gate kernels are built for

struct Mix {
  int64_t B, L, C, h, w, H, Dk, Dv, rows, K, V, n0, n1, n2, nz;  // n0 | n1 | n2: ends of the q/k/v, gate and low-rank columns
  bool act, out_act, bf16;
  double norm_eps, eps, inv_norm, clamp;
  std::vector<int64_t> ints() const { return {B, L, h, w, H, Dk, Dv, act, out_act, bf16}; }
  std::vector<double> reals() const { return {norm_eps, eps, inv_norm, clamp}; }
  static Mix from(const std::vector<int64_t>& i, const std::vector<double>& d) {
    Mix m;
    m.B = i[0], m.L = i[1], m.h = i[2], m.w = i[3], m.H = i[4], m.Dk = i[5], m.Dv = i[6], m.act = i[7], m.out_act = i[8],
    m.bf16 = i[9];
    m.norm_eps = d[0], m.eps = d[1], m.inv_norm = d[2], m.clamp = d[3];
    m.rows = m.B * m.L, m.K = m.H * m.Dk, m.V = m.H * m.Dv, m.C = m.V;
    m.n0 = 2 * m.K + m.V, m.n1 = m.n0 + m.V, m.n2 = m.n1 + kRank, m.nz = (m.n2 + 127) / 128 * 128;
    return m;
  }
  // whether the op reads q, k and v out of the projection's rows and writes their gradients into those of its gradient: wherever its kernels can, the passes
  // that split and gather them cost more at any size (gla_backward_mfma.hip)
  bool in_place() const { return bf16 && Dv == 64 && Dk >= 32 && L <= 256 && nz <= (1 << 20); }
  at::ScalarType type() const { return bf16 ? at::kBFloat16 : at::kFloat; }
  int code() const { return bf16 ? VIG_BF16 : VIG_F32; }
};

at::ScalarType scalar_type(bool bf16) { return bf16 ? at::kBFloat16 : at::kFloat; }

void* at_elem(const Tensor& t, int64_t i) { return static_cast<char*>(t.data_ptr()) + i * t.element_size(); }
float* fptr(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }

// The weights of a step in one buffer, filled by one launch: pieces of whole 16-byte units, addressed by offset.
struct Packer {
  int64_t size = 0;
  std::vector<const void*> src;
  std::vector<int64_t> off;
  std::vector<int> n, cols, sd;
  int64_t add(const Tensor& t, int64_t count, int64_t transposed_cols = 0, bool align = true) {
    if (align) size = (size + 63) / 64 * 64;
    const int64_t at = size;
    src.push_back(t.defined() ? t.data_ptr() : nullptr);
    sd.push_back(t.defined() ? dtype_code(t) : VIG_F32);
    off.push_back(at), n.push_back((int)count), cols.push_back((int)transposed_cols);
    size += count;
    return at;
  }
  Tensor run(at::ScalarType type, const Tensor& like) const {
    if (src.empty()) return Tensor();
    Tensor buf = at::empty({size}, like.options().dtype(type));
    std::vector<void*> dst;
    for (auto o : off) dst.push_back(at_elem(buf, o));
    const std::vector<int> dd(src.size(), dtype_code(buf));
    check_rc(vig_cast_many(src.data(), dst.data(), n.data(), cols.data(), sd.data(), dd.data(), (int)src.size(), stream_of(like)),
             "vig_cast_many");
    return buf;
  }
};

Tensor matrix(const Tensor& buf, int64_t off, int64_t rows, int64_t cols) {
  return buf.as_strided({rows, cols}, {cols, 1}, buf.storage_offset() + off);
}

bool aligned(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// out = A B^T (+ bias) (+ add) of fp32 rows, A [M, K] or its transpose lying as rows, B [N, K] or its transpose, on the matrix cores;
// false where the library's product is to be taken.
// Where the line lies: a call costs 4 us of host time here and 22 us there, and products of up to about 5e9 multiply-adds take 0.4 to
// 1.24 of the library's time on the device (us, here / library; layer, input gradient, weight gradient with column sums): 400 x 2048 x 384 10 / 10, 18 / 17, 18 / 22;
// 1960 x 768 x 768 28 / 26, 30 / 30, 34 / 42; 8100 x 192 x 512 21 / 17, 24 / 30, 29 / 71; 8100 x 768 x 768 87 / 80, 85 / 90, 106 / 117; beyond,
// 8100 x 2048 x 384 117 / 103, 106 / 110, 146 / 121.  Training passes (ms, line here / library alone): 32 images of 224 px, ViG-T
// 7.9 / 10.1; 30, ViG-S 13.3 / 15.0 (line at 2.5e9: 14.2; at 9e9: 13.5).
bool matmul_f32(const Tensor& a, bool a_across, const Tensor& b, bool b_across, const float* bias, const Tensor& add, Tensor& out,
                float* a_sums = nullptr) {
  const int64_t M = a.size(a_across), K = a.size(!a_across), N = b.size(b_across);
  if ((double)M * N * K > 5e9 || !aligned(a) || !aligned(b) || a.stride(1) != 1 || b.stride(1) != 1) return false;
  const auto ld = [](const Tensor& t) { return t.size(0) == 1 ? t.size(1) : t.stride(0); };  // (a single row's stride says nothing)
  const size_t need = vig_matmul_f32_workspace(M, (int)N, K);
  const Tensor ws = need ? bytes_like(need, a) : Tensor();
  const int rc = vig_matmul_f32(fptr(a), ld(a), a_across, fptr(b), ld(b), b_across, bias, add.defined() ? fptr(add) : nullptr,
                                add.defined() ? ld(add) : 0, fptr(out), ld(out), a_sums, M, (int)N, K,
                                need ? ws.data_ptr() : nullptr, need, stream_of(a));
  if (rc == VIG_ENOTSUP) return false;
  check_rc(rc, "vig_matmul_f32");
  return true;
}

// The sums over partial rows that a node's kernels leave, one launch at its end; what is read and written then stays until it is out.
// (Whatever is handed on, cast or viewed has to wait for run().)  Twelve blocks: 24 or 48 launches fewer, of 4.7 us on the device and 3.5 of host time.
struct Sums {
  vig_sum_jobs jobs{};
  std::vector<Tensor> held;
  void run(const Tensor& like) {
    if (jobs.count) check_rc(vig_sum_jobs_run(&jobs, stream_of(like)), "vig_sum_jobs_run");
    held.clear();
  }
};

// Weight gradients dy^T x in fp32 (and the column sums of dy) of a node's layers; rows of both may lie in wider matrices.  Those of
// bf16 rows are gathered and go out together (run), as many as the library takes at once; the tensors handed out are filled with the
// node's sums.
struct WeightGrads {
  static constexpr int kMost = 4;
  // Past this the partial tiles are added up at once, by a launch of their own, while the caches hold them (ms a pass, 72 launches of sums / 48 so / 24:
  // ViG-S, 128 images of 224 px 10.86 / 10.83 / 10.91, ViG-B, 32 9.62 / 9.60 / 9.67, ViG-T, 128 6.35 / 6.31).
  static constexpr size_t kSumsAtOnce = 16 << 20;
  std::vector<Tensor> keep;
  Sums& sums;
  explicit WeightGrads(Sums& s) : sums(s) {}
  const void *dy[kMost], *x[kMost];
  long long ldy[kMost], ldx[kMost], rows = 0;
  float *dw[kMost], *db[kMost];
  int N[kMost], K[kMost], count = 0;

  Tensor add(const Tensor& d, const Tensor& in, Tensor* bias_grad) {
    const int64_t n = d.size(1), k = in.size(1);
    if (d.scalar_type() == at::kFloat) {
      Tensor w = at::empty({n, k}, d.options()), b;
      if (bias_grad) b = at::empty({n}, d.options());
      if (!matmul_f32(d, true, in, true, nullptr, Tensor(), w, bias_grad ? fptr(b) : nullptr)) {
        if (bias_grad) b = d.sum(0);
        at::mm_out(w, d.t(), in);
      }
      if (bias_grad) *bias_grad = b;
      return w;
    }
    if (count == kMost) run();
    Tensor w = at::empty({n, k}, d.options().dtype(at::kFloat));
    if (bias_grad) *bias_grad = at::empty({n}, w.options());
    dy[count] = d.data_ptr(), ldy[count] = d.stride(0), x[count] = in.data_ptr(), ldx[count] = in.stride(0);
    dw[count] = fptr(w), db[count] = bias_grad ? fptr(*bias_grad) : nullptr, N[count] = (int)n, K[count] = (int)k;
    rows = d.size(0), ++count;
    keep.insert(keep.end(), {d, in});
    sums.held.push_back(w);
    if (bias_grad) sums.held.push_back(*bias_grad);
    return w;
  }
  void run() {
    if (!count) return;
    const size_t need = vig_linear_bwd_weight_many_workspace(rows, N, K, count);
    Tensor ws = bytes_like(need, keep[0]);
    vig_sum_jobs* const later = need > kSumsAtOnce ? nullptr : &sums.jobs;
    check_rc(vig_linear_bwd_weight_many_later(dy, ldy, x, ldx, dw, db, ws.data_ptr(), need, rows, N, K, count, later, stream_of(keep[0])),
             "vig_linear_bwd_weight_many");
    if (later) sums.held.push_back(ws);
    keep.clear(), count = 0;
  }
};

// x w^T (+ bias) for rows x [M, K] (packed ones in bf16), packed w [N, K]
Tensor product(const Tensor& x, const Tensor& w, const Tensor& bias) {
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  if (x.scalar_type() == at::kBFloat16 && vig_linear_preferred(M, (int)N, (int)K) && aligned(x) && aligned(w) &&
      (!bias.defined() || aligned(bias))) {
    Tensor y = at::empty({M, N}, x.options());
    check_rc(vig_linear_fwd(x.data_ptr(), K, w.data_ptr(), bias.defined() ? bias.data_ptr() : nullptr, y.data_ptr(), N, M, (int)N, (int)K,
                            stream_of(x)),
             "vig_linear_fwd");
    return y;
  }
  if (x.scalar_type() == at::kFloat) {
    Tensor y = at::empty({M, N}, x.options());
    if (matmul_f32(x, false, w, false, bias.defined() ? fptr(bias) : nullptr, Tensor(), y)) return y;
  }
  return bias.defined() ? at::addmm(bias, x, w.t()) : at::mm(x, w.t());
}

// dy w for packed rows dy [M, N], w [N, K]
Tensor input_grad(const Tensor& dy, const Tensor& w) {
  const int64_t M = dy.size(0), N = w.size(0), K = w.size(1);
  if (dy.scalar_type() == at::kBFloat16 && vig_linear_bwd_input_preferred(M, (int)N, (int)K) && dy.is_contiguous() && aligned(dy) && aligned(w)) {
    Tensor dx = at::empty({M, K}, dy.options());
    check_rc(vig_linear_bwd_input(dy.data_ptr(), w.data_ptr(), dx.data_ptr(), M, (int)N, (int)K, VIG_BF16, stream_of(dy)),
             "vig_linear_bwd_input");
    return dx;
  }
  if (dy.scalar_type() == at::kFloat) {
    Tensor dx = at::empty({M, K}, dy.options());
    if (matmul_f32(dy, false, w, true, nullptr, Tensor(), dx)) return dx;
  }
  return at::mm(dy, w);
}

// residual-add + RMS norm: (y, sum); without a residual the sum is x itself
std::pair<Tensor, Tensor> norm_fwd(const Tensor& x, const Tensor& residual, const float* weight, double eps, at::ScalarType type) {
  const int64_t C = x.size(-1), rows = x.numel() / C;
  Tensor y = at::empty(x.sizes(), x.options().dtype(type));
  const Tensor sum = residual.defined() ? at::empty(x.sizes(), residual.options()) : x;
  check_rc(vig_rmsnorm_mixed_fwd(x.data_ptr(), residual.defined() ? residual.data_ptr() : nullptr, weight, y.data_ptr(),
                                 residual.defined() ? sum.data_ptr() : nullptr, rows, (int)C, (float)eps, residual.defined(),
                                 dtype_code(x), dtype_code(sum), dtype_code(y), stream_of(x)),
           "vig_rmsnorm_mixed_fwd");
  return {y, sum};
}

// its backward: (gradient of the residual, gradient of the branch, gradient of the weight or none)
struct NormGrads {
  Tensor residual, branch, weight;
};
NormGrads norm_bwd(const Tensor& sum, const float* weight, const Tensor& dy, Tensor d_sum, bool narrow_branch, bool need_weight,
                   double eps, Sums& sums) {
  const int64_t C = sum.size(-1), rows = sum.numel() / C;
  if (d_sum.defined() && !plain(d_sum, sum.device())) d_sum = d_sum.clone(at::MemoryFormat::Contiguous);
  NormGrads g;
  g.residual = at::empty_like(sum);
  g.branch = narrow_branch ? at::empty(sum.sizes(), dy.options()) : g.residual;
  size_t need = 0;
  Tensor ws;
  if (need_weight) {
    g.weight = at::empty({C}, sum.options().dtype(at::kFloat));
    need = vig_rmsnorm_bwd_workspace(rows, (int)C);
    ws = bytes_like(need, sum);
    sums.held.insert(sums.held.end(), {g.weight, ws});
  }
  check_rc(vig_rmsnorm_mixed_bwd_later(sum.data_ptr(), weight, dy.data_ptr(), d_sum.defined() ? d_sum.data_ptr() : nullptr,
                                 g.residual.data_ptr(), narrow_branch ? g.branch.data_ptr() : nullptr,
                                 need_weight ? fptr(g.weight) : nullptr, need ? ws.data_ptr() : nullptr, need, rows, (int)C,
                                 (float)eps, dtype_code(sum), dtype_code(dy), &sums.jobs, stream_of(sum)),
           "vig_rmsnorm_mixed_bwd");
  return g;
}

// a gradient that arrives in the right type, as rows; zeros where none arrived
Tensor grad_rows(const Tensor& g, int64_t rows, int64_t cols, const Tensor& like, at::ScalarType type) {
  if (!g.defined()) return at::zeros({rows, cols}, like.options().dtype(type));
  Tensor r = g.contiguous();
  if (reinterpret_cast<uintptr_t>(r.data_ptr()) % 16) r = r.clone();
  return r.view({rows, cols});
}
Tensor like_param(const Tensor& grad, const Tensor& param_like, at::IntArrayRef shape) {
  return grad.defined() ? grad.view(shape).to(param_like.scalar_type()) : grad;
}

// The kernels take what they are given in the type they are given: casts are explicit here.
struct NoAutocast {
  c10::impl::ExcludeDispatchKeyGuard guard{c10::DispatchKeySet({c10::DispatchKey::AutocastCUDA})};
};

enum MixParam { kNormW, kConvW, kConvB, kQkvW, kGateW, kGateB, kLowW, kUpW, kUpB, kGNorm, kLNorm, kOutW, kMixParams };

struct MixNode : torch::autograd::Function<MixNode> {
  static variable_list forward(AutogradContext* ctx, const Tensor& branch, const std::optional<Tensor>& residual_arg,
                               const Tensor& norm_w, const Tensor& conv_w, const std::optional<Tensor>& conv_b,
                               const Tensor& qkv_w, const Tensor& gate_w, const Tensor& gate_b, const Tensor& low_w,
                               const Tensor& up_w, const Tensor& up_b, const Tensor& g_norm, const Tensor& l_norm,
                               const Tensor& out_w, const Mix& m) {
    const NoAutocast no_autocast;
    const c10::DeviceGuard guard(branch.device());
    void* const stream = stream_of(branch);
    const auto type = m.type();
    const auto opts = branch.options().dtype(type);
    const Tensor residual = residual_arg ? *residual_arg : Tensor();
    const bool same = qkv_w.scalar_type() == type, wide = qkv_w.scalar_type() == at::kFloat;
    // ---- this step's weights: stacked input projection and its bias, and what the kernels read in another type ----
    Packer p, f;
    const int64_t w_off = p.add(qkv_w, m.n0 * m.C);
    p.add(gate_w, m.V * m.C, 0, false), p.add(low_w, kRank * m.C, 0, false);
    if (m.nz > m.n2) p.add(Tensor(), (m.nz - m.n2) * m.C, 0, false);
    const int64_t b_off = p.add(Tensor(), m.n0);
    p.add(gate_b, m.V, 0, false), p.add(Tensor(), m.nz - m.n1, 0, false);
    int64_t out_off = 0, up_off = 0, upb_off = 0, upt_off = 0;
    if (!same) out_off = p.add(out_w, m.C * m.V), up_off = p.add(up_w, 2 * m.K * kRank), upb_off = p.add(up_b, 2 * m.K);
    if (m.bf16) upt_off = p.add(up_w, 2 * m.K * kRank, kRank);
    const Tensor packed = p.run(type, branch);
    Tensor small;  // the kernels' fp32 weights
    int64_t f_off[5] = {0, 0, 0, 0, 0};
    if (!wide) {
      f_off[0] = f.add(norm_w, m.C), f_off[1] = f.add(conv_w, m.C * 9), f_off[2] = f.add(g_norm, m.Dv), f_off[3] = f.add(l_norm, m.Dv);
      if (conv_b) f_off[4] = f.add(*conv_b, m.C);
      small = f.run(at::kFloat, branch);
    }
    auto f32 = [&](const Tensor& t, int i) { return wide ? fptr(t) : fptr(small) + f_off[i]; };
    const Tensor w_in = matrix(packed, w_off, m.nz, m.C);
    const Tensor b_in = packed.as_strided({m.nz}, {1}, b_off);
    const Tensor w_out = same ? out_w : matrix(packed, out_off, m.C, m.V);

    auto [y, sum] = norm_fwd(branch, residual, f32(norm_w, 0), m.norm_eps, type);
    Tensor xs = at::empty({m.B, m.L, m.C}, opts), pre;
    if (m.act) pre = at::empty_like(xs);
    check_rc(vig_dwconv3x3_fwd_pre(y.data_ptr(), f32(conv_w, 1), conv_b ? f32(*conv_b, 4) : nullptr, xs.data_ptr(),
                                   m.act ? pre.data_ptr() : nullptr, (int)m.B, (int)m.h, (int)m.w, (int)m.C, m.act, m.code(), stream),
             "vig_dwconv3x3_fwd_pre");
    const Tensor z = product(xs.view({m.rows, m.C}), w_in, b_in);
    Tensor q, k, v;  // head-major copies, where the op does not take its operands out of z
    if (!m.in_place()) {
      q = at::empty({m.B, m.H, m.L, m.Dk}, opts), k = at::empty_like(q), v = at::empty({m.B, m.H, m.L, m.Dv}, opts);
      check_rc(vig_split_heads_fwd(z.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), (int)m.B, (int)m.L, (int)m.H, (int)m.Dk,
                                   (int)m.Dv, m.nz, m.code(), stream),
               "vig_split_heads_fwd");
    }
    Tensor gates = at::empty({2 * m.B, m.H, m.L, m.Dk}, opts), gate_lin;
    if (m.bf16) {
      check_rc(vig_dirgate_lowrank_fwd(at_elem(z, m.n1), m.nz, same ? up_w.data_ptr() : at_elem(packed, up_off),
                                       same ? up_b.data_ptr() : at_elem(packed, upb_off), gates.data_ptr(), (int)m.B, (int)m.L,
                                       (int)m.H, (int)m.Dk, (int)kRank, (float)m.inv_norm, (float)m.clamp, VIG_BF16, VIG_BF16, stream),
               "vig_dirgate_lowrank_fwd");
    } else {
      gate_lin = product(z.narrow(1, m.n1, kRank), up_w, up_b);
      check_rc(vig_dirgate_fwd(gate_lin.data_ptr(), gates.data_ptr(), (int)m.B, (int)m.L, (int)m.H, (int)m.Dk, (float)m.inv_norm,
                               (float)m.clamp, VIG_F32, VIG_F32, stream),
               "vig_dirgate_fwd");
    }
    Call c{(int)m.B, (int)m.H, (int)m.L, (int)m.Dk, (int)m.Dv, m.code(), m.code(), (float)std::pow((double)m.Dk, -0.5), 0.5f};
    Tensor o;
    if (m.in_place()) {
      o = at::empty({m.B, m.H, m.L, m.Dv}, opts);
      const long long sk[3] = {m.L * m.nz, m.Dk, m.nz}, sv[3] = {m.L * m.nz, m.Dv, m.nz};
      check_rc(vig_gla_bidir_fwd_strided(z.data_ptr(), at_elem(z, m.K), at_elem(z, 2 * m.K), gates.data_ptr(), at_elem(gates, gates.numel() / 2),
                                         o.data_ptr(), c.B, c.H, c.L, c.Dk, c.Dv, sk, sk, sv, c.scale, c.out_scale, c.io, c.gd, stream),
               "vig_gla_bidir_fwd_strided");
    } else {
      check_rc(run_forward(q, k, v, gates, Tensor(), true, kDefault, c, o), "vig_gla_bidir_fwd");
    }
    Tensor blend = at::empty_like(xs);
    Tensor a;
    // At any number of tokens (us, fused / blend and product): C 192: 49 4.8 / 10.7, 1568 5.3 / 12.4, 25088 16 / 29; C 384: 49 7.7 / 11.2,
    // 1568 8.8 / 16.4, 25088 26 / 37; a single token 7.0 / 4.8.
    if (m.bf16 && m.Dv == 64 && m.V == m.C && (m.C == 384 || m.C == 192) && aligned(w_out)) {
      a = at::empty({m.B, m.L, m.C}, opts);
      check_rc(vig_locality_blend_linear_kept_fwd(o.data_ptr(), xs.data_ptr(), at_elem(z, m.n0), f32(g_norm, 2), f32(l_norm, 3),
                                                  w_out.data_ptr(), blend.data_ptr(), a.data_ptr(), (int)m.B, (int)m.H, (int)m.L, (int)m.Dv,
                                                  (int)m.C, m.nz, (float)m.eps, m.out_act, m.code(), stream),
               "vig_locality_blend_linear_kept_fwd");
    } else {
      check_rc(vig_locality_blend_fwd(o.data_ptr(), xs.data_ptr(), at_elem(z, m.n0), f32(g_norm, 2), f32(l_norm, 3), blend.data_ptr(),
                                      (int)m.B, (int)m.H, (int)m.L, (int)m.Dv, m.nz, (float)m.eps, m.out_act, m.code(), stream),
               "vig_locality_blend_fwd");
      a = product(blend.view({m.rows, m.V}), w_out, Tensor()).view({m.B, m.L, m.C});
    }

    ctx->set_materialize_grads(false);
    ctx->save_for_backward({sum, y, xs, pre, z, q, k, v, gates, gate_lin, o, blend, packed, small, norm_w, conv_w, g_norm, l_norm,
                            out_w, up_w, up_b});
    ctx->saved_data["ints"] = m.ints();
    ctx->saved_data["reals"] = m.reals();
    ctx->saved_data["at"] = std::vector<int64_t>{w_off, out_off, up_off, upb_off, upt_off, f_off[0], f_off[1], f_off[2], f_off[3],
                                                 branch.scalar_type() != sum.scalar_type(), conv_b.has_value(), residual.defined()};
    return {a, sum};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const at::NoGradGuard no_grad;
    const NoAutocast no_autocast;
    const auto s = ctx->get_saved_variables();
    const Tensor &sum = s[0], &y = s[1], &xs = s[2], &pre = s[3], &z = s[4], &q = s[5], &k = s[6], &v = s[7], &gates = s[8],
                 &gate_lin = s[9], &o = s[10], &blend = s[11], &packed = s[12], &small = s[13], &norm_w = s[14], &conv_w = s[15],
                 &g_norm = s[16], &l_norm = s[17], &out_w = s[18], &up_w = s[19], &up_b = s[20];
    const Mix m = Mix::from(ctx->saved_data["ints"].toIntVector(), ctx->saved_data["reals"].toDoubleVector());
    const auto off = ctx->saved_data["at"].toIntVector();
    const c10::DeviceGuard guard(sum.device());
    void* const stream = stream_of(sum);
    const auto type = m.type();
    const bool same = out_w.scalar_type() == type, wide = out_w.scalar_type() == at::kFloat;
    auto f32 = [&](const Tensor& t, int i) { return wide ? fptr(t) : fptr(small) + off[5 + i]; };
    const Tensor w_in = matrix(packed, off[0], m.n2, m.C);
    const Tensor w_out = same ? out_w : matrix(packed, off[1], m.C, m.V);
    // (an argument that was absent has no edge)
    auto wants = [&](int param) { return ctx->needs_input_grad(param + (off[11] ? 2 : 1) - (param > kConvB && !off[10])); };
    auto opts = xs.options();
    variable_list out(2 + kMixParams + 1);

    const Tensor da = grad_rows(grads[0], m.rows, m.C, xs, type);
    Sums sums;
    WeightGrads weights(sums);
    Tensor dw_out, dw_up, db_up, dw_in, db_in;
    if (wants(kOutW)) dw_out = weights.add(da, blend.view({m.rows, m.V}), nullptr);
    const Tensor d_blend = input_grad(da, w_out);
    // gradients of the stacked projection's columns, written in place by the three kernels that produce them
    Tensor dz = at::empty({m.rows, m.nz}, opts);
    Tensor d_o = at::empty_like(o), d_xs = at::empty({m.rows, m.C}, opts);
    Tensor d_norms = at::empty({2, m.Dv}, opts.dtype(at::kFloat));
    {
      const size_t need = vig_locality_blend_bwd_workspace((int)m.B, (int)m.L, (int)m.Dv);
      Tensor ws = bytes_like(need, sum);
      sums.held.insert(sums.held.end(), {ws, d_norms});
      check_rc(vig_locality_blend_bwd_strided_later(o.data_ptr(), xs.data_ptr(), at_elem(z, m.n0), f32(g_norm, 2), f32(l_norm, 3),
                                              d_blend.data_ptr(), d_o.data_ptr(), d_xs.data_ptr(), at_elem(dz, m.n0), fptr(d_norms),
                                              ws.data_ptr(), need, (int)m.B, (int)m.H, (int)m.L, (int)m.Dv, m.nz, m.nz,
                                              (float)m.eps, m.out_act, m.code(), &sums.jobs, stream),
               "vig_locality_blend_bwd_strided");
    }
    Tensor dg = at::empty_like(gates);
    if (m.in_place()) {
      const size_t need = vig_gla_bidir_bwd_workspace_for((int)m.B, (int)m.H, (int)m.L, (int)m.Dk, (int)m.Dv, m.code(), m.code(), 1);
      Tensor ws = bytes_like(need, sum);
      const int64_t half = gates.numel() / 2;
      check_rc(vig_gla_bidir_bwd_rows(z.data_ptr(), at_elem(z, m.K), at_elem(z, 2 * m.K), m.nz, gates.data_ptr(), at_elem(gates, half),
                                      d_o.data_ptr(), dz.data_ptr(), at_elem(dz, m.K), at_elem(dz, 2 * m.K), m.nz, dg.data_ptr(),
                                      at_elem(dg, half), ws.data_ptr(), need, (int)m.B, (int)m.H, (int)m.L, (int)m.Dk, (int)m.Dv,
                                      (float)std::pow((double)m.Dk, -0.5), 0.5f, m.code(), m.code(), stream),
               "vig_gla_bidir_bwd_rows");
    } else {
      Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
      const size_t need = vig_gla_bidir_bwd_workspace_for((int)m.B, (int)m.H, (int)m.L, (int)m.Dk, (int)m.Dv, m.code(), m.code(), 1);
      Tensor ws = bytes_like(need, sum);
      const int64_t half = gates.numel() / 2;
      check_rc(vig_gla_bidir_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), gates.data_ptr(), at_elem(gates, half), d_o.data_ptr(),
                                 dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dg.data_ptr(), at_elem(dg, half), ws.data_ptr(), need,
                                 (int)m.B, (int)m.H, (int)m.L, (int)m.Dk, (int)m.Dv, (float)std::pow((double)m.Dk, -0.5), 0.5f,
                                 m.code(), m.code(), stream),
               "vig_gla_bidir_bwd");
      check_rc(vig_split_heads_bwd_strided(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dz.data_ptr(), m.nz, (int)m.B, (int)m.L,
                                           (int)m.H, (int)m.Dk, (int)m.Dv, m.code(), stream),
               "vig_split_heads_bwd_strided");
    }
    Tensor dx = at::empty({m.rows, 2 * m.K}, opts);
    if (m.bf16) {
      check_rc(vig_dirgate_lowrank_bwd(at_elem(z, m.n1), m.nz, same ? up_w.data_ptr() : at_elem(packed, off[2]),
                                       at_elem(packed, off[4]), same ? up_b.data_ptr() : at_elem(packed, off[3]), dg.data_ptr(),
                                       dx.data_ptr(), at_elem(dz, m.n1), m.nz, (int)m.B, (int)m.L, (int)m.H, (int)m.Dk,
                                       (int)kRank, (float)m.inv_norm, (float)m.clamp, VIG_BF16, VIG_BF16, stream),
               "vig_dirgate_lowrank_bwd");
    } else {
      check_rc(vig_dirgate_bwd(gate_lin.data_ptr(), dg.data_ptr(), dx.data_ptr(), (int)m.B, (int)m.L, (int)m.H, (int)m.Dk,
                               (float)m.inv_norm, (float)m.clamp, VIG_F32, VIG_F32, stream),
               "vig_dirgate_bwd");
      Tensor d_low = dz.narrow(1, m.n1, kRank);
      if (!matmul_f32(dx, false, up_w, true, nullptr, Tensor(), d_low)) at::mm_out(d_low, dx, up_w);
    }
    const Tensor dzs = dz.narrow(1, 0, m.n2);
    if (wants(kUpW) || wants(kUpB)) dw_up = weights.add(dx, z.narrow(1, m.n1, kRank), &db_up);
    if (wants(kQkvW) || wants(kGateW) || wants(kGateB) || wants(kLowW))
      dw_in = weights.add(dzs, xs.view({m.rows, m.C}), wants(kGateB) ? &db_in : nullptr);
    weights.run();
    if (m.bf16 || !matmul_f32(dzs, false, w_in, true, nullptr, d_xs, d_xs)) at::addmm_out(d_xs, d_xs, dzs, w_in);
    const bool conv_grads = wants(kConvW) || (off[10] && wants(kConvB));
    Tensor d_y = at::empty({m.B, m.L, m.C}, opts), dw_db, ws;
    size_t need = 0;
    if (conv_grads) {
      dw_db = at::empty({m.C * 10}, opts.dtype(at::kFloat));
      need = vig_dwconv3x3_bwd_weight_workspace((int)m.B, (int)m.C);
      ws = bytes_like(need, sum);
      sums.held.insert(sums.held.end(), {dw_db, ws});
    }
    check_rc(vig_dwconv3x3_bwd_later(y.data_ptr(), d_xs.data_ptr(), m.act ? pre.data_ptr() : nullptr, f32(conv_w, 1), d_y.data_ptr(),
                               conv_grads ? fptr(dw_db) : nullptr, need ? ws.data_ptr() : nullptr, need, (int)m.B, (int)m.h,
                               (int)m.w, (int)m.C, m.code(), &sums.jobs, stream),
             "vig_dwconv3x3_bwd");
    const auto g = norm_bwd(sum, f32(norm_w, 0), d_y, grads[1], off[9], wants(kNormW), m.norm_eps, sums);
    sums.run(sum);
    if (wants(kGNorm)) out[2 + kGNorm] = like_param(d_norms.select(0, 0), g_norm, {m.Dv});
    if (wants(kLNorm)) out[2 + kLNorm] = like_param(d_norms.select(0, 1), l_norm, {m.Dv});
    out[2 + kOutW] = like_param(dw_out, out_w, {m.C, m.V});
    out[2 + kUpW] = like_param(dw_up, up_w, {2 * m.K, kRank});
    out[2 + kUpB] = like_param(db_up, up_w, {2 * m.K});
    if (dw_in.defined()) {
      out[2 + kQkvW] = like_param(dw_in.narrow(0, 0, m.n0), out_w, {m.n0, m.C});
      out[2 + kGateW] = like_param(dw_in.narrow(0, m.n0, m.V), out_w, {m.V, m.C});
      out[2 + kLowW] = like_param(dw_in.narrow(0, m.n1, kRank), out_w, {kRank, m.C});
      if (db_in.defined()) out[2 + kGateB] = like_param(db_in.narrow(0, m.n0, m.V), out_w, {m.V});
    }
    if (wants(kConvW)) out[2 + kConvW] = like_param(dw_db.narrow(0, 0, m.C * 9), conv_w, conv_w.sizes());
    if (off[10] && wants(kConvB)) out[2 + kConvB] = like_param(dw_db.narrow(0, m.C * 9, m.C), conv_w, {m.C});
    out[0] = g.branch;
    if (off[11]) out[1] = g.residual;
    out[2 + kNormW] = like_param(g.weight, norm_w, {m.C});
    return out;
  }
};

struct MlpNode : torch::autograd::Function<MlpNode> {
  static variable_list forward(AutogradContext* ctx, const Tensor& branch, const Tensor& residual, const Tensor& norm_w,
                               const Tensor& gate_w, const Tensor& down_w, double eps, bool bf16) {
    const NoAutocast no_autocast;
    const c10::DeviceGuard guard(branch.device());
    const auto type = scalar_type(bf16);
    const int64_t C = branch.size(-1), rows = branch.numel() / C, I = down_w.size(1);
    const bool same = gate_w.scalar_type() == type, wide = gate_w.scalar_type() == at::kFloat;
    Packer p, f;
    int64_t gate_off = 0, down_off = 0;
    if (!same) gate_off = p.add(gate_w, 2 * I * C), down_off = p.add(down_w, C * I);
    const Tensor packed = p.run(type, branch);
    Tensor small;
    if (!wide) f.add(norm_w, C), small = f.run(at::kFloat, branch);
    const Tensor wg = same ? gate_w : matrix(packed, gate_off, 2 * I, C), wd = same ? down_w : matrix(packed, down_off, C, I);
    auto [y, sum] = norm_fwd(branch, residual, wide ? fptr(norm_w) : fptr(small), eps, type);
    Tensor z, prod = at::empty({rows, I}, y.options());
    // At any number of tokens (us, fused / product and SwiGLU pass): C 192: 1 4.0 / 4.1, 196 4.4 / 4.6, 1568 5.2 / 7.4, 25088 27 / 36; C 384:
    // 49 5.3 / 4.8 (and a launch more), 196 5.6 / 5.7, 1568 10.6 / 12.7, 12544 37 / 66, 25088 66 / 71.
    if (type == at::kBFloat16 && (C == 384 || C == 192) && I % 32 == 0 && aligned(y) && aligned(wg)) {
      z = at::empty({rows, 2 * I}, y.options());
      check_rc(vig_linear_swiglu_kept_fwd(y.data_ptr(), wg.data_ptr(), z.data_ptr(), prod.data_ptr(), rows, (int)C, (int)I, VIG_BF16,
                                          stream_of(z)),
               "vig_linear_swiglu_kept_fwd");
    } else {
      z = product(y.view({rows, C}), wg, Tensor());
      check_rc(vig_swiglu_fwd(z.data_ptr(), prod.data_ptr(), rows, (int)I, dtype_code(z), stream_of(z)), "vig_swiglu_fwd");
    }
    const Tensor out = product(prod, wd, Tensor()).view(branch.sizes());
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({sum, y, z, prod, packed, small, norm_w, gate_w, down_w});
    ctx->saved_data["at"] = std::vector<int64_t>{gate_off, down_off, bf16, branch.scalar_type() != sum.scalar_type()};
    ctx->saved_data["eps"] = eps;
    return {out, sum};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const at::NoGradGuard no_grad;
    const NoAutocast no_autocast;
    const auto s = ctx->get_saved_variables();
    const Tensor &sum = s[0], &y = s[1], &z = s[2], &prod = s[3], &packed = s[4], &small = s[5], &norm_w = s[6], &gate_w = s[7],
                 &down_w = s[8];
    const auto off = ctx->saved_data["at"].toIntVector();
    const c10::DeviceGuard guard(sum.device());
    const auto type = scalar_type(off[2]);
    const int64_t C = sum.size(-1), rows = sum.numel() / C, I = prod.size(1);
    const bool same = gate_w.scalar_type() == type, wide = gate_w.scalar_type() == at::kFloat;
    const Tensor wg = same ? gate_w : matrix(packed, off[0], 2 * I, C), wd = same ? down_w : matrix(packed, off[1], C, I);
    variable_list out(7);
    const Tensor d_out = grad_rows(grads[0], rows, C, y, type);
    Sums sums;
    WeightGrads weights(sums);
    Tensor dw_gate, dw_down;
    if (ctx->needs_input_grad(4)) dw_down = weights.add(d_out, prod, nullptr);
    Tensor dz = at::empty_like(z);
    // At any number of tokens (us, fused / input gradient and SwiGLU pass): C 192: 1 3.5 / 6.6, 1568 5.0 / 9.2, 25088 28 / 41; C 384: 1 3.9 / 5.8,
    // 1568 8.5 / 13.7, 25088 53 / 72.
    if (type == at::kBFloat16 && d_out.scalar_type() == type && (C == 384 || C == 192) && I % 32 == 0 && d_out.is_contiguous() && aligned(d_out) && aligned(wd)) {
      check_rc(vig_linear_swiglu_bwd(d_out.data_ptr(), wd.data_ptr(), z.data_ptr(), dz.data_ptr(), rows, (int)C, (int)I, VIG_BF16,
                                     stream_of(z)),
               "vig_linear_swiglu_bwd");
    } else {
      const Tensor d_prod = input_grad(d_out, wd);
      check_rc(vig_swiglu_bwd(z.data_ptr(), d_prod.data_ptr(), dz.data_ptr(), rows, (int)I, dtype_code(z), stream_of(z)),
               "vig_swiglu_bwd");
    }
    if (ctx->needs_input_grad(3)) dw_gate = weights.add(dz, y.view({rows, C}), nullptr);
    weights.run();
    const Tensor d_y = type == at::kFloat ? input_grad(dz, wg) : at::mm(dz, wg);
    const auto g = norm_bwd(sum, wide ? fptr(norm_w) : fptr(small), d_y, grads[1], off[3], ctx->needs_input_grad(2),
                            ctx->saved_data["eps"].toDouble(), sums);
    sums.run(sum);
    out[3] = like_param(dw_gate, gate_w, {2 * I, C});
    out[4] = like_param(dw_down, down_w, {C, I});
    out[0] = g.branch, out[1] = g.residual;
    out[2] = like_param(g.weight, norm_w, {C});
    return out;
  }
};

// A layer norm of the patch embedding with the bias of the convolution in front and, if asked for, the SiLU behind it.  x [B, C, h, w] in
// channels-last memory.
struct StemNormNode : torch::autograd::Function<StemNormNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const std::optional<Tensor>& pre_arg, const Tensor& weight, const Tensor& bias,
                        double eps, bool silu, bool narrow) {
    const c10::DeviceGuard guard(x.device());
    const Tensor pre = pre_arg ? *pre_arg : Tensor();
    const int64_t C = x.size(1), rows = x.numel() / C;
    Tensor y = at::empty(x.sizes(), x.options().dtype(scalar_type(narrow)).memory_format(at::MemoryFormat::ChannelsLast));
    check_rc(vig_stem_norm_fwd(x.data_ptr(), pre.defined() ? fptr(pre) : nullptr, fptr(weight), fptr(bias), y.data_ptr(), rows, (int)C, (float)eps,
                               silu, dtype_code(x), dtype_code(y), stream_of(x)),
             "vig_stem_norm_fwd");
    ctx->save_for_backward({x, pre, weight, bias});
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["silu"] = silu;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const NoAutocast no_autocast;
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &pre = s[1], &weight = s[2], &bias = s[3];
    const double eps = ctx->saved_data["eps"].toDouble();
    const bool silu = ctx->saved_data["silu"].toBool();
    variable_list out(7);
    // (an absent bias has no edge)
    const int first = pre.defined() ? 2 : 1;
    const bool wants[4] = {ctx->needs_input_grad(0), pre.defined() && ctx->needs_input_grad(1), ctx->needs_input_grad(first),
                           ctx->needs_input_grad(first + 1)};
    if (at::GradMode::is_enabled()) {  // a graph of the gradients is wanted: the same from operators that have one
      Tensor z = x.permute({0, 2, 3, 1}).to(at::kFloat);
      if (pre.defined()) z = z + pre;
      z = at::layer_norm(z, {x.size(1)}, weight, bias, eps);
      if (silu) z = at::silu(z);
      z = z.to(grads[0].scalar_type()).permute({0, 3, 1, 2});
      variable_list in;
      for (int i = 0; i < 4; ++i)
        if (wants[i]) in.push_back(s[i]);
      const auto g = torch::autograd::grad({z}, in, {grads[0]}, true, true, true);
      for (int i = 0, at = 0; i < 4; ++i)
        if (wants[i]) out[i] = g[at++];
      return out;
    }
    const c10::DeviceGuard guard(x.device());
    Tensor dy = grads[0].contiguous(at::MemoryFormat::ChannelsLast);
    if (!dy.permute({0, 2, 3, 1}).is_contiguous() || !aligned(dy)) dy = dy.permute({0, 2, 3, 1}).clone(at::MemoryFormat::Contiguous).permute({0, 3, 1, 2});
    const int64_t C = x.size(1), rows = x.numel() / C;
    Tensor dx, dparams = at::empty({3, C}, weight.options());
    if (wants[0]) dx = at::empty_like(x);
    const size_t need = vig_stem_norm_bwd_workspace(rows, (int)C);
    Tensor ws = bytes_like(need, x);
    check_rc(vig_stem_norm_bwd(x.data_ptr(), pre.defined() ? fptr(pre) : nullptr, fptr(weight), fptr(bias), dy.data_ptr(),
                               dx.defined() ? dx.data_ptr() : nullptr, fptr(dparams), ws.data_ptr(), need, rows, (int)C, (float)eps, silu,
                               dtype_code(x), dtype_code(dy), stream_of(x)),
             "vig_stem_norm_bwd");
    out[0] = dx;
    if (wants[1]) out[1] = dparams.select(0, 2);
    if (wants[2]) out[2] = dparams.select(0, 0);
    if (wants[3]) out[3] = dparams.select(0, 1);
    return out;
  }
};

// A convolution of the patch embedding without its bias: the library's kernel forward, torch's operator for the gradients.  x bf16, as it arrives
// ([B, Cin, H, W] in memory) in front of the first one, channels-last for the second; w bf16 in channels-last memory.
struct StemConvNode : torch::autograd::Function<StemConvNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, int64_t stride) {
    const NoAutocast no_autocast;
    const c10::DeviceGuard guard(x.device());
    const int B = (int)x.size(0), Cin = (int)x.size(1), H = (int)x.size(2), W = (int)x.size(3), Cout = (int)w.size(0), KH = (int)w.size(2),
              KW = (int)w.size(3);
    Tensor y = at::empty({B, Cout, (H + 2 - KH) / stride + 1, (W + 2 - KW) / stride + 1}, x.options().memory_format(at::MemoryFormat::ChannelsLast));
    if (stride == 2) {
      check_rc(vig_conv3x3s2_fwd(x.data_ptr(), w.data_ptr(), y.data_ptr(), B, H, W, Cin, Cout, stream_of(x)), "vig_conv3x3s2_fwd");
    } else {
      Tensor packed = at::zeros({Cout, Cin, KH, 16}, w.options().memory_format(at::MemoryFormat::Contiguous));
      packed.narrow(3, 0, KW).copy_(w);
      check_rc(vig_patch_conv_fwd(x.data_ptr(), packed.data_ptr(), y.data_ptr(), B, Cin, H, W, KH, KW, (int)stride, 1, Cout, VIG_BF16, stream_of(x)),
               "vig_patch_conv_fwd");
    }
    ctx->save_for_backward({x, w});
    ctx->saved_data["stride"] = stride;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const NoAutocast no_autocast;
    const auto s = ctx->get_saved_variables();
    const int64_t stride = ctx->saved_data["stride"].toInt();
    const auto g = at::convolution_backward(grads[0], s[0], s[1], c10::nullopt, {stride, stride}, {1, 1}, {1, 1}, false, {0, 0}, 1,
                                            {ctx->needs_input_grad(0), ctx->needs_input_grad(1), false});
    return {std::get<0>(g), std::get<1>(g), Tensor()};
  }
};

// Whether branch and residual are rows the nodes take and the weights share one usable type; sets the products' type.
bool stream_ok(const Tensor& branch, const Tensor& residual, const Tensor* const* params, int n, bool& bf16) {
  if (!branch.defined() || !branch.is_cuda() || branch.dim() != 3 || branch.numel() == 0 || observed()) return false;
  const auto dev = branch.device();
  if (!plain(branch, dev) || dtype_code(branch) < 0) return false;
  if (residual.defined() && (!plain(residual, dev) || residual.sizes() != branch.sizes() || dtype_code(residual) < 0)) return false;
  const auto sum = residual.defined() ? residual.scalar_type() : branch.scalar_type();
  const auto param = params[0]->scalar_type();
  at::ScalarType type = param;
  if (at::autocast::is_autocast_enabled(at::kCUDA)) {
    type = at::autocast::get_autocast_dtype(at::kCUDA);
    if (type != at::kBFloat16) return false;
  }
  if ((type != at::kBFloat16 && type != at::kFloat) || (param != type && param != at::kFloat)) return false;
  bf16 = type == at::kBFloat16;
  for (int i = 0; i < n; ++i)
    if (params[i] && (!plain(*params[i], dev) || params[i]->scalar_type() != param)) return false;
  const int64_t C = branch.size(2), rows = branch.size(0) * branch.size(1);
  if (C % 8 || C > 1024 || rows > 0x7fffffff - 8192) return false;
  return (branch.scalar_type() == type && sum == type) || (sum == at::kFloat && bf16);
}

bool is_shape(const Tensor& t, std::initializer_list<int64_t> shape) { return t.sizes() == at::IntArrayRef(shape); }

}  // namespace

// block_mix(branch, residual or None, norm, conv weight, conv bias or None, qkv, gate weight, gate bias, low-rank, up weight,
// up bias, global norm, local norm, out, h, w, heads, key width, value width, conv SiLU, output SiLU, norm eps, eps,
// gate normaliser, clamp or None) -> (mixer output, residual stream), or None for a call the node does not take
PyObject* block_mix(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 25, "block_mix takes 25 arguments");
  for (int i = 0; i < 14; ++i)
    if (!is_tensor(a[i]) && !((i == 1 || i == 4) && a[i] == Py_None)) Py_RETURN_NONE;
  const Tensor& branch = THPVariable_Unpack(a[0]);
  const Tensor residual = tensor_arg(a[1]), conv_b = tensor_arg(a[4]);
  const Tensor* params[kMixParams];
  for (int i = 0; i < kMixParams; ++i) params[i] = i == kConvB ? (conv_b.defined() ? &conv_b : nullptr) : &THPVariable_Unpack(a[2 + i]);
  bool bf16;
  if (!stream_ok(branch, residual, params, kMixParams, bf16)) Py_RETURN_NONE;
  const int64_t h = PyLong_AsLong(a[14]), w = PyLong_AsLong(a[15]), H = PyLong_AsLong(a[16]), Dk = PyLong_AsLong(a[17]),
                Dv = PyLong_AsLong(a[18]);
  const bool act = PyObject_IsTrue(a[19]), out_act = PyObject_IsTrue(a[20]);
  const double norm_eps = PyFloat_AsDouble(a[21]), eps = PyFloat_AsDouble(a[22]), normalizer = PyFloat_AsDouble(a[23]);
  const double clamp = a[24] == Py_None ? std::nan("") : PyFloat_AsDouble(a[24]);
  if (PyErr_Occurred()) return nullptr;
  const int64_t B = branch.size(0), L = branch.size(1), C = branch.size(2);
  if (H <= 0 || h <= 0 || w <= 0 || (Dk != 16 && Dk != 32 && Dk != 64) || (Dv != 32 && Dv != 64)) Py_RETURN_NONE;
  const Mix m = Mix::from({B, L, h, w, H, Dk, Dv, act, out_act, bf16}, {norm_eps, eps, 1.0 / normalizer, clamp});
  // (a grid row with its halo has to fit the stencil's tile three times)
  if (h * w != L || C != m.V || B > 65535 || (w + 2) * 64 * (bf16 ? 2 : 4) * 3 > 48 * 1024) Py_RETURN_NONE;
  if (!is_shape(*params[kNormW], {C}) || params[kConvW]->numel() != C * 9 || (conv_b.defined() && !is_shape(conv_b, {C})) ||
      !is_shape(*params[kQkvW], {m.n0, C}) || !is_shape(*params[kGateW], {m.V, C}) || !is_shape(*params[kGateB], {m.V}) ||
      !is_shape(*params[kLowW], {kRank, C}) || !is_shape(*params[kUpW], {2 * m.K, kRank}) || !is_shape(*params[kUpB], {2 * m.K}) ||
      !is_shape(*params[kGNorm], {Dv}) || !is_shape(*params[kLNorm], {Dv}) || !is_shape(*params[kOutW], {C, m.V}))
    Py_RETURN_NONE;
  const auto opt = [](const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; };
  auto r = MixNode::apply(branch, opt(residual), *params[kNormW], *params[kConvW], opt(conv_b), *params[kQkvW], *params[kGateW],
                          *params[kGateB], *params[kLowW], *params[kUpW], *params[kUpB], *params[kGNorm], *params[kLNorm],
                          *params[kOutW], m);
  return Py_BuildValue("(NN)", THPVariable_Wrap(r[0]), THPVariable_Wrap(r[1]));
  END_HANDLE_TH_ERRORS
}

// block_mlp(branch, residual, norm, gate and up weight, down weight, eps) -> (MLP output, residual stream), or None
PyObject* block_mlp(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 6, "block_mlp takes 6 arguments");
  for (int i = 0; i < 5; ++i)
    if (!is_tensor(a[i])) Py_RETURN_NONE;
  const Tensor &branch = THPVariable_Unpack(a[0]), &residual = THPVariable_Unpack(a[1]), &norm_w = THPVariable_Unpack(a[2]),
               &gate_w = THPVariable_Unpack(a[3]), &down_w = THPVariable_Unpack(a[4]);
  const Tensor* params[3] = {&norm_w, &gate_w, &down_w};
  bool bf16;
  const double eps = PyFloat_AsDouble(a[5]);
  if (PyErr_Occurred()) return nullptr;
  if (!stream_ok(branch, residual, params, 3, bf16)) Py_RETURN_NONE;
  const int64_t C = branch.size(2);
  if (down_w.dim() != 2 || down_w.size(0) != C) Py_RETURN_NONE;
  const int64_t I = down_w.size(1);
  if (I <= 0 || I % 8 || !is_shape(norm_w, {C}) || !is_shape(gate_w, {2 * I, C})) Py_RETURN_NONE;
  auto r = MlpNode::apply(branch, residual, norm_w, gate_w, down_w, eps, bf16);
  return Py_BuildValue("(NN)", THPVariable_Wrap(r[0]), THPVariable_Wrap(r[1]));
  END_HANDLE_TH_ERRORS
}

// stem_conv(x, weight, stride) -> the convolution with padding 1 and without a bias, under bf16 autocast, or None for a call the node does not take: the
// kernels' shapes (the first convolution of images three channels deep, 9 x 9 at stride 8; 3 x 3 at stride 2), as in evaluation.
// us, 128 images of 224 px, the convolution library's (the first with the layout change in front of it) / here: 192 channels 93 / 41, 384 98 / 55; a training
// pass of ViG-S under autocast 10.37 -> 10.25 ms.
PyObject* stem_conv(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 3, "stem_conv takes 3 arguments");
  if (!is_tensor(a[0]) || !is_tensor(a[1])) Py_RETURN_NONE;
  const Tensor &x = THPVariable_Unpack(a[0]), &weight = THPVariable_Unpack(a[1]);
  const int64_t stride = PyLong_AsLong(a[2]);
  if (PyErr_Occurred()) return nullptr;
  if ((stride != 2 && stride != 8) || !x.defined() || !x.is_cuda() || x.dim() != 4 || weight.dim() != 4 || x.numel() == 0 || weight.numel() == 0 || observed() ||
      !at::autocast::is_autocast_enabled(at::kCUDA) || at::autocast::get_autocast_dtype(at::kCUDA) != at::kBFloat16 ||
      c10::impl::tls_local_dispatch_key_set().included_.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
    Py_RETURN_NONE;
  for (const Tensor* t : {&x, &weight})
    if (t->unsafeGetTensorImpl()->is_python_dispatch() || t->layout() != at::kStrided || t->device() != x.device() || t->_fw_grad(0).defined() ||
        (t->scalar_type() != at::kFloat && t->scalar_type() != at::kBFloat16))
      Py_RETURN_NONE;
  const int64_t Cout = weight.size(0), Cin = weight.size(1), KH = weight.size(2), KW = weight.size(3), H = x.size(2), W = x.size(3);
  if (x.size(1) != Cin || x.numel() > 0x7fffffff || x.size(0) * Cout > 0x7fffffff / ((H / stride + 1) * (W / stride + 1)) ||
      !weight.permute({0, 2, 3, 1}).is_contiguous())
    Py_RETURN_NONE;
  if (stride == 2) {
    if (KH != 3 || KW != 3 || Cin % 32 || Cout % 8 || !x.permute({0, 2, 3, 1}).is_contiguous()) Py_RETURN_NONE;
  } else if (KW > 16 || Cin * KH != 27 || H + 2 < KH || W + 2 < KW || W % 8 || (W > 248 && KW > 9) || Cout % 32 ||
             !((Cout >= 64 && Cout <= 256) || Cout == 384) || !x.is_contiguous()) {
    Py_RETURN_NONE;
  }
  const Tensor xb = at::autocast::cached_cast(at::kBFloat16, x, at::kCUDA), wb = at::autocast::cached_cast(at::kBFloat16, weight, at::kCUDA);
  if (!aligned(xb) || !aligned(wb) || !wb.permute({0, 2, 3, 1}).is_contiguous()) Py_RETURN_NONE;
  return THPVariable_Wrap(StemConvNode::apply(xb, wb, stride));
  END_HANDLE_TH_ERRORS
}

// stem_norm(x, convolution's bias or None, weight, bias, eps, silu, last) -> the norm of the map (in the products' type, the last one in fp32), or
// None for a call the node does not take
PyObject* stem_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 7, "stem_norm takes 7 arguments");
  for (int i = 0; i < 4; ++i)
    if (!is_tensor(a[i]) && !(i == 1 && a[i] == Py_None)) Py_RETURN_NONE;
  const Tensor &x = THPVariable_Unpack(a[0]), &weight = THPVariable_Unpack(a[2]), &bias = THPVariable_Unpack(a[3]);
  const Tensor pre = tensor_arg(a[1]);
  const double eps = PyFloat_AsDouble(a[4]);
  if (PyErr_Occurred()) return nullptr;
  const bool silu = PyObject_IsTrue(a[5]), last = PyObject_IsTrue(a[6]);
  if (!x.defined() || !x.is_cuda() || x.dim() != 4 || x.numel() == 0 || observed() ||
      c10::impl::tls_local_dispatch_key_set().included_.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
    Py_RETURN_NONE;
  const auto dev = x.device();
  if (x.unsafeGetTensorImpl()->is_python_dispatch() || x.layout() != at::kStrided || !x.is_contiguous(at::MemoryFormat::ChannelsLast) ||
      !x.permute({0, 2, 3, 1}).is_contiguous() || !aligned(x))
    Py_RETURN_NONE;
  const int64_t C = x.size(1), rows = x.numel() / C;
  for (const Tensor* t : {&weight, &bias, &pre})
    if (t->defined() && (!plain(*t, dev) || t->scalar_type() != at::kFloat || !is_shape(*t, {C}))) Py_RETURN_NONE;
  for (const Tensor* t : {&x, &weight, &bias, &pre})
    if (t->defined() && t->_fw_grad(0).defined()) Py_RETURN_NONE;  // (forward-mode derivatives: the operators have them)
  const bool mixed = at::autocast::is_autocast_enabled(at::kCUDA);
  // the norm under autocast is one in fp32 whatever it reads, and the next convolution casts; without, map and parameters are of one type
  if (x.scalar_type() != (mixed ? at::kBFloat16 : at::kFloat) || (mixed && at::autocast::get_autocast_dtype(at::kCUDA) != at::kBFloat16)) Py_RETURN_NONE;
  if (C % 8 || C > 1024 || rows > VIG_STEM_NORM_ROWS) Py_RETURN_NONE;
  return THPVariable_Wrap(StemNormNode::apply(x, pre.defined() ? std::optional<Tensor>(pre) : std::nullopt, weight, bias, eps, silu, mixed && !last));
  END_HANDLE_TH_ERRORS
}

}  // namespace vig_host
