// Native driver of the layers' hot calls: one call into this module takes a dense layer, an attention or a whole inference
// block through its allocations, weight copies and launches of libf3d_hip.so, and the backward nodes of training are C++
// autograd functions.  The kernels and their order are those of the layers' Python code (layers/nn_ops.py, buck_swin.py,
// stage.py), which stays the path of everything this module declines (it then returns None): other dtypes, devices,
// activations and widths, and modules with hooks or other classes in place of the package's own.
//
// Why: a launch cost the Python layers 20 us of interpreter time in inference and 25 to 35 us in training (module calls, checks,
// argument conversion, autograd functions), more than the kernels of a small model take.
//
// Nothing is kept by the address or identity of an input.  A WeightCache keeps copies of parameters between eval-mode
// forwards without gradients (no_grad, inference_mode) while their address, version, dtype and device stay, as
// layers/nn_ops.py does.
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include "../../../include/f3d_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

struct Place {
  int device;
  void* stream;
};
Place place_of(const Tensor& t) {
  const int d = (int)t.get_device();
  return {d, (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)d).stream()};
}
void check(int rc) {
  if (rc != F3D_OK) throw std::runtime_error(f3d_last_error());
}
void check_covered(int rc) {      // a shape outside the kernels is told apart
  if (rc == F3D_ERR_UNSUPPORTED) C10_THROW_ERROR(NotImplementedError, f3d_last_error());
  check(rc);
}

f3d_bf16_t* bf(const Tensor& t) { return t.defined() ? (f3d_bf16_t*)t.data_ptr() : nullptr; }
float* f32(const Tensor& t) { return t.defined() ? (float*)t.data_ptr() : nullptr; }
uint32_t ld(const Tensor& t) { return t.defined() ? (uint32_t)t.stride(0) : 0u; }
Tensor or_undefined(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }

Tensor empty_like_device(at::IntArrayRef shape, at::ScalarType type, const Tensor& like) {
  return at::empty(shape, at::TensorOptions().dtype(type).device(like.device()));
}
Tensor bf16_rows(const Tensor& t) {      // bf16 with unit column stride
  Tensor r = t.scalar_type() == at::kBFloat16 ? t : t.to(at::kBFloat16);
  return r.stride(-1) == 1 ? r : r.contiguous();
}
// an output's gradient for the kernels, as autograd hands it over (a column slice of a wider one, one row expanded to all):
// copied where its rows are not at multiples of 16 bytes, each with a place of its own
Tensor grad_rows(const Tensor& t) {
  const Tensor r = bf16_rows(t);
  const bool readable = r.stride(0) >= r.size(1) && r.stride(0) % 8 == 0 && ((uintptr_t)r.data_ptr() & 15u) == 0;
  return readable ? r : r.clone(at::MemoryFormat::Contiguous);
}
bool master(const Tensor& p, const Tensor& x, at::IntArrayRef shape) {      // an fp32 parameter this module takes
  return !p.defined() || (p.scalar_type() == at::kFloat && p.device() == x.device() && p.is_contiguous() && p.sizes() == shape);
}
bool plain(const Tensor& t) { return t.layout() == at::kStrided && !t.is_neg() && !t.is_conj(); }
bool activations(const Tensor& t, int64_t cols) {      // ... of a training node, which saves them: no inference tensors
  return t.defined() && t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.dim() >= 1 && t.size(-1) == cols && plain(t) && !t.is_inference();
}
bool fold_width(int64_t c) { return c == 32 || c == 64 || c == 128 || c == 256 || c == 512; }      // LayerNorm kernels
Tensor two_axes(const Tensor& t) { return t.dim() == 2 ? t : t.reshape({-1, t.size(-1)}); }

// bf16 copies of fp32 tensors in one launch and one buffer, transposed copies where asked, and a second buffer for copies
// that the backward does not read (layers/nn_ops.py: _fresh_copies)
struct Copies {
  std::vector<Tensor> copy, turned;
};
Copies cast(const std::vector<Tensor>& ts, const std::vector<int>& turned, const std::vector<int>& apart) {
  auto has = [](const std::vector<int>& v, int i) { return std::find(v.begin(), v.end(), i) != v.end(); };
  const int n = (int)ts.size();
  std::vector<int64_t> at_copy(n, 0), at_turned(n, 0);
  int64_t total = 0, total_apart = 0;      // every copy starts at a multiple of 16 bytes
  const Tensor* first = nullptr;
  for (int i = 0; i < n; ++i) {
    if (!ts[i].defined()) continue;
    if (!first) first = &ts[i];
    const int64_t room = (ts[i].numel() + 7) / 8 * 8;
    int64_t& end = has(apart, i) ? total_apart : total;
    at_copy[i] = end;
    end += room;
    if (has(turned, i)) {
      at_turned[i] = total;
      total += room;
    }
  }
  Copies c;
  const Tensor flat = empty_like_device({total}, at::kBFloat16, *first);
  const Tensor second = total_apart ? empty_like_device({total_apart}, at::kBFloat16, *first) : flat;
  std::vector<uint64_t> table;
  uint32_t count = 0;
  for (int i = 0; i < n; ++i) {
    const Tensor& t = ts[i];
    if (!t.defined()) {
      c.copy.emplace_back();
      if (has(turned, i)) c.turned.emplace_back();
      continue;
    }
    const int64_t rows = t.dim() == 2 ? t.size(0) : 1, cols = t.size(-1);
    const Tensor& buf = has(apart, i) ? second : flat;
    c.copy.push_back(t.dim() == 2 ? buf.as_strided({rows, cols}, {cols, 1}, at_copy[i]) : buf.as_strided({cols}, {1}, at_copy[i]));
    uint64_t to_turned = 0;
    if (has(turned, i)) {
      c.turned.push_back(flat.as_strided({cols, rows}, {rows, 1}, at_turned[i]));
      to_turned = (uint64_t)(uintptr_t)flat.data_ptr() + 2 * at_turned[i];
    }
    table.insert(table.end(), {(uint64_t)(uintptr_t)t.data_ptr(), (uint64_t)(uintptr_t)buf.data_ptr() + 2 * at_copy[i], to_turned,
                               (uint64_t)rows, (uint64_t)cols});
    ++count;
  }
  const Place p = place_of(*first);
  check(f3d_cast_bf16(table.data(), count, p.device, p.stream));
  return c;
}

// which inputs of a backward node want a gradient: the engine numbers the defined ones
struct Wanted {
  AutogradContext* ctx;
  const std::vector<int64_t> edge;
  Wanted(AutogradContext* c, const char* key) : ctx(c), edge(c->saved_data[key].toIntVector()) {}
  bool operator()(int i) const { return edge[i] >= 0 && ctx->needs_input_grad((size_t)edge[i]); }
};
std::vector<int64_t> edges(std::initializer_list<const Tensor*> ts) {
  std::vector<int64_t> e;
  int64_t n = 0;
  for (const Tensor* t : ts) e.push_back(t->defined() ? n++ : -1);
  return e;
}
Tensor as_grad_of(const Tensor& g, const Tensor& like) {
  if (!g.defined()) return g;
  return g.to(like.scalar_type()).reshape(like.sizes());
}

struct LnGrads {
  Tensor dx, dg, db;
};
// dres: another gradient of x, added before the one rounding to bf16, or (`apart`) after it
LnGrads ln_backward(const Tensor& x, const Tensor& dh, const Tensor& g16, const Tensor& dres, double eps, bool apart = false) {
  const int64_t m = x.size(0), c = x.size(1);
  LnGrads r{empty_like_device({m, c}, at::kBFloat16, x), empty_like_device({c}, at::kFloat, x), empty_like_device({c}, at::kFloat, x)};
  const Place p = place_of(x);
  check_covered((apart ? f3d_layernorm_bwd_add_bf16 : f3d_layernorm_bwd_bf16)(
      bf(x), ld(x), bf(dh), ld(dh), bf(g16), bf(dres), ld(dres), bf(r.dx), ld(r.dx), f32(r.dg), f32(r.db), (uint32_t)m, (uint32_t)c,
      (float)eps, 0, p.device, p.stream));
  return r;
}
void wgrad(const Tensor& dy, const Tensor& x, const Tensor& dw, const Tensor& db) {
  const Place p = place_of(x);
  check(f3d_linear_wgrad_bf16(bf(dy), ld(dy), bf(x), ld(x), f32(dw), f32(db), (uint32_t)dy.size(0), (uint32_t)dy.size(1),
                              (uint32_t)x.size(1), 0, p.device, p.stream));
}
void linear(const Tensor& x, const Tensor& w, const Tensor& b, const Tensor& residual, const Tensor& y) {
  const Place p = place_of(x);
  check(f3d_linear_bf16(bf(x), ld(x), bf(w), bf(b), bf(residual), ld(residual), bf(y), ld(y), (uint32_t)x.size(0),
                        (uint32_t)w.size(0), (uint32_t)w.size(1), F3D_ACT_NONE, p.device, p.stream));
}
int ln_linear_code(const Tensor& x, const Tensor& g, const Tensor& be, double eps, const Tensor& w, const Tensor& b,
                   const Tensor& residual, const Tensor& y, uint32_t act) {
  const Place p = place_of(x);
  return f3d_ln_linear_bf16(bf(x), ld(x), bf(g), bf(be), (float)eps, bf(w), bf(b), bf(residual), ld(residual), bf(y), ld(y),
                            (uint32_t)x.size(0), (uint32_t)w.size(0), (uint32_t)w.size(1), act, p.device, p.stream);
}
void ln_linear(const Tensor& x, const Tensor& g, const Tensor& be, double eps, const Tensor& w, const Tensor& b,
               const Tensor& residual, const Tensor& y, uint32_t act) {
  check(ln_linear_code(x, g, be, eps, w, b, residual, y, act));
}
void layernorm(const Tensor& x, const Tensor& g, const Tensor& be, const Tensor& y, double eps) {
  const Place p = place_of(x);
  check(f3d_layernorm_bf16(bf(x), bf(g), bf(be), bf(y), (uint32_t)x.size(0), (uint32_t)x.size(1), (float)eps, p.device, p.stream));
}
// LayerNorm + gated MLP (+ residual): one kernel where there is one and it is wanted, else fc1 with the gate, then fc2
void gated_mlp(const Tensor& x, const Tensor& g, const Tensor& be, double eps, const Tensor& w1, const Tensor& b1, const Tensor& w2,
               const Tensor& b2, const Tensor& residual, const Tensor& y, bool one_kernel) {
  const int64_t m = x.size(0), c = x.size(1), hid = w2.size(1);
  const Place p = place_of(x);
  if (one_kernel) {
    const int rc = f3d_ln_mlp_swiglu_bf16(bf(x), ld(x), bf(g), bf(be), (float)eps, bf(w1), bf(b1), bf(w2), bf(b2), bf(residual),
                                          ld(residual), bf(y), ld(y), (uint32_t)m, (uint32_t)c, (uint32_t)hid, p.device, p.stream);
    if (rc != F3D_ERR_UNSUPPORTED) {
      check(rc);
      return;
    }
  }
  const Tensor h = empty_like_device({m, hid}, at::kBFloat16, x);
  ln_linear(x, g, be, eps, w1, b1, Tensor(), h, F3D_ACT_SWIGLU);
  linear(h, w2, b2, residual, y);
}

// ---- training ---------------------------------------------------------------------------------------------------

// y = [LayerNorm](x) w^T + b (+ residual); the backward of layers/nn_ops.py: _LinearGrad
struct LinearNode : torch::autograd::Function<LinearNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const OptTensor& bias_, const OptTensor& residual_,
                        const OptTensor& ln_w_, const OptTensor& ln_b_, double eps) {
    const Tensor bias = or_undefined(bias_), residual = or_undefined(residual_), ln_w = or_undefined(ln_w_), ln_b = or_undefined(ln_b_);
    const Copies c = cast({weight, bias, ln_w, ln_b}, {0}, {0});
    const Tensor x2 = bf16_rows(x), r2 = residual.defined() ? bf16_rows(residual) : residual;
    const Tensor y = empty_like_device({x2.size(0), weight.size(0)}, at::kBFloat16, x);
    if (ln_w.defined()) ln_linear(x2, c.copy[2], c.copy[3], eps, c.copy[0], c.copy[1], r2, y, F3D_ACT_NONE);
    else linear(x2, c.copy[0], c.copy[1], r2, y);
    ctx->save_for_backward({x, weight, bias, residual, ln_w, ln_b, c.copy[2], c.copy[3], c.turned[0]});
    ctx->saved_data["edges"] = edges({&x, &weight, &bias, &residual, &ln_w, &ln_b});
    ctx->saved_data["eps"] = eps;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &x = s[0], &weight = s[1], &bias = s[2], &residual = s[3], &ln_w = s[4], &ln_b = s[5], &g16 = s[6], &b16 = s[7], &wt = s[8];
    const Wanted want(ctx, "edges");
    const double eps = ctx->saved_data["eps"].toDouble();
    const Tensor dy = grad_rows(grads[0]), x2 = bf16_rows(x);
    const int64_t m = x2.size(0), k = x2.size(1), n = dy.size(1);
    Tensor h = x2;
    if (ln_w.defined()) {
      h = empty_like_device({m, k}, at::kBFloat16, x2);
      layernorm(x2.contiguous(), g16, b16, h, eps);
    }
    Tensor dw, db, dx, dg, dbeta;
    if (want(1) || want(2)) {
      dw = empty_like_device({n, k}, at::kFloat, x2);
      if (bias.defined()) db = empty_like_device({n}, at::kFloat, x2);
      wgrad(dy, h, dw, db);
    }
    if (want(0) || want(4) || want(5)) {
      const Tensor dh = empty_like_device({m, k}, at::kBFloat16, x2);
      linear(dy, wt, Tensor(), Tensor(), dh);
      if (ln_w.defined()) {
        LnGrads r = ln_backward(x2, dh, g16, Tensor(), eps);
        dx = r.dx; dg = r.dg; dbeta = r.db;
      } else {
        dx = dh;
      }
    }
    return {want(0) ? as_grad_of(dx, x) : Tensor(), want(1) ? as_grad_of(dw, weight) : Tensor(), want(2) ? as_grad_of(db, bias) : Tensor(),
            want(3) ? as_grad_of(dy, residual) : Tensor(), want(4) ? as_grad_of(dg, ln_w) : Tensor(),
            want(5) ? as_grad_of(dbeta, ln_b) : Tensor(), Tensor()};
  }
};

// y = LayerNorm(x) w^T + b and x itself once more, for a residual: the gradient that comes back by that way is added where
// LayerNorm's own dx is written (with the bits of adding the two tensors), instead of by a pass over both
struct ForkNode : torch::autograd::Function<ForkNode> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const OptTensor& bias_, const Tensor& ln_w,
                               const OptTensor& ln_b_, double eps) {
    const Tensor bias = or_undefined(bias_), ln_b = or_undefined(ln_b_);
    const Copies c = cast({weight, bias, ln_w, ln_b}, {0}, {0});
    const Tensor x2 = bf16_rows(x);
    const Tensor y = empty_like_device({x2.size(0), weight.size(0)}, at::kBFloat16, x);
    ln_linear(x2, c.copy[2], c.copy[3], eps, c.copy[0], c.copy[1], Tensor(), y, F3D_ACT_NONE);
    ctx->save_for_backward({x, weight, bias, ln_w, ln_b, c.copy[2], c.copy[3], c.turned[0]});
    ctx->saved_data["edges"] = edges({&x, &weight, &bias, &ln_w, &ln_b});
    ctx->saved_data["eps"] = eps;
    return {y, x};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &x = s[0], &weight = s[1], &bias = s[2], &ln_w = s[3], &ln_b = s[4], &g16 = s[5], &b16 = s[6], &wt = s[7];
    const Wanted want(ctx, "edges");
    const double eps = ctx->saved_data["eps"].toDouble();
    const Tensor dy = grad_rows(grads[0]), dres = grad_rows(grads[1]), x2 = bf16_rows(x);
    const int64_t m = x2.size(0), k = x2.size(1), n = dy.size(1);
    const Tensor h = empty_like_device({m, k}, at::kBFloat16, x2);
    layernorm(x2.contiguous(), g16, b16, h, eps);
    Tensor dw, db;
    if (want(1) || want(2)) {
      dw = empty_like_device({n, k}, at::kFloat, x2);
      if (bias.defined()) db = empty_like_device({n}, at::kFloat, x2);
      wgrad(dy, h, dw, db);
    }
    LnGrads r;
    if (want(0) || want(3) || want(4)) {
      linear(dy, wt, Tensor(), Tensor(), h);      // h <- dh
      r = ln_backward(x2, h, g16, dres, eps, true);
    }
    return {want(0) ? as_grad_of(r.dx, x) : Tensor(), want(1) ? as_grad_of(dw, weight) : Tensor(), want(2) ? as_grad_of(db, bias) : Tensor(),
            want(3) ? as_grad_of(r.dg, ln_w) : Tensor(), want(4) ? as_grad_of(r.db, ln_b) : Tensor(), Tensor()};
  }
};

// None: not a case of this module (the caller's Python path takes it, and raises what there is to raise)
py::object linear_train(const Tensor& x, const Tensor& weight, const OptTensor& bias, const OptTensor& residual, const OptTensor& ln_w,
                        const OptTensor& ln_b, double eps) {
  if (weight.dim() != 2) return py::none();
  const int64_t n = weight.size(0), k = weight.size(1);
  const bool norm = ln_w.has_value();
  if (n == 0 || k == 0 || !activations(x, k) || !x.requires_grad() || n % 8 || k % 8 || !master(weight, x, {n, k}) || !master(or_undefined(bias), x, {n}) ||
      (norm && !master(*ln_w, x, {k})) || (ln_b.has_value() && (!norm || !master(*ln_b, x, {k}))))
    return py::none();
  Tensor r2;
  if (residual.has_value()) {
    if (!activations(*residual, n) || residual->device() != x.device() || residual->numel() / n != x.numel() / k) return py::none();
    r2 = two_axes(*residual);
  }
  const Tensor y = LinearNode::apply(two_axes(x), weight, bias, r2.defined() ? OptTensor(r2) : std::nullopt, ln_w, ln_b, eps);
  if (x.dim() == 2) return py::cast(y);
  std::vector<int64_t> shape = x.sizes().vec();
  shape.back() = n;
  return py::cast(y.view(shape));
}

py::object linear_fork(const Tensor& x, const Tensor& weight, const OptTensor& bias, const Tensor& ln_w, const OptTensor& ln_b, double eps) {
  if (weight.dim() != 2) return py::none();
  const int64_t n = weight.size(0), k = weight.size(1);
  if (!activations(x, k) || !x.requires_grad() || n % 8 || !fold_width(k) || !master(weight, x, {n, k}) || !master(or_undefined(bias), x, {n}) ||
      !master(ln_w, x, {k}) || !master(or_undefined(ln_b), x, {k}))
    return py::none();
  const variable_list r = ForkNode::apply(two_axes(x), weight, bias, ln_w, ln_b, eps);
  if (x.dim() == 2) return py::make_tuple(r[0], r[1]);
  std::vector<int64_t> shape = x.sizes().vec();
  shape.back() = n;
  return py::make_tuple(r[0].view(shape), r[1].view(x.sizes()));
}

// the gated MLP with its LayerNorm (+ residual); the backward of layers/nn_ops.py: _GatedMLPGrad
struct MlpNode : torch::autograd::Function<MlpNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const OptTensor& residual_, const Tensor& ln_w, const Tensor& ln_b,
                        const Tensor& w1, const Tensor& b1, const Tensor& w2, const Tensor& b2, double eps, bool one_kernel) {
    const Tensor residual = or_undefined(residual_);
    const Copies c = cast({ln_w, ln_b, w1, b1, w2, b2}, {2, 4}, {4});
    const Tensor x2 = bf16_rows(x).contiguous(), r2 = residual.defined() ? bf16_rows(residual) : residual;
    const Tensor y = empty_like_device(x2.sizes(), at::kBFloat16, x2);
    gated_mlp(x2, c.copy[0], c.copy[1], eps, c.copy[2], c.copy[3], c.copy[4], c.copy[5], r2, y, one_kernel);
    ctx->save_for_backward({x, residual, ln_w, ln_b, w1, b1, w2, b2, c.copy[0], c.copy[1], c.copy[2], c.copy[3], c.turned[0], c.turned[1]});
    ctx->saved_data["edges"] = edges({&x, &residual, &ln_w, &ln_b, &w1, &b1, &w2, &b2});
    ctx->saved_data["eps"] = eps;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &x = s[0], &residual = s[1], &ln_w = s[2], &ln_b = s[3], &w1 = s[4], &b1 = s[5], &w2 = s[6], &b2 = s[7], &g16 = s[8],
                 &be16 = s[9], &w1_16 = s[10], &b1_16 = s[11], &w1t = s[12], &w2t = s[13];
    const Wanted want(ctx, "edges");
    const double eps = ctx->saved_data["eps"].toDouble();
    const Tensor dy = grad_rows(grads[0]), x2 = bf16_rows(x).contiguous();
    const int64_t m = x2.size(0), c = x2.size(1), hid = w2.size(1);
    const Tensor h = empty_like_device({m, c}, at::kBFloat16, x2);
    layernorm(x2, g16, be16, h, eps);
    const Tensor dz = empty_like_device({m, 2 * hid}, at::kBFloat16, x2), a = empty_like_device({m, hid}, at::kBFloat16, x2);
    const Place p = place_of(x2);
    const int rc = f3d_mlp_gate_bwd_bf16(bf(h), ld(h), bf(dy), ld(dy), bf(w1_16), bf(b1_16), bf(w2t), bf(dz), ld(dz), bf(a), ld(a),
                                         (uint32_t)m, (uint32_t)c, (uint32_t)hid, p.device, p.stream);
    if (rc == F3D_ERR_UNSUPPORTED) {
      linear(h, w1_16, b1_16, Tensor(), dz);
      linear(dy, w2t, Tensor(), Tensor(), a);
      check(f3d_swiglu_bwd_bf16(bf(dz), ld(dz), bf(a), ld(a), bf(dz), ld(dz), bf(a), ld(a), (uint32_t)m, (uint32_t)hid, p.device, p.stream));
    } else {
      check(rc);
    }
    const Tensor dw2 = empty_like_device({c, hid}, at::kFloat, x2), db2 = empty_like_device({c}, at::kFloat, x2);
    wgrad(dy, a, dw2, db2);
    const Tensor dw1 = empty_like_device({2 * hid, c}, at::kFloat, x2), db1 = empty_like_device({2 * hid}, at::kFloat, x2);
    wgrad(dz, h, dw1, db1);
    linear(dz, w1t, Tensor(), Tensor(), h);      // h <- dh
    // a residual that is the input itself: one gradient tensor for both routes
    const bool shared = residual.defined() && want(0) && want(1) && residual.data_ptr() == x.data_ptr() && residual.sizes() == x.sizes() &&
                        residual.scalar_type() == x.scalar_type() && residual.strides() == x.strides();
    const LnGrads r = ln_backward(x2, h, g16, shared ? dy : Tensor(), eps);
    return {want(0) ? as_grad_of(r.dx, x) : Tensor(), want(1) && !shared ? as_grad_of(dy, residual) : Tensor(),
            want(2) ? as_grad_of(r.dg, ln_w) : Tensor(), want(3) ? as_grad_of(r.db, ln_b) : Tensor(),
            want(4) ? as_grad_of(dw1, w1) : Tensor(), want(5) ? as_grad_of(db1, b1) : Tensor(),
            want(6) ? as_grad_of(dw2, w2) : Tensor(), want(7) ? as_grad_of(db2, b2) : Tensor(), Tensor(), Tensor()};
  }
};

py::object mlp_train(const Tensor& x, const OptTensor& residual, const Tensor& ln_w, const Tensor& ln_b, const Tensor& w1, const Tensor& b1,
                     const Tensor& w2, const Tensor& b2, double eps, bool one_kernel) {
  if (w2.dim() != 2) return py::none();
  const int64_t c = w2.size(0), hid = w2.size(1);
  if (!fold_width(c) || hid % 8 || !activations(x, c) || !x.requires_grad() || !master(ln_w, x, {c}) || !master(ln_b, x, {c}) ||
      !master(w1, x, {2 * hid, c}) || !master(b1, x, {2 * hid}) || !master(w2, x, {c, hid}) || !master(b2, x, {c}))
    return py::none();
  Tensor r2;
  if (residual.has_value()) {
    if (!activations(*residual, c) || residual->device() != x.device() || residual->numel() != x.numel()) return py::none();
    r2 = two_axes(*residual);
  }
  const Tensor y = MlpNode::apply(two_axes(x), r2.defined() ? OptTensor(r2) : std::nullopt, ln_w, ln_b, w1, b1, w2, b2, eps, one_kernel);
  return py::cast(x.dim() == 2 ? y : y.view(x.sizes()));
}

// attention over the thirds of one projection output; layers/buck_swin.py: BuckSwinQKVFunction
struct Heads {
  int64_t B, L, H, D;
  Tensor O, lse;
};
Heads attention(const Tensor& qkv, const Tensor& scopes, int64_t bucket, int64_t heads, bool covers) {
  const int64_t B = qkv.size(0), L = qkv.size(1), C = qkv.size(2) / 3, D = C / heads;
  Heads r{B, L, heads, D, empty_like_device({B, L, heads, D}, at::kBFloat16, qkv), {}};
  const auto f = at::TensorOptions().dtype(at::kFloat).device(qkv.device());
  r.lse = covers ? at::empty({B, L, heads}, f) : at::zeros({B, L, heads}, f);
  const Place p = place_of(qkv);
  const f3d_bf16_t* q = bf(qkv);
  check(f3d_buck_swin_fwd_strided(q, q + C, q + 2 * C, (uint32_t)(3 * C), bf(r.O), f32(r.lse), (const uint32_t*)scopes.data_ptr(),
                                  (uint32_t)scopes.size(0), (uint32_t)scopes.size(1), (uint32_t)bucket, (uint32_t)B, (uint32_t)L,
                                  (uint32_t)heads, (uint32_t)D, nullptr, p.device, p.stream));
  return r;
}
struct AttentionNode : torch::autograd::Function<AttentionNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& scopes, int64_t bucket, int64_t heads, bool covers) {
    const Heads r = attention(qkv, scopes, bucket, heads, covers);
    ctx->save_for_backward({qkv, r.O, r.lse});
    ctx->saved_data["scopes"] = scopes;
    ctx->saved_data["bucket"] = bucket;
    ctx->saved_data["covers"] = covers;
    return r.O;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &qkv = s[0], &O = s[1], &lse = s[2];
    const Tensor scopes = ctx->saved_data["scopes"].toTensor();
    const bool covers = ctx->saved_data["covers"].toBool();
    const int64_t B = O.size(0), L = O.size(1), H = O.size(2), D = O.size(3), C = H * D;
    const Tensor dO = (grads[0].scalar_type() == at::kBFloat16 ? grads[0] : grads[0].to(at::kBFloat16)).contiguous();
    // rows that no scope covers are not written
    const Tensor dqkv = covers ? at::empty_like(qkv) : at::zeros_like(qkv);
    const Tensor delta = at::zeros({B, L, H}, at::TensorOptions().dtype(at::kFloat).device(qkv.device()));
    const Place p = place_of(qkv);
    const f3d_bf16_t* q = bf(qkv);
    f3d_bf16_t* g = bf(dqkv);
    check_covered(f3d_buck_swin_bwd_strided(q, q + C, q + 2 * C, (uint32_t)(3 * C), bf(O), bf(dO), f32(lse), f32(delta), g, g + C, g + 2 * C,
                                    (uint32_t)(3 * C), (const uint32_t*)scopes.data_ptr(), (uint32_t)scopes.size(0),
                                    (uint32_t)scopes.size(1), (uint32_t)ctx->saved_data["bucket"].toInt(), (uint32_t)B, (uint32_t)L,
                                    (uint32_t)H, (uint32_t)D, nullptr, p.device, p.stream));
    return {dqkv, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};
bool attention_covers(const Tensor& qkv, const Tensor& scopes, int64_t heads) {
  return qkv.dim() == 3 && qkv.is_cuda() && qkv.scalar_type() == at::kBFloat16 && qkv.is_contiguous() && plain(qkv) && heads > 0 &&
         qkv.size(2) % (3 * heads) == 0 && scopes.dim() == 2 && scopes.scalar_type() == at::kUInt32 && scopes.is_contiguous() &&
         scopes.device() == qkv.device();
}
py::object attention_qkv(const Tensor& qkv, const Tensor& scopes, int64_t bucket, int64_t heads, bool covers) {
  if (!attention_covers(qkv, scopes, heads)) return py::none();
  if (at::GradMode::is_enabled() && qkv.requires_grad()) return py::cast(AttentionNode::apply(qkv, scopes, bucket, heads, covers));
  return py::cast(attention(qkv, scopes, bucket, heads, covers).O);
}

// ---- inference --------------------------------------------------------------------------------------------------

// y = x w^T + b (+ residual) on bf16 copies of the parameters
py::object linear_infer(const Tensor& x, const Tensor& w, const OptTensor& b_, const OptTensor& residual_) {
  const Tensor b = or_undefined(b_), residual = or_undefined(residual_);
  if (w.dim() != 2 || w.numel() == 0 || x.dim() < 1 || x.numel() == 0) return py::none();
  const int64_t n = w.size(0), k = w.size(1);
  auto ours = [&](const Tensor& t) { return t.scalar_type() == at::kBFloat16 && t.layout() == at::kStrided && t.device() == x.device(); };
  if (!x.is_cuda() || !ours(x) || x.size(-1) != k || x.stride(-1) != 1 || !ours(w) || !w.is_contiguous() ||
      (b.defined() && (!ours(b) || !b.is_contiguous() || b.dim() != 1 || b.size(0) != n)) ||
      (residual.defined() && (!ours(residual) || residual.dim() < 1 || residual.size(-1) != n || residual.stride(-1) != 1 || residual.numel() / n != x.numel() / k)))
    return py::none();
  const Tensor x2 = two_axes(x), y = empty_like_device({x2.size(0), n}, at::kBFloat16, x);
  linear(x2, w, b, residual.defined() ? two_axes(residual) : residual, y);
  if (x.dim() == 2) return py::cast(y);
  std::vector<int64_t> shape = x.sizes().vec();
  shape.back() = n;
  return py::cast(y.view(shape));
}

// bf16 copies of a block's parameters and the buffers in which the kernels keep what they prepare from them, between
// eval-mode forwards without gradients: current while every parameter keeps its address, version, dtype and device (one without a
// version is not taken; activations need none)
struct WeightCache {
  struct Key {
    const void* at = nullptr;
    uint32_t version = 0;
    at::ScalarType type = at::kFloat;
    int device = -1;
    bool operator==(const Key& o) const { return at == o.at && version == o.version && type == o.type && device == o.device; }
  };
  struct Slot {
    Key key;
    Tensor source, value;      // the source is held: its memory is not handed out again while the key stands
    bool filled = false;
  };
  struct Staged {
    Tensor buf;
    bool ready = false;
    double eps = 0;
    int kind = -1;
  };
  std::vector<Slot> slots;
  Staged staged[2];      // 0: LayerNorm + QKV, 1: the MLP

  void clear() {
    slots.clear();
    for (Staged& s : staged) s.ready = false;
  }
  // the parameters' copies; false where one is not a case of this module
  bool update(const std::vector<Tensor>& ps, const std::vector<int>& first_of_staged) {
    if (slots.size() != ps.size()) {
      clear();
      slots.resize(ps.size());
    }
    for (size_t i = 0; i < ps.size(); ++i) {
      const Tensor& p = ps[i];
      Slot& s = slots[i];
      Key k;
      if (p.defined()) {
        if (p.is_inference()) return false;
        k = {p.data_ptr(), p.unsafeGetTensorImpl()->version_counter().current_version(), p.scalar_type(), (int)p.get_device()};
      }
      if (s.filled && s.key == k) continue;
      for (int b = 0; b < 2; ++b)
        if ((int)i >= first_of_staged[2 * b] && (int)i < first_of_staged[2 * b + 1]) staged[b].ready = false;
      s.source = p.defined() ? p.detach() : Tensor();
      if (!p.defined()) s.value = Tensor();
      else if (p.scalar_type() == at::kBFloat16 && p.is_contiguous()) s.value = s.source;
      else s.value = s.source.to(at::kBFloat16).contiguous();
      s.key = k;
      s.filled = true;
    }
    return true;
  }
  // the code of call(), the dense call that prepares w [rows, cols], with the buffer staged for it.  The buffer is ready once
  // the call has left the weights there, and the staging ends, however the call ends.
  template <typename Call>
  int staged_call(int b, const Tensor& w, double eps, int kind, Call call) {
    const int64_t rows = w.size(0), cols = w.size(1), need = 3 * rows * cols + 4 * rows + 2 * cols + 512;
    Staged& s = staged[b];
    if (!s.buf.defined() || s.buf.numel() < need || s.buf.device() != w.device()) {
      s.ready = false;
      s.buf = empty_like_device({need}, at::kByte, w);
    }
    const bool ready = s.ready && s.eps == eps && s.kind == kind;
    s.ready = false;
    s.eps = eps;
    s.kind = kind;
    check(f3d_stage_weights(s.buf.data_ptr(), (size_t)s.buf.numel(), ready ? 1 : 0));
    struct End {
      Staged& s;
      ~End() { s.ready = f3d_staged_weights_kept() != 0; }
    } end{s};
    return call();
  }
};

// One block at inference: LayerNorm + QKV, attention, out-projection + MLP in one kernel (`one_half`) or out-projection with
// the residual and then the MLP (`one_mlp`: as one kernel).  ps: norm w, b; qkv w, b; proj w, b; LayerNorm w, b, fc1 w, b,
// fc2 w, b of the MLP.  None: not a case of this module.
py::object block_infer(WeightCache& cache, const Tensor& x, const std::vector<OptTensor>& params, double eps, double mlp_eps, const Tensor& scopes,
                       int64_t bucket, int64_t heads, bool covers, bool one_half, bool one_mlp) {
  std::vector<Tensor> ps;
  ps.reserve(12);
  for (const OptTensor& p : params) ps.push_back(or_undefined(p));
  if (ps.size() != 12 || !ps[0].defined() || !ps[2].defined() || !ps[4].defined() || !ps[6].defined() || !ps[8].defined() || !ps[10].defined())
    return py::none();
  if (x.dim() != 2 || ps[10].dim() != 2) return py::none();
  const int64_t m = x.size(0), c = x.size(1), hid = ps[10].size(1);
  const std::vector<std::vector<int64_t>> shapes = {{c}, {c}, {3 * c, c}, {3 * c}, {c, c}, {c}, {c}, {c}, {2 * hid, c}, {2 * hid}, {c, hid}, {c}};
  for (int i = 0; i < 12; ++i)
    if (ps[i].defined() && (ps[i].device() != x.device() || ps[i].sizes() != at::IntArrayRef(shapes[i]) ||
                            (ps[i].scalar_type() != at::kFloat && ps[i].scalar_type() != at::kBFloat16) || ps[i].layout() != at::kStrided))
      return py::none();
  if (!fold_width(c) || !x.is_cuda() || x.scalar_type() != at::kBFloat16 || x.layout() != at::kStrided || x.stride(1) != 1 ||
      scopes.dim() != 2 || scopes.scalar_type() != at::kUInt32 || !scopes.is_contiguous() || scopes.device() != x.device() ||
      heads <= 0 || c % heads != 0 || m == 0 || !plain(x))
    return py::none();
  if (!cache.update(ps, {0, 4, 6, 12})) return py::none();
  auto w = [&](int i) -> const Tensor& { return cache.slots[i].value; };

  const Tensor qkv = empty_like_device({1, m, 3 * c}, at::kBFloat16, x), qkv_rows = qkv.view({m, 3 * c});
  check(cache.staged_call(0, w(2), eps, 0,
                          [&] { return ln_linear_code(x, w(0), w(1), eps, w(2), w(3), Tensor(), qkv_rows, F3D_ACT_NONE); }));
  const Tensor o = attention(qkv, scopes, bucket, heads, covers).O.view({m, c});
  const Tensor y = empty_like_device({m, c}, at::kBFloat16, x);
  const Place p = place_of(x);
  if (one_half) {
    const int rc = cache.staged_call(1, w(8), mlp_eps, 1, [&] {
      return f3d_proj_ln_mlp_swiglu_bf16(bf(o), ld(o), bf(w(4)), bf(w(5)), bf(x), ld(x), bf(w(6)), bf(w(7)), (float)mlp_eps, bf(w(8)),
                                         bf(w(9)), bf(w(10)), bf(w(11)), bf(y), ld(y), (uint32_t)m, (uint32_t)c, (uint32_t)hid, p.device,
                                         p.stream);
    });
    if (rc != F3D_ERR_UNSUPPORTED) {
      check(rc);
      return py::cast(y);
    }
  }
  const Tensor mid = empty_like_device({m, c}, at::kBFloat16, x);
  linear(o, w(4), w(5), x, mid);
  if (one_mlp) {
    const int rc = cache.staged_call(1, w(8), mlp_eps, 1, [&] {
      return f3d_ln_mlp_swiglu_bf16(bf(mid), ld(mid), bf(w(6)), bf(w(7)), (float)mlp_eps, bf(w(8)), bf(w(9)), bf(w(10)), bf(w(11)), bf(mid),
                                    ld(mid), bf(y), ld(y), (uint32_t)m, (uint32_t)c, (uint32_t)hid, p.device, p.stream);
    });
    if (rc != F3D_ERR_UNSUPPORTED) {
      check(rc);
      return py::cast(y);
    }
  }
  const Tensor h = empty_like_device({m, hid}, at::kBFloat16, x);
  check(cache.staged_call(1, w(8), mlp_eps, 2,
                          [&] { return ln_linear_code(mid, w(6), w(7), mlp_eps, w(8), w(9), Tensor(), h, F3D_ACT_SWIGLU); }));
  linear(h, w(10), w(11), mid, y);
  return py::cast(y);
}

}  // namespace

PYBIND11_MODULE(_f3d_host, m) {
  m.def("linear_train", &linear_train);
  m.def("linear_fork", &linear_fork);
  m.def("mlp_train", &mlp_train);
  m.def("attention_qkv", &attention_qkv);
  m.def("linear_infer", &linear_infer);
  m.def("block_infer", &block_infer);
  py::class_<WeightCache>(m, "WeightCache").def(py::init<>()).def("clear", &WeightCache::clear);
}
