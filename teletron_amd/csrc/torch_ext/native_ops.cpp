// Python module `native_ops`: the operators of teletron_amd/ops.py as one call each, for the tensors a
// model passes in earnest (dense bf16 activations, evenly spaced bf16 or fp32 parameters).  Checks,
// output allocation, workspace and launch cost 25-45 us of Python and ctypes per operator, several
// times the kernels' own time for a text-token tensor (RMSNorm 512 x 5120: 4 us forward, 6 + 3 us backward).  A function returns
// None, and has done nothing, wherever its arguments are anything else: ops.py then takes the call, with
// its own checks and errors.  Holds no kernels.
//
// The second half are the same operators as nodes of the autograd graph, for the Functions of functional.py: their
// backward runs on the engine's thread without the interpreter.
#include "glue.hpp"

#include <ATen/TensorSubclassLikeUtils.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

namespace py = pybind11;
using at::Tensor;
using std::optional;

namespace {

void clear_workspaces() {
  auto& w = tt_glue::workspaces();
  std::lock_guard<std::mutex> lock(w.mu);
  w.kept.clear();
}

bool plain(const Tensor& t) { return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !at::isTensorSubclassLike(t); }
bool activation(const Tensor& t) {
  return plain(t) && t.scalar_type() == at::kBFloat16 && t.dim() >= 1 && t.numel() > 0 && t.is_contiguous();
}
bool like(const Tensor& t, const Tensor& x) { return activation(t) && t.sizes() == x.sizes() && t.device() == x.device(); }
bool aligned(std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (reinterpret_cast<uintptr_t>(t->data_ptr()) % 16) return false;
  return true;
}

// A parameter as n vectors of `cols` values, `stride` apart.
struct Vectors {
  int64_t n = 0, stride = 0;
};
bool vectors(const Tensor& p, const Tensor& x, int64_t cols, Vectors* v) {
  if (!plain(p) || p.scalar_type() != at::kBFloat16 || p.device() != x.device() || p.dim() < 1 || p.size(-1) != cols ||
      p.numel() == 0 || (p.stride(-1) != 1 && !p.is_contiguous()))
    return false;
  v->n = 1;
  v->stride = cols;
  for (int64_t d = 0; d < p.dim() - 1; ++d) {
    if (p.size(d) == 1) continue;
    if (v->n != 1) {   // more than one outer dimension: only where they are dense
      if (!p.is_contiguous()) return false;
      v->n = p.numel() / cols;
      v->stride = cols;
      return true;
    }
    v->n = p.size(d);
    v->stride = p.stride(d);
  }
  return true;
}
Tensor dense(const Tensor& p, bool save, int64_t n, int64_t cols) {
  return p.is_contiguous() || !save ? p : at::empty({n, cols}, p.options());
}
void* copy_of(const Tensor& p, const Tensor& kept) { return kept.is_same(p) ? nullptr : kept.data_ptr(); }

struct Launch {
  c10::hip::HIPGuard guard;
  hipStream_t stream;
  explicit Launch(const Tensor& x)
      : guard(x.device().index()), stream(c10::hip::getCurrentHIPStream(x.device().index()).stream()) {}
};

// The launch itself may wait for room in the queue: other Python threads run meanwhile.  (The autograd engine calls
// without the interpreter's lock.)
template <typename F>
bool launched(F f) {
  optional<py::gil_scoped_release> unlocked;
  if (PyGILState_Check()) unlocked.emplace();
  return f() == TT_OK;
}
// The same with the backward workspace: f(memory, bytes).
template <typename F>
bool launched(size_t bytes, const Tensor& ref, F f) {
  return tt_glue::with_workspace(bytes, ref, f) == TT_OK;
}
// Errors of the allocator and of tensors without memory are raised by ops.py, as its own types.
template <typename F>
bool tried(F f) {
  try {
    return f();
  } catch (const c10::Error&) {
    return false;
  }
}

// What a forward returns and keeps for backward.
struct Forward {
  Tensor y, s, kept, kept_gate;
};

bool adaln_forward(const Tensor& x, const Tensor& scale, const Tensor& shift, double eps, bool save, Forward* f) {
  if (!activation(x)) return false;
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  Vectors a, b;
  if (!vectors(scale, x, cols, &a) || !vectors(shift, x, cols, &b) || a.n != b.n || rows % a.n != 0) return false;
  Launch on(x);
  f->y = at::empty_like(x);
  f->kept = dense(scale, save, a.n, cols);
  return launched([&] { return tt_adaln_forward_strided(f->y.data_ptr(), x.data_ptr(), scale.data_ptr(), a.stride, shift.data_ptr(), b.stride,
                               copy_of(scale, f->kept), rows, cols, rows / a.n, (float)eps, on.stream); });
}

// What a backward returns, in the order of the operator's arguments.
struct Backward {
  Tensor dx, d1, d2, d3, d4;
};

bool adaln_backward(const Tensor& dy, const Tensor& x, const Tensor& scale, double eps, bool bf16,
                    at::IntArrayRef scale_shape, at::IntArrayRef shift_shape, Backward* g) {
  if (!activation(x) || !like(dy, x)) return false;
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  Vectors a;
  if (!vectors(scale, x, cols, &a) || !scale.is_contiguous() || rows % a.n != 0 || !aligned({&x, &dy, &scale}))
    return false;
  Launch on(x);
  const auto opts = x.options().dtype(bf16 ? at::kBFloat16 : at::kFloat);
  g->dx = at::empty_like(x);
  Tensor dscale = g->d1 = at::empty(scale_shape, opts), dshift = g->d2 = at::empty(shift_shape, opts);
  if (dscale.numel() != a.n * cols || dshift.numel() != a.n * cols) return false;
  return launched(tt_adaln_backward_workspace_bytes(rows, cols, rows / a.n), x,
                [&](void* ws, size_t ws_bytes) { return tt_adaln_backward_typed(g->dx.data_ptr(), dscale.data_ptr(), dshift.data_ptr(), bf16, dy.data_ptr(), x.data_ptr(),
                              scale.data_ptr(), ws, ws_bytes, rows, cols, rows / a.n, (float)eps,
                              on.stream); });
}

bool rmsnorm_forward(const Tensor& x, const Tensor& weight, double eps, bool save, Forward* f) {
  if (!activation(x) || !plain(weight)) return false;
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  const bool f32 = weight.scalar_type() == at::kFloat;
  if ((!f32 && weight.scalar_type() != at::kBFloat16) || weight.device() != x.device() || weight.dim() < 1 ||
      weight.size(-1) != cols || weight.numel() != cols || !weight.is_contiguous())
    return false;
  Launch on(x);
  const Tensor y = f->y = at::empty_like(x), kept = f->kept = f32 && save ? at::empty({cols}, x.options()) : weight;
  return launched([&] {
    return f32 ? tt_rmsnorm_forward_f32_weight(y.data_ptr(), x.data_ptr(), static_cast<const float*>(weight.data_ptr()),
                                                     copy_of(weight, kept), rows, cols, (float)eps, on.stream)
                     : tt_rmsnorm_forward(y.data_ptr(), x.data_ptr(), weight.data_ptr(), nullptr, rows, cols, (float)eps,
                                          on.stream);
  });
}

// freqs: none, or fp32 [seq, head_dim / 2, 2]; heads 0: all heads of a token in one row.
bool rope_forward(const Tensor& x, const Tensor& weight, const Tensor& freqs, double eps, int64_t head_dim,
                  int64_t heads, Forward* f) {
  Vectors w;
  if (!activation(x) || !vectors(weight, x, x.size(-1), &w) || w.n != 1 || !plain(freqs) || freqs.device() != x.device() ||
      freqs.scalar_type() != at::kFloat || !freqs.is_contiguous() || freqs.numel() == 0 || head_dim <= 0 ||
      freqs.numel() % head_dim != 0)
    return false;
  const int64_t cols = x.size(-1), rows = x.numel() / cols, seq = freqs.numel() / head_dim;
  if (heads == 0 ? x.dim() < 2 || x.size(-2) != seq : x.dim() < 3 || x.size(-2) != heads || x.size(-3) != seq)
    return false;
  Launch on(x);
  const Tensor y = f->y = at::empty_like(x);
  const float* table = static_cast<const float*>(freqs.data_ptr());
  return launched([&] {
    return heads == 0 ? tt_rmsnorm_rope_forward(y.data_ptr(), x.data_ptr(), weight.data_ptr(), table, nullptr, rows, cols,
                                                      head_dim, seq, (float)eps, on.stream)
                            : tt_rmsnorm_rope_heads_forward(y.data_ptr(), x.data_ptr(), weight.data_ptr(), table, nullptr, rows,
                                                            cols, heads, seq, (float)eps, on.stream);
  });
}

bool rmsnorm_backward(const Tensor& dy, const Tensor& x, const Tensor& weight, const optional<Tensor>& freqs, double eps,
                      int64_t head_dim, int64_t heads, bool bf16, at::IntArrayRef weight_shape, Backward* g) {
  Vectors w;
  if (!activation(x) || !like(dy, x) || !vectors(weight, x, x.size(-1), &w) || w.n != 1 || !aligned({&x, &dy, &weight}))
    return false;
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  int64_t seq = 0;
  if (freqs) {
    if (!plain(*freqs) || freqs->device() != x.device() || freqs->scalar_type() != at::kFloat || !freqs->is_contiguous() ||
        head_dim <= 0 || freqs->numel() == 0 || freqs->numel() % head_dim != 0)
      return false;
    seq = freqs->numel() / head_dim;
  }
  Launch on(x);
  const Tensor dx = g->dx = at::empty_like(x), dweight = g->d1 = at::empty(weight_shape, x.options().dtype(bf16 ? at::kBFloat16 : at::kFloat));
  if (dweight.numel() != cols) return false;
  return launched(tt_rmsnorm_backward_workspace_bytes(rows, cols), x,
                [&](void* ws, size_t ws_bytes) { return tt_rmsnorm_backward_typed(dx.data_ptr(), dweight.data_ptr(), bf16, dy.data_ptr(), x.data_ptr(), weight.data_ptr(),
                                freqs ? static_cast<const float*>(freqs->data_ptr()) : nullptr, head_dim, heads, seq,
                                ws, ws_bytes, rows, cols, (float)eps, on.stream); });
}

bool gate_forward(const Tensor& x, const Tensor& gate, const Tensor& residual, bool save, Forward* f) {
  if (!activation(x) || !like(residual, x)) return false;
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  Vectors g;
  if (!vectors(gate, x, cols, &g) || rows % g.n != 0) return false;
  Launch on(x);
  const Tensor out = f->y = at::empty_like(x), kept = f->kept = dense(gate, save, g.n, cols);
  return launched([&] { return tt_gate_residual_forward_strided(out.data_ptr(), x.data_ptr(), gate.data_ptr(), g.stride, copy_of(gate, kept),
                                       residual.data_ptr(), rows, cols, rows / g.n, on.stream); });
}

bool gate_backward(const Tensor& dout, const Tensor& gate, const Tensor& residual, bool bf16, at::IntArrayRef gate_shape,
                   Backward* b) {
  if (!activation(dout) || !like(residual, dout)) return false;
  const int64_t cols = dout.size(-1), rows = dout.numel() / cols;
  Vectors g;
  if (!vectors(gate, dout, cols, &g) || !gate.is_contiguous() || rows % g.n != 0) return false;
  Launch on(dout);
  const Tensor dres = b->d2 = at::empty_like(dout), dgate = b->d1 = at::empty(gate_shape, dout.options().dtype(bf16 ? at::kBFloat16 : at::kFloat));
  if (dgate.numel() != g.n * cols) return false;
  return launched(tt_gate_residual_backward_workspace_bytes(rows, cols, rows / g.n), dout,
                [&](void* ws, size_t ws_bytes) { return tt_gate_residual_backward_typed(dres.data_ptr(), dgate.data_ptr(), bf16, dout.data_ptr(), gate.data_ptr(),
                                      residual.data_ptr(), ws, ws_bytes, rows, cols, rows / g.n,
                                      on.stream); });
}

bool residual_norm_forward(const Tensor& x, const Tensor& r, const optional<Tensor>& gate, const Tensor& scale,
                           const Tensor& shift, double eps, bool affine, bool save, Forward* f) {
  if (!activation(x) || !like(r, x)) return false;
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  Vectors a, b, g;
  g.n = 1;
  if (!vectors(scale, x, cols, &a) || !vectors(shift, x, cols, &b) || a.n != b.n) return false;
  if (gate && !vectors(*gate, x, cols, &g)) return false;
  const int64_t nb = a.n > g.n ? a.n : g.n;
  if ((a.n != 1 && a.n != nb) || (g.n != 1 && g.n != nb) || rows % nb != 0) return false;
  Launch on(x);
  const Tensor s = f->s = at::empty_like(x), y = f->y = at::empty_like(x), kept = f->kept = dense(scale, save, a.n, cols);
  const Tensor kept_gate = f->kept_gate = gate ? dense(*gate, save, g.n, cols) : Tensor();
  return launched([&] { return tt_residual_norm_forward_strided(s.data_ptr(), y.data_ptr(), x.data_ptr(), r.data_ptr(), gate ? gate->data_ptr() : nullptr,
                                       g.n, g.stride, gate ? copy_of(*gate, kept_gate) : nullptr, scale.data_ptr(), a.stride,
                                       copy_of(scale, kept), shift.data_ptr(), b.stride, a.n, affine, nullptr, nullptr,
                                       rows, cols, rows / nb, (float)eps, on.stream); });
}

bool residual_norm_backward(const Tensor& dy, const optional<Tensor>& ds_in, const Tensor& s, const optional<Tensor>& r,
                            const optional<Tensor>& gate, const Tensor& scale, double eps, bool affine, bool bf16, Backward* b) {
  if (!activation(s) || !like(dy, s) || (ds_in && !like(*ds_in, s)) || (gate && (!r || !like(*r, s)))) return false;
  const int64_t cols = s.size(-1), rows = s.numel() / cols;
  Vectors a, g;
  g.n = 1;
  if (!vectors(scale, s, cols, &a) || !scale.is_contiguous()) return false;
  if (gate && (!vectors(*gate, s, cols, &g) || !gate->is_contiguous())) return false;
  const int64_t nb = a.n > g.n ? a.n : g.n;
  if ((a.n != 1 && a.n != nb) || (g.n != 1 && g.n != nb) || rows % nb != 0) return false;
  Launch on(s);
  const auto opts = s.options().dtype(bf16 ? at::kBFloat16 : at::kFloat);
  const Tensor dx = b->dx = at::empty_like(s), dr = b->d1 = gate ? at::empty_like(s) : dx,
               dscale = b->d3 = at::empty({nb, cols}, opts), dshift = b->d4 = at::empty({nb, cols}, opts),
               dgate = b->d2 = gate ? at::empty({nb, cols}, opts) : Tensor();
  return launched(tt_residual_norm_backward_workspace_bytes(rows, cols, rows / nb, gate ? 1 : 0), s,
                [&](void* ws, size_t ws_bytes) { return tt_residual_norm_backward_typed(dx.data_ptr(), gate ? dr.data_ptr() : nullptr, dscale.data_ptr(), dshift.data_ptr(),
                                      gate ? dgate.data_ptr() : nullptr, bf16, dy.data_ptr(), ds_in ? ds_in->data_ptr() : nullptr,
                                      s.data_ptr(), gate ? r->data_ptr() : nullptr, gate ? gate->data_ptr() : nullptr, g.n,
                                      scale.data_ptr(), a.n, affine, ws, ws_bytes, rows, cols, rows / nb, (float)eps,
                                      on.stream); });
}

// ---------------------------------------------------------------- the operators as autograd nodes
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Where a backward's gradients are not what the functions above take (another dtype, an address that is not 16-byte
// aligned), ops.py computes it, with its own checks and errors: name -> function.
py::dict& python_backwards() {
  static auto* d = new py::dict();
  return *d;
}
template <typename... A>
Backward python_backward(const char* name, const A&... args) {
  py::gil_scoped_acquire gil;
  try {
    const py::tuple out = python_backwards()[name](args...);
    Backward g;
    Tensor* to[] = {&g.dx, &g.d1, &g.d2, &g.d3, &g.d4};
    for (size_t i = 0; i < out.size(); ++i)
      if (!out[i].is_none()) *to[i] = py::cast<Tensor>(out[i]);
    return g;
  } catch (py::error_already_set& e) {   // crosses the engine's thread as torch's own exceptions do
    e.restore();
    python_error error;
    error.persist();
    throw error;
  }
}

Tensor needed(AutogradContext* ctx, size_t edge, const Tensor& g) { return ctx->needs_input_grad(edge) ? g : Tensor(); }
optional<Tensor> maybe(const Tensor& t) { return t.defined() ? optional<Tensor>(t) : std::nullopt; }

// A node's forward only records what has been computed: `f`, passed as something that is no input of the graph.
struct Done {
  Forward f;
  double eps = 0;
  int64_t head_dim = 0, heads = 0;   // rotary embedding: heads 0, or one head a row
  bool affine = false, transposed = false;
};

struct AdaLNModelFunction : torch::autograd::Function<AdaLNModelFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& scale, const Tensor& shift, const Done& d) {
    ctx->save_for_backward({x, d.f.kept});
    ctx->saved_data["eps"] = d.eps;
    ctx->saved_data["scale"] = scale.sizes().vec();
    ctx->saved_data["shift"] = shift.sizes().vec();
    return d.f.y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const double eps = ctx->saved_data["eps"].toDouble();
    const auto scale = ctx->saved_data["scale"].toIntVector(), shift = ctx->saved_data["shift"].toIntVector();
    const Tensor dy = grads[0].contiguous();
    Backward g;
    if (!tried([&] { return adaln_backward(dy, saved[0], saved[1], eps, true, scale, shift, &g); })) {
      g = python_backward("adaln", dy, saved[0], saved[1], eps);
      g.d1 = g.d1.reshape(scale);
      g.d2 = g.d2.reshape(shift);
    }
    return {needed(ctx, 0, g.dx), needed(ctx, 1, g.d1), needed(ctx, 2, g.d2), Tensor()};
  }
};

// RMSNorm, alone and with the rotary embedding behind it.
struct RMSNormModelFunction : torch::autograd::Function<RMSNormModelFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const Tensor* freqs, const Done& d) {
    ctx->save_for_backward({x, d.f.kept, freqs ? *freqs : Tensor()});
    ctx->saved_data["eps"] = d.eps;
    ctx->saved_data["weight"] = weight.sizes().vec();
    ctx->saved_data["bf16"] = weight.scalar_type() == at::kBFloat16;
    ctx->saved_data["head_dim"] = d.head_dim;
    ctx->saved_data["heads"] = d.heads;
    ctx->saved_data["transposed"] = d.transposed;
    return d.transposed ? d.f.y.transpose(-2, -3) : d.f.y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    auto& data = ctx->saved_data;
    const double eps = data["eps"].toDouble();
    const int64_t head_dim = data["head_dim"].toInt(), heads = data["heads"].toInt();
    const bool bf16 = data["bf16"].toBool(), transposed = data["transposed"].toBool();
    const auto shape = data["weight"].toIntVector();
    const auto freqs = maybe(saved[2]);
    const Tensor x = transposed ? saved[0].transpose(-2, -3) : saved[0];
    const Tensor dy = (transposed ? grads[0].transpose(-2, -3) : grads[0]).contiguous();
    Backward g;
    if (!tried([&] { return rmsnorm_backward(dy, x, saved[1], freqs, eps, head_dim, heads, bf16, shape, &g); })) {
      g = python_backward("rmsnorm", dy, x, saved[1], freqs, eps, head_dim, heads, bf16);
      g.d1 = g.d1.reshape(shape);
    }
    return {needed(ctx, 0, transposed ? g.dx.transpose(-2, -3) : g.dx), needed(ctx, 1, g.d1), Tensor(), Tensor()};
  }
};

struct GateResidualFunction : torch::autograd::Function<GateResidualFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& gate, const Tensor& residual, const Done& d) {
    ctx->save_for_backward({d.f.kept, residual});
    ctx->saved_data["gate"] = gate.sizes().vec();
    return d.f.y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const auto shape = ctx->saved_data["gate"].toIntVector();
    Backward g;
    if (ctx->needs_input_grad(1) || ctx->needs_input_grad(2)) {
      const Tensor dout = grads[0].contiguous();
      if (!tried([&] { return gate_backward(dout, saved[0], saved[1], true, shape, &g); })) {
        g = python_backward("gate", dout, saved[0], saved[1]);
        g.d1 = g.d1.reshape(shape);
      }
    }
    return {needed(ctx, 0, grads[0]), needed(ctx, 1, g.d1), needed(ctx, 2, g.d2), Tensor()};
  }
};

struct ResidualNormFunction : torch::autograd::Function<ResidualNormFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& r, const optional<Tensor>& gate,
                               const Tensor& scale, const Tensor& shift, const Done& d) {
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({d.f.s, gate ? r : Tensor(), d.f.kept_gate, d.f.kept});
    ctx->saved_data["eps"] = d.eps;
    ctx->saved_data["affine"] = d.affine;
    ctx->saved_data["gate"] = gate ? gate->sizes().vec() : std::vector<int64_t>();
    ctx->saved_data["scale"] = scale.sizes().vec();
    ctx->saved_data["shift"] = shift.sizes().vec();
    return {d.f.s, d.f.y};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &s = saved[0], &kept_gate = saved[2], &kept = saved[3];
    auto& data = ctx->saved_data;
    const double eps = data["eps"].toDouble();
    const bool affine = data["affine"].toBool(), gated = kept_gate.defined();
    const std::vector<int64_t> shapes[] = {data["gate"].toIntVector(), data["scale"].toIntVector(), data["shift"].toIntVector()};
    // one rounding in the kernel where every gradient leaves as it is: one vector per batch
    const int64_t n = gated && kept_gate.numel() > kept.numel() ? kept_gate.numel() : kept.numel();
    bool direct = true;
    for (int i = gated ? 0 : 1; i < 3; ++i) direct = direct && c10::multiply_integers(shapes[i]) == n;
    const Tensor dy = grads[1].defined() ? grads[1].contiguous() : at::zeros_like(s);
    const optional<Tensor> ds = grads[0].defined() ? optional<Tensor>(grads[0].contiguous()) : std::nullopt;
    Backward g;
    if (!tried([&] { return residual_norm_backward(dy, ds, s, maybe(saved[1]), maybe(kept_gate), kept, eps, affine, direct, &g); }))
      g = python_backward("residual_norm", dy, ds, s, maybe(saved[1]), maybe(kept_gate), kept, eps, affine, direct);
    const auto param = [&](size_t edge, const Tensor& t, const std::vector<int64_t>& shape) {
      if (!ctx->needs_input_grad(edge)) return Tensor();
      const Tensor sum = t.numel() == c10::multiply_integers(shape) ? t : t.sum(0);   // one vector shared by several batches
      return sum.to(at::kBFloat16).reshape(shape);
    };
    const size_t e = gated ? 1 : 0;   // an absent gate has no edge
    return {needed(ctx, 0, g.dx), needed(ctx, 1, g.d1), gated ? param(2, g.d2, shapes[0]) : Tensor(),
            param(2 + e, g.d3, shapes[1]), param(3 + e, g.d4, shapes[2]), Tensor()};
  }
};

// The contract of reference_api.py: x_norm and the row statistics are saved.
struct SavedAdaLNFunction : torch::autograd::Function<SavedAdaLNFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& scale, const Tensor& shift, const Done& d) {
    ctx->save_for_backward({d.f.s, scale, d.f.kept});
    return d.f.y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x_norm = saved[0], &scale = saved[1], &rstd = saved[2], dy = grads[0].contiguous();
    const int64_t cols = scale.numel(), rows = rstd.numel();
    tt_glue::check_act(dy, "dout", rows, cols);
    Launch on(dy);
    const Tensor dx = at::empty_like(x_norm), dscale = at::empty_like(scale), dshift = at::empty_like(scale);
    const int rc = tt_glue::with_workspace(tt_adaln_backward_workspace_bytes(rows, cols, rows), dy, [&](void* ws, size_t bytes) {
      return tt_launch_adaln_backward(dx.data_ptr(), dscale.data_ptr(), dshift.data_ptr(), dy.data_ptr(), x_norm.data_ptr(),
                                      scale.data_ptr(), static_cast<const float*>(rstd.data_ptr()), rows, cols, ws, bytes,
                                      on.stream);
    });
    tt_glue::check_status(rc, "torch_launch_adaln_backward");
    return {needed(ctx, 0, dx), needed(ctx, 1, dscale), needed(ctx, 2, dshift), Tensor()};
  }
};

// Arguments of a Function's apply, as long as they are what these nodes take.
struct Call {
  const py::args& a;
  bool ok;
  Call(const py::args& args, size_t least, size_t most) : a(args), ok(args.size() >= least && args.size() <= most) {
    // a tracer has to see the Python class (functorch's transforms: see NativeFirst in functional.py)
    ok = ok && !torch::jit::tracer::isTracing();
  }
  const Tensor& tensor(size_t i) {
    static const Tensor none;
    if (!ok || !(ok = THPVariable_CheckExact(a[i].ptr()))) return none;
    const Tensor& t = THPVariable_Unpack(a[i].ptr());
    ok = t.defined() && !t._fw_grad(0).defined();
    return t;
  }
  double number(size_t i) {
    if (!ok || !(ok = PyFloat_Check(a[i].ptr()) || PyLong_Check(a[i].ptr()))) return 0;
    return py::cast<double>(a[i]);
  }
  int64_t integer(size_t i) {
    if (!ok || !(ok = PyLong_Check(a[i].ptr()))) return 0;
    return py::cast<int64_t>(a[i]);
  }
};
bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}
// As _check_row_groups of functional.py, which names the error.
bool row_groups(const Tensor& x, const Tensor& p) {
  if (x.dim() < 3 || p.dim() != x.dim()) return true;
  bool broadcasting = false;
  for (int64_t i = 0; i < x.dim() - 1; ++i) {
    if (p.size(i) == x.size(i) && (!broadcasting || p.size(i) == 1)) continue;
    if (p.size(i) != 1) return false;
    broadcasting = true;
  }
  return p.size(-1) == x.size(-1);
}
// Exceptions of Python code inside (hooks on saved tensors) go on as they are.
template <typename F>
py::object graph(F f) {
  try {
    return f();
  } catch (python_error& e) {
    e.restore();
    throw py::error_already_set();
  }
}

py::object adaln(const py::args& args) {
  Call c(args, 5, 5);
  const Tensor &x = c.tensor(0), &scale = c.tensor(1), &shift = c.tensor(2);
  Done d;
  d.eps = c.number(3);
  const int64_t cols = c.integer(4);
  if (!c.ok || x.dim() < 1 || x.size(-1) != cols || !row_groups(x, scale) || !row_groups(x, shift)) return py::none();
  const bool save = wants_grad({&x, &scale, &shift});
  if (!tried([&] { return adaln_forward(x, scale, shift, d.eps, save, &d.f); })) return py::none();
  return save ? graph([&] { return py::cast(AdaLNModelFunction::apply(x, scale, shift, d)); }) : py::cast(d.f.y);
}

py::object rmsnorm(const py::args& args) {
  Call c(args, 4, 4);
  const Tensor &x = c.tensor(0), &weight = c.tensor(1);
  Done d;
  d.eps = c.number(2);
  const int64_t cols = c.integer(3);
  if (!c.ok || x.dim() < 1 || x.size(-1) != cols) return py::none();
  const bool save = wants_grad({&x, &weight});
  if (!tried([&] { return rmsnorm_forward(x, weight, d.eps, save, &d.f); })) return py::none();
  if (!save) return py::cast(d.f.y);
  return graph([&] { return py::cast(RMSNormModelFunction::apply(x, weight, static_cast<const Tensor*>(nullptr), d)); });
}

// heads_apart: x [B, S, H, D], or its [B, H, S, D] transposed view; otherwise all heads of a token in one row.
py::object rope(const py::args& args, bool heads_apart) {
  Call c(args, heads_apart ? 4 : 5, heads_apart ? 4 : 5);
  const Tensor &x = c.tensor(0), &weight = c.tensor(1), &freqs = c.tensor(2);
  Done d;
  d.eps = c.number(3);
  const int64_t n = heads_apart ? 1 : c.integer(4);
  if (!c.ok || x.dim() < 1 || n <= 0 || x.size(-1) % n != 0) return py::none();
  d.head_dim = x.size(-1) / n;
  if (freqs.dim() != 3 || freqs.size(1) * 2 != d.head_dim || freqs.size(2) != 2 || freqs.requires_grad() ||
      weight.scalar_type() != at::kBFloat16 || !weight.is_contiguous() || weight.numel() != x.size(-1))
    return py::none();
  Tensor rows = x;   // in memory order
  if (heads_apart) {
    if (x.dim() != 4) return py::none();
    if (!x.is_contiguous()) {
      if (x.stride(0) < x.stride(2) || x.stride(2) <= x.stride(1)) return py::none();
      d.transposed = true;
      at::NoGradGuard no_grad;
      rows = x.transpose(1, 2);
    }
    d.heads = rows.size(2);
  }
  const bool save = wants_grad({&x, &weight});
  if (!tried([&] { return rope_forward(rows, weight, freqs, d.eps, d.head_dim, d.heads, &d.f); })) return py::none();
  d.f.kept = weight;
  if (!save) return py::cast(d.transposed ? d.f.y.transpose(1, 2) : d.f.y);
  return graph([&] { return py::cast(RMSNormModelFunction::apply(x, weight, &freqs, d)); });
}

py::object gate_residual(const py::args& args) {
  Call c(args, 3, 3);
  const Tensor &x = c.tensor(0), &gate = c.tensor(1), &residual = c.tensor(2);
  if (!c.ok || !row_groups(x, gate)) return py::none();
  Done d;
  const bool save = wants_grad({&x, &gate, &residual});
  if (!tried([&] { return gate_forward(x, gate, residual, save, &d.f); })) return py::none();
  return save ? graph([&] { return py::cast(GateResidualFunction::apply(x, gate, residual, d)); }) : py::cast(d.f.y);
}

py::object residual_norm(const py::args& args) {
  Call c(args, 7, 8);
  if (c.ok && args.size() == 8 && !args[7].is_none()) return py::none();   // a reduction hook
  const Tensor &x = c.tensor(0), &r = c.tensor(1);
  const optional<Tensor> gate = c.ok && !args[2].is_none() ? optional<Tensor>(c.tensor(2)) : std::nullopt;
  const Tensor &scale = c.tensor(3), &shift = c.tensor(4);
  Done d;
  d.eps = c.number(5);
  if (!c.ok || !PyBool_Check(args[6].ptr())) return py::none();
  d.affine = py::cast<bool>(args[6]);
  if ((gate && !row_groups(x, *gate)) || !row_groups(x, scale) || !row_groups(x, shift)) return py::none();
  const Tensor no_gate;
  const bool save = wants_grad({&x, &r, gate ? &*gate : &no_gate, &scale, &shift});
  if (!tried([&] { return residual_norm_forward(x, r, gate, scale, shift, d.eps, d.affine, save, &d.f); })) return py::none();
  if (!save) return py::make_tuple(d.f.s, d.f.y);
  return graph([&] {
    const auto out = ResidualNormFunction::apply(x, r, gate, scale, shift, d);
    return py::object(py::make_tuple(out[0], out[1]));
  });
}

py::object adaln_saved(const py::args& args) {
  Call c(args, 5, 5);
  const Tensor &x = c.tensor(0), &scale = c.tensor(1), &shift = c.tensor(2);
  Done d;
  d.eps = c.number(3);
  const int64_t cols = c.integer(4);
  if (!c.ok || !activation(x) || cols <= 0 || x.numel() % cols != 0) return py::none();
  for (const Tensor* p : {&scale, &shift})
    if (!plain(*p) || p->scalar_type() != at::kBFloat16 || p->device() != x.device() || !p->is_contiguous() || p->numel() != cols)
      return py::none();
  const int64_t rows = x.numel() / cols;
  const bool done = tried([&] {
    Launch on(x);
    d.f.y = at::empty_like(x);
    d.f.s = at::empty_like(x);
    d.f.kept = at::empty({rows}, x.options().dtype(at::kFloat));
    return launched([&] { return tt_launch_adaln_forward(d.f.y.data_ptr(), d.f.s.data_ptr(), x.data_ptr(), scale.data_ptr(),
                                                         shift.data_ptr(), rows, cols, d.eps,
                                                         static_cast<float*>(d.f.kept.data_ptr()), on.stream); });
  });
  if (!done) return py::none();
  if (!wants_grad({&x, &scale, &shift})) return py::cast(d.f.y);
  return graph([&] { return py::cast(SavedAdaLNFunction::apply(x, scale, shift, d)); });
}

}  // namespace

// The operators' halves, for ops.py and the Functions' own forward and backward.
PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  using V = std::vector<int64_t>;
  using T = const Tensor&;
  using O = const optional<Tensor>&;
  const auto none = [] { return py::object(py::none()); };
  m.def("adaln_forward", [none](T x, T scale, T shift, double eps, bool save) {
    Forward f;
    return tried([&] { return adaln_forward(x, scale, shift, eps, save, &f); }) ? py::make_tuple(f.y, f.kept) : none();
  });
  m.def("adaln_backward", [none](T dy, T x, T scale, double eps, bool bf16, const V& scale_shape, const V& shift_shape) {
    Backward g;
    return tried([&] { return adaln_backward(dy, x, scale, eps, bf16, scale_shape, shift_shape, &g); })
               ? py::make_tuple(g.dx, g.d1, g.d2) : none();
  });
  m.def("rmsnorm_forward", [none](T x, T weight, double eps, bool save) {
    Forward f;
    return tried([&] { return rmsnorm_forward(x, weight, eps, save, &f); }) ? py::make_tuple(f.y, f.kept) : none();
  });
  m.def("rope_forward", [none](T x, T weight, T freqs, double eps, int64_t head_dim, int64_t heads) {
    Forward f;
    return tried([&] { return rope_forward(x, weight, freqs, eps, head_dim, heads, &f); }) ? py::cast(f.y) : none();
  });
  m.def("rmsnorm_backward", [none](T dy, T x, T weight, O freqs, double eps, int64_t head_dim, int64_t heads, bool bf16, const V& shape) {
    Backward g;
    return tried([&] { return rmsnorm_backward(dy, x, weight, freqs, eps, head_dim, heads, bf16, shape, &g); })
               ? py::make_tuple(g.dx, g.d1) : none();
  });
  m.def("gate_forward", [none](T x, T gate, T residual, bool save) {
    Forward f;
    return tried([&] { return gate_forward(x, gate, residual, save, &f); }) ? py::make_tuple(f.y, f.kept) : none();
  });
  m.def("gate_backward", [none](T dout, T gate, T residual, bool bf16, const V& shape) {
    Backward g;
    return tried([&] { return gate_backward(dout, gate, residual, bf16, shape, &g); }) ? py::make_tuple(g.d2, g.d1) : none();
  });
  m.def("residual_norm_forward", [none](T x, T r, O gate, T scale, T shift, double eps, bool affine, bool save) {
    Forward f;
    return tried([&] { return residual_norm_forward(x, r, gate, scale, shift, eps, affine, save, &f); })
               ? py::make_tuple(f.s, f.y, maybe(f.kept_gate), f.kept) : none();
  });
  m.def("residual_norm_backward", [none](T dy, O ds, T s, O r, O gate, T scale, double eps, bool affine, bool bf16) {
    Backward g;
    return tried([&] { return residual_norm_backward(dy, ds, s, r, gate, scale, eps, affine, bf16, &g); })
               ? py::make_tuple(g.dx, g.d1, g.d3, g.d4, maybe(g.d2)) : none();
  });
  m.def("clear_workspaces", &clear_workspaces);
  // What the Functions' apply returns, or None.
  m.def("adaln", &adaln);
  m.def("rmsnorm", &rmsnorm);
  m.def("rope", [](const py::args& a) { return rope(a, false); });
  m.def("rope_heads", [](const py::args& a) { return rope(a, true); });
  m.def("gate_residual", &gate_residual);
  m.def("residual_norm", &residual_norm);
  m.def("adaln_saved", &adaln_saved);
  m.def("set_python_backwards", [](const py::dict& d) { python_backwards() = d; });
}
