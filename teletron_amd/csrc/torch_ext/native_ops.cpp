// Python module `native_ops`: the operators of teletron_amd/ops.py as one call each, for the tensors a
// model passes in earnest (dense bf16 activations, evenly spaced bf16 or fp32 parameters).  Checks,
// output allocation, workspace and launch cost 25-45 us of Python and ctypes per operator, several
// times the kernels' own time for a text-token tensor (512 x 5120: 4 us forward, 10 us backward).  A function returns
// None, and has done nothing, wherever its arguments are anything else: ops.py then takes the call, with
// its own checks and errors.  Holds no kernels.
#include "glue.hpp"

#include <ATen/TensorSubclassLikeUtils.h>

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

// The launch itself may wait for room in the queue: other Python threads run meanwhile.
template <typename F>
bool launched(F f) {
  py::gil_scoped_release unlocked;
  return f() == TT_OK;
}
// The same with the backward workspace: f(memory, bytes).
template <typename F>
bool launched(size_t bytes, const Tensor& ref, F f) {
  return tt_glue::with_workspace(bytes, ref, f) == TT_OK;
}
// Errors of the allocator and of tensors without memory are raised by ops.py, as its own types.
template <typename... A>
auto guarded(py::object (*f)(A...)) {
  return [f](A... a) -> py::object {
    try {
      return f(a...);
    } catch (const c10::Error&) {
      return py::none();
    }
  };
}

py::object adaln_forward(const Tensor& x, const Tensor& scale, const Tensor& shift, double eps, bool save) {
  if (!activation(x)) return py::none();
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  Vectors a, b;
  if (!vectors(scale, x, cols, &a) || !vectors(shift, x, cols, &b) || a.n != b.n || rows % a.n != 0) return py::none();
  Launch on(x);
  Tensor y = at::empty_like(x), kept = dense(scale, save, a.n, cols);
  if (!launched([&] { return tt_adaln_forward_strided(y.data_ptr(), x.data_ptr(), scale.data_ptr(), a.stride, shift.data_ptr(), b.stride,
                               copy_of(scale, kept), rows, cols, rows / a.n, (float)eps, on.stream); }))
    return py::none();
  return py::make_tuple(y, kept);
}

py::object adaln_backward(const Tensor& dy, const Tensor& x, const Tensor& scale, double eps, bool bf16,
                          const std::vector<int64_t>& scale_shape, const std::vector<int64_t>& shift_shape) {
  if (!activation(x) || !like(dy, x)) return py::none();
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  Vectors a;
  if (!vectors(scale, x, cols, &a) || !scale.is_contiguous() || rows % a.n != 0 || !aligned({&x, &dy, &scale}))
    return py::none();
  Launch on(x);
  const auto opts = x.options().dtype(bf16 ? at::kBFloat16 : at::kFloat);
  Tensor dx = at::empty_like(x), dscale = at::empty(scale_shape, opts), dshift = at::empty(shift_shape, opts);
  if (dscale.numel() != a.n * cols || dshift.numel() != a.n * cols) return py::none();
  if (!launched(tt_adaln_backward_workspace_bytes(rows, cols, rows / a.n), x,
                [&](void* ws, size_t ws_bytes) { return tt_adaln_backward_typed(dx.data_ptr(), dscale.data_ptr(), dshift.data_ptr(), bf16, dy.data_ptr(), x.data_ptr(),
                              scale.data_ptr(), ws, ws_bytes, rows, cols, rows / a.n, (float)eps,
                              on.stream); }))
    return py::none();
  return py::make_tuple(dx, dscale, dshift);
}

py::object rmsnorm_forward(const Tensor& x, const Tensor& weight, double eps, bool save) {
  if (!activation(x) || !plain(weight)) return py::none();
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  const bool f32 = weight.scalar_type() == at::kFloat;
  if ((!f32 && weight.scalar_type() != at::kBFloat16) || weight.device() != x.device() || weight.dim() < 1 ||
      weight.size(-1) != cols || weight.numel() != cols || !weight.is_contiguous())
    return py::none();
  Launch on(x);
  Tensor y = at::empty_like(x), kept = f32 && save ? at::empty({cols}, x.options()) : weight;
  const bool ok = launched([&] {
    return f32 ? tt_rmsnorm_forward_f32_weight(y.data_ptr(), x.data_ptr(), static_cast<const float*>(weight.data_ptr()),
                                                     copy_of(weight, kept), rows, cols, (float)eps, on.stream)
                     : tt_rmsnorm_forward(y.data_ptr(), x.data_ptr(), weight.data_ptr(), nullptr, rows, cols, (float)eps,
                                          on.stream);
  });
  if (!ok) return py::none();
  return py::make_tuple(y, kept);
}

// freqs: none, or fp32 [seq, head_dim / 2, 2]; heads 0: all heads of a token in one row.
py::object rope_forward(const Tensor& x, const Tensor& weight, const Tensor& freqs, double eps, int64_t head_dim,
                        int64_t heads) {
  Vectors w;
  if (!activation(x) || !vectors(weight, x, x.size(-1), &w) || w.n != 1 || !plain(freqs) || freqs.device() != x.device() ||
      freqs.scalar_type() != at::kFloat || !freqs.is_contiguous() || freqs.numel() == 0 || head_dim <= 0 ||
      freqs.numel() % head_dim != 0)
    return py::none();
  const int64_t cols = x.size(-1), rows = x.numel() / cols, seq = freqs.numel() / head_dim;
  if (heads == 0 ? x.dim() < 2 || x.size(-2) != seq : x.dim() < 3 || x.size(-2) != heads || x.size(-3) != seq)
    return py::none();
  Launch on(x);
  Tensor y = at::empty_like(x);
  const float* f = static_cast<const float*>(freqs.data_ptr());
  const bool ok = launched([&] {
    return heads == 0 ? tt_rmsnorm_rope_forward(y.data_ptr(), x.data_ptr(), weight.data_ptr(), f, nullptr, rows, cols,
                                                      head_dim, seq, (float)eps, on.stream)
                            : tt_rmsnorm_rope_heads_forward(y.data_ptr(), x.data_ptr(), weight.data_ptr(), f, nullptr, rows,
                                                            cols, heads, seq, (float)eps, on.stream);
  });
  return ok ? py::cast(y) : py::object(py::none());
}

py::object rmsnorm_backward(const Tensor& dy, const Tensor& x, const Tensor& weight, const optional<Tensor>& freqs, double eps,
                            int64_t head_dim, int64_t heads, bool bf16, const std::vector<int64_t>& weight_shape) {
  Vectors w;
  if (!activation(x) || !like(dy, x) || !vectors(weight, x, x.size(-1), &w) || w.n != 1 || !aligned({&x, &dy, &weight}))
    return py::none();
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  int64_t seq = 0;
  if (freqs) {
    if (!plain(*freqs) || freqs->device() != x.device() || freqs->scalar_type() != at::kFloat || !freqs->is_contiguous() ||
        head_dim <= 0 || freqs->numel() == 0 || freqs->numel() % head_dim != 0)
      return py::none();
    seq = freqs->numel() / head_dim;
  }
  Launch on(x);
  Tensor dx = at::empty_like(x), dweight = at::empty(weight_shape, x.options().dtype(bf16 ? at::kBFloat16 : at::kFloat));
  if (dweight.numel() != cols) return py::none();
  if (!launched(tt_rmsnorm_backward_workspace_bytes(rows, cols), x,
                [&](void* ws, size_t ws_bytes) { return tt_rmsnorm_backward_typed(dx.data_ptr(), dweight.data_ptr(), bf16, dy.data_ptr(), x.data_ptr(), weight.data_ptr(),
                                freqs ? static_cast<const float*>(freqs->data_ptr()) : nullptr, head_dim, heads, seq,
                                ws, ws_bytes, rows, cols, (float)eps, on.stream); }))
    return py::none();
  return py::make_tuple(dx, dweight);
}

py::object gate_forward(const Tensor& x, const Tensor& gate, const Tensor& residual, bool save) {
  if (!activation(x) || !like(residual, x)) return py::none();
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  Vectors g;
  if (!vectors(gate, x, cols, &g) || rows % g.n != 0) return py::none();
  Launch on(x);
  Tensor out = at::empty_like(x), kept = dense(gate, save, g.n, cols);
  if (!launched([&] { return tt_gate_residual_forward_strided(out.data_ptr(), x.data_ptr(), gate.data_ptr(), g.stride, copy_of(gate, kept),
                                       residual.data_ptr(), rows, cols, rows / g.n, on.stream); }))
    return py::none();
  return py::make_tuple(out, kept);
}

py::object gate_backward(const Tensor& dout, const Tensor& gate, const Tensor& residual, bool bf16,
                         const std::vector<int64_t>& gate_shape) {
  if (!activation(dout) || !like(residual, dout)) return py::none();
  const int64_t cols = dout.size(-1), rows = dout.numel() / cols;
  Vectors g;
  if (!vectors(gate, dout, cols, &g) || !gate.is_contiguous() || rows % g.n != 0) return py::none();
  Launch on(dout);
  Tensor dres = at::empty_like(dout), dgate = at::empty(gate_shape, dout.options().dtype(bf16 ? at::kBFloat16 : at::kFloat));
  if (dgate.numel() != g.n * cols) return py::none();
  if (!launched(tt_gate_residual_backward_workspace_bytes(rows, cols, rows / g.n), dout,
                [&](void* ws, size_t ws_bytes) { return tt_gate_residual_backward_typed(dres.data_ptr(), dgate.data_ptr(), bf16, dout.data_ptr(), gate.data_ptr(),
                                      residual.data_ptr(), ws, ws_bytes, rows, cols, rows / g.n,
                                      on.stream); }))
    return py::none();
  return py::make_tuple(dres, dgate);
}

py::object residual_norm_forward(const Tensor& x, const Tensor& r, const optional<Tensor>& gate, const Tensor& scale,
                                 const Tensor& shift, double eps, bool affine, bool save) {
  if (!activation(x) || !like(r, x)) return py::none();
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  Vectors a, b, g;
  g.n = 1;
  if (!vectors(scale, x, cols, &a) || !vectors(shift, x, cols, &b) || a.n != b.n) return py::none();
  if (gate && !vectors(*gate, x, cols, &g)) return py::none();
  const int64_t nb = a.n > g.n ? a.n : g.n;
  if ((a.n != 1 && a.n != nb) || (g.n != 1 && g.n != nb) || rows % nb != 0) return py::none();
  Launch on(x);
  Tensor s = at::empty_like(x), y = at::empty_like(x), kept = dense(scale, save, a.n, cols), kept_gate;
  if (gate) kept_gate = dense(*gate, save, g.n, cols);
  if (!launched([&] { return tt_residual_norm_forward_strided(s.data_ptr(), y.data_ptr(), x.data_ptr(), r.data_ptr(), gate ? gate->data_ptr() : nullptr,
                                       g.n, g.stride, gate ? copy_of(*gate, kept_gate) : nullptr, scale.data_ptr(), a.stride,
                                       copy_of(scale, kept), shift.data_ptr(), b.stride, a.n, affine, nullptr, nullptr,
                                       rows, cols, rows / nb, (float)eps, on.stream); }))
    return py::none();
  return py::make_tuple(s, y, gate ? py::cast(kept_gate) : py::object(py::none()), kept);
}

py::object residual_norm_backward(const Tensor& dy, const optional<Tensor>& ds_in, const Tensor& s, const optional<Tensor>& r,
                                  const optional<Tensor>& gate, const Tensor& scale, double eps, bool affine, bool bf16) {
  if (!activation(s) || !like(dy, s) || (ds_in && !like(*ds_in, s)) || (gate && (!r || !like(*r, s)))) return py::none();
  const int64_t cols = s.size(-1), rows = s.numel() / cols;
  Vectors a, g;
  g.n = 1;
  if (!vectors(scale, s, cols, &a) || !scale.is_contiguous()) return py::none();
  if (gate && (!vectors(*gate, s, cols, &g) || !gate->is_contiguous())) return py::none();
  const int64_t nb = a.n > g.n ? a.n : g.n;
  if ((a.n != 1 && a.n != nb) || (g.n != 1 && g.n != nb) || rows % nb != 0) return py::none();
  Launch on(s);
  const auto opts = s.options().dtype(bf16 ? at::kBFloat16 : at::kFloat);
  Tensor dx = at::empty_like(s), dr = gate ? at::empty_like(s) : dx, dscale = at::empty({nb, cols}, opts),
         dshift = at::empty({nb, cols}, opts), dgate;
  if (gate) dgate = at::empty({nb, cols}, opts);
  if (!launched(tt_residual_norm_backward_workspace_bytes(rows, cols, rows / nb, gate ? 1 : 0), s,
                [&](void* ws, size_t ws_bytes) { return tt_residual_norm_backward_typed(dx.data_ptr(), gate ? dr.data_ptr() : nullptr, dscale.data_ptr(), dshift.data_ptr(),
                                      gate ? dgate.data_ptr() : nullptr, bf16, dy.data_ptr(), ds_in ? ds_in->data_ptr() : nullptr,
                                      s.data_ptr(), gate ? r->data_ptr() : nullptr, gate ? gate->data_ptr() : nullptr, g.n,
                                      scale.data_ptr(), a.n, affine, ws, ws_bytes, rows, cols, rows / nb, (float)eps,
                                      on.stream); }))
    return py::none();
  return py::make_tuple(dx, dr, dscale, dshift, gate ? py::cast(dgate) : py::object(py::none()));
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("adaln_forward", guarded(&adaln_forward));
  m.def("adaln_backward", guarded(&adaln_backward));
  m.def("rmsnorm_forward", guarded(&rmsnorm_forward));
  m.def("rope_forward", guarded(&rope_forward));
  m.def("rmsnorm_backward", guarded(&rmsnorm_backward));
  m.def("gate_forward", guarded(&gate_forward));
  m.def("gate_backward", guarded(&gate_backward));
  m.def("residual_norm_forward", guarded(&residual_norm_forward));
  m.def("residual_norm_backward", guarded(&residual_norm_backward));
  m.def("clear_workspaces", &clear_workspaces);
}
