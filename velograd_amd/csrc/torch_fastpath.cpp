// Host fast path for launch-bound calls (decode shapes, short training steps): each entry point's
// common case — contiguous tensors of one dtype on the current device — validated, allocated and
// launched in C++, so a Python call costs one pybind11 crossing instead of ctypes argument
// conversion plus the torch views and allocations from Python.  Calls that do not qualify return
// an empty list and take the general Python path (velograd_amd/kernels/__init__.py), which
// validates and raises.  The kernels are the C ABI's (include/velograd_kernels.h); this file only
// binds them to torch tensors.
#include <torch/extension.h>

#include <c10/hip/HIPStream.h>

#include <stdexcept>
#include <string>
#include <vector>

#include "velograd_kernels.h"

namespace {

int32_t dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return VELOGRAD_DTYPE_F32;
    case at::kHalf: return VELOGRAD_DTYPE_F16;
    case at::kBFloat16: return VELOGRAD_DTYPE_BF16;
    default: return -1;
  }
}

// [y, h, inv_rms] of velograd_rmsnorm_residual_fwd (min_mean_sq == 0) or velograd_rmsnorm_fwd,
// with h the very tensor x when residual is None; [] when the call does not qualify.
std::vector<at::Tensor> forward(const at::Tensor& x, const c10::optional<at::Tensor>& residual,
                                const c10::optional<at::Tensor>& weight, double eps,
                                double min_mean_sq) {
  const int32_t code = dtype_code(x.scalar_type());
  if (code < 0 || !x.is_cuda() || x.dim() == 0 || !x.is_contiguous() || x.numel() == 0) return {};
  if (x.get_device() != c10::hip::current_device()) return {};
  const int64_t d = x.size(-1);
  const int64_t rows = x.numel() / d;
  if (residual.has_value()) {
    const at::Tensor& r = *residual;
    if (r.scalar_type() != x.scalar_type() || !r.is_contiguous() || r.sizes() != x.sizes() ||
        r.device() != x.device())
      return {};
  }
  int32_t wcode = code;
  if (weight.has_value()) {
    const at::Tensor& w = *weight;
    if (w.dim() != 1 || w.size(0) != d || !w.is_contiguous() || w.device() != x.device())
      return {};
    wcode = dtype_code(w.scalar_type());
    if (wcode != code && wcode != VELOGRAD_DTYPE_F32) return {};
  }
  at::Tensor y = at::empty_like(x);
  at::Tensor h = residual.has_value() ? at::empty_like(x) : x;
  std::vector<int64_t> stat(x.sizes().begin(), x.sizes().end() - 1);
  stat.push_back(1);
  at::Tensor inv = at::empty(stat, x.options().dtype(at::kFloat));
  void* stream = c10::hip::getCurrentHIPStream(x.get_device()).stream();
  const void* rp = residual.has_value() ? residual->data_ptr() : nullptr;
  const void* wp = weight.has_value() ? weight->data_ptr() : nullptr;
  void* hp = residual.has_value() ? h.data_ptr() : nullptr;
  // Any nonzero floor (a negative or NaN one included) goes to the entry point that checks it.
  const int32_t rc =
      min_mean_sq != 0.0
          ? velograd_rmsnorm_fwd(x.data_ptr(), rp, wp, y.data_ptr(), hp, inv.data_ptr<float>(),
                                 rows, d, d, d, d, d, code, wcode, (float)eps, (float)min_mean_sq,
                                 stream)
          : velograd_rmsnorm_residual_fwd(x.data_ptr(), rp, wp, y.data_ptr(), hp,
                                          inv.data_ptr<float>(), rows, d, d, d, d, d, code, wcode,
                                          (float)eps, stream);
  if (rc != 0) {
    const std::string msg = std::string("velograd_rmsnorm forward failed (status ") +
                            std::to_string(rc) + "): " + velograd_kernels_last_error();
    if (rc == VELOGRAD_ERR_UNSUPPORTED_DTYPE) throw pybind11::type_error(msg);
    if (rc < 0) throw pybind11::value_error(msg);
    throw std::runtime_error(msg);
  }
  return {y, h, inv};
}

using OptTensor = c10::optional<at::Tensor>;
using Tensors = std::vector<at::Tensor>;

// The exceptions of velograd_amd/_lib.py's check() for a C status.
void check(int32_t rc, const char* what) {
  if (rc == 0) return;
  const std::string msg = std::string(what) + " failed (status " + std::to_string(rc) +
                          "): " + velograd_kernels_last_error();
  if (rc == VELOGRAD_ERR_UNSUPPORTED_DTYPE) throw pybind11::type_error(msg);
  if (rc == VELOGRAD_ERR_INVALID_ARGUMENT || rc == VELOGRAD_ERR_WORKSPACE_TOO_SMALL)
    throw pybind11::value_error(msg);
  throw std::runtime_error(msg);
}

// A plain dense tensor on the current device: data of its own to point at (no functorch or other
// wrapper, whose data the general path refuses), row-major, not empty.
bool plain(const at::Tensor& t) {
  return t.is_cuda() && t.has_storage() && !t.is_neg() &&
         !t.unsafeGetTensorImpl()->is_python_dispatch() &&
         t.layout() == at::kStrided && t.is_contiguous() && t.numel() > 0 &&
         t.get_device() == c10::hip::current_device();
}

// t, when given, is plain and shaped and typed like x.
bool like(const OptTensor& t, const at::Tensor& x) {
  return !t.has_value() || (plain(*t) && t->scalar_type() == x.scalar_type() &&
                            t->sizes() == x.sizes() && t->device() == x.device());
}

// The weight's dtype code (the activations' without one), -1 when it does not qualify.
int32_t weight_code(const OptTensor& w, const at::Tensor& x) {
  const int32_t code = dtype_code(x.scalar_type());
  if (!w.has_value()) return code;
  if (!plain(*w) || w->dim() != 1 || w->size(0) != x.size(-1) || w->device() != x.device())
    return -1;
  const int32_t wcode = dtype_code(w->scalar_type());
  return wcode == code || wcode == VELOGRAD_DTYPE_F32 ? wcode : -1;
}

const void* ptr(const OptTensor& t) { return t.has_value() ? t->data_ptr() : nullptr; }

std::vector<int64_t> with_last(const at::Tensor& x, int64_t last) {
  std::vector<int64_t> v(x.sizes().begin(), x.sizes().end());
  v.back() = last;
  return v;
}

at::Tensor row_stat(const at::Tensor& x) {
  return at::empty(with_last(x, 1), x.options().dtype(at::kFloat));
}

void* stream_of(const at::Tensor& x) {
  return c10::hip::getCurrentHIPStream(x.get_device()).stream();
}

// inv_rms as a backward takes it: one plain float per row.
bool stat_ok(const at::Tensor& inv_rms, const at::Tensor& x, int64_t rows) {
  return plain(inv_rms) && inv_rms.scalar_type() == at::kFloat && inv_rms.numel() == rows &&
         inv_rms.device() == x.device();
}

// [codes, scales, h, inv_rms] of the quantising forwards; mx_format < 0: fp8 with a scale per row.
Tensors forward_quantised(const at::Tensor& x, const OptTensor& residual, const OptTensor& weight,
                          double eps, int64_t mx_format) {
  const int32_t code = dtype_code(x.scalar_type());
  if (code < 0 || x.dim() == 0 || !plain(x) || !like(residual, x)) return {};
  const int32_t wcode = weight_code(weight, x);
  const int64_t d = x.size(-1), rows = x.numel() / d;
  if (wcode < 0 || (mx_format >= 0 && d % 32 != 0)) return {};
  const bool mx = mx_format >= 0, fp4 = mx_format == VELOGRAD_MX_E2M1;
  const int64_t y_last = fp4 ? d / 2 : d;
  const auto bytes = x.options().dtype(at::kByte);
  at::Tensor y = at::empty(with_last(x, y_last), bytes);
  at::Tensor scale = mx ? at::empty(with_last(x, d / 32), bytes) : row_stat(x);
  at::Tensor h = residual.has_value() ? at::empty(x.sizes(), x.options()) : x;
  at::Tensor inv = row_stat(x);
  void* hp = residual.has_value() ? h.data_ptr() : nullptr;
  if (mx) {
    check(velograd_rmsnorm_residual_fwd_mx(
              x.data_ptr(), ptr(residual), ptr(weight), y.data_ptr<uint8_t>(),
              scale.data_ptr<uint8_t>(), hp, inv.data_ptr<float>(), rows, d, d, d, y_last, d / 32, d,
              code, wcode, (int32_t)mx_format, (float)eps, stream_of(x)),
          "velograd_rmsnorm_residual_fwd_mx");
    return {y.view(fp4 ? at::kFloat4_e2m1fn_x2 : at::kFloat8_e4m3fn),
            scale.view(at::kFloat8_e8m0fnu), h, inv};
  }
  check(velograd_rmsnorm_residual_fwd_fp8(x.data_ptr(), ptr(residual), ptr(weight),
                                          y.data_ptr<uint8_t>(), scale.data_ptr<float>(), hp,
                                          inv.data_ptr<float>(), rows, d, d, d, d, d, code, wcode,
                                          (float)eps, stream_of(x)),
        "velograd_rmsnorm_residual_fwd_fp8");
  return {y.view(at::kFloat8_e4m3fn), scale, h, inv};
}

// What a backward writes: dx, dweight (undefined without a weight) and its scratch.
struct BwdBuffers {
  at::Tensor dx, dweight, ws;
  int64_t ws_bytes = 0;
  BwdBuffers(const at::Tensor& g, const OptTensor& weight, int64_t rows, int64_t d) {
    dx = at::empty(g.sizes(), g.options());
    if (!weight.has_value()) return;
    dweight = at::empty({d}, g.options().dtype(at::kFloat));
    ws_bytes = (int64_t)velograd_rmsnorm_residual_bwd_workspace_bytes(rows, d, g.get_device());
    ws = at::empty({ws_bytes}, g.options().dtype(at::kByte));
  }
  float* dw() { return dweight.defined() ? dweight.data_ptr<float>() : nullptr; }
  void* scratch() { return ws.defined() ? ws.data_ptr() : nullptr; }
};

// [dx, dweight] of velograd_rmsnorm_residual_bwd.
Tensors backward(const at::Tensor& g, const at::Tensor& saved, const OptTensor& weight,
                 const at::Tensor& inv_rms, bool saved_is_h, const OptTensor& dres,
                 const OptTensor& grad_h) {
  const int32_t code = dtype_code(g.scalar_type());
  if (code < 0 || g.dim() == 0 || !plain(g) || !like(saved, g) || !like(dres, g) ||
      !like(grad_h, g))
    return {};
  const int64_t d = g.size(-1), rows = g.numel() / d;
  const int32_t wcode = weight_code(weight, g);
  if (wcode < 0 || !stat_ok(inv_rms, g, rows)) return {};
  BwdBuffers b(g, weight, rows, d);
  check(velograd_rmsnorm_residual_bwd(
            g.data_ptr(), saved.data_ptr(), saved_is_h ? 1 : 0, ptr(weight),
            inv_rms.data_ptr<float>(), ptr(grad_h), b.dx.data_ptr(),
            dres.has_value() ? dres->data_ptr() : nullptr, b.dw(), b.scratch(),
            (size_t)b.ws_bytes, rows, d, d, d, d, d, d, code, wcode, stream_of(g)),
        "velograd_rmsnorm_residual_bwd");
  return {b.dx, b.dweight};
}

// x rotated (velograd_rope) over its axes as [outer, seq, heads, dim].
at::Tensor rotate(const at::Tensor& x, int64_t outer, int64_t seq, int64_t heads, int64_t dim,
                  int64_t rot_dim, double theta, bool inverse, int32_t pairing) {
  at::Tensor out = at::empty(x.sizes(), x.options());
  check(velograd_rope(x.data_ptr(), out.data_ptr(), outer, seq, heads, dim, rot_dim, (float)theta,
                      inverse ? 1 : 0, pairing, dtype_code(x.scalar_type()), stream_of(x)),
        "velograd_rope");
  return out;
}

// [q_rot, k_rot (undefined without k)] of q and k shaped [..., seq, heads, dim]; head_dim 0: all
// of dim.
Tensors rope(const at::Tensor& q, const OptTensor& k, int64_t head_dim, double theta,
             bool inverse) {
  auto ok = [](const at::Tensor& t) {
    return dtype_code(t.scalar_type()) >= 0 && t.dim() >= 3 && plain(t);
  };
  if (!ok(q)) return {};
  const int64_t rot = head_dim != 0 ? head_dim : q.size(-1), seq = q.size(-3);
  if (rot < 2 || rot % 2 != 0 || q.size(-1) < rot) return {};
  if (k.has_value() && (!ok(*k) || k->device() != q.device() || k->dim() != q.dim() ||
                        k->size(-3) != seq || k->size(-1) < rot))
    return {};
  auto one = [&](const at::Tensor& t) {
    const int64_t heads = t.size(-2), dim = t.size(-1);
    return rotate(t, t.numel() / (seq * heads * dim), seq, heads, dim, rot, theta, inverse,
                  VELOGRAD_ROPE_HALF);
  };
  at::Tensor q_rot = one(q);
  return {q_rot, k.has_value() ? one(*k) : at::Tensor()};
}

// [x_rot] of interleaved pairs over x's last axis, positions along axis -2.
Tensors rope_interleaved(const at::Tensor& x, double base, bool inverse) {
  if (dtype_code(x.scalar_type()) < 0 || x.dim() < 2 || !plain(x) || x.size(-1) % 2 != 0) return {};
  const int64_t seq = x.size(-2), dim = x.size(-1);
  return {rotate(x, x.numel() / (seq * dim), seq, 1, dim, dim, base, inverse,
                 VELOGRAD_ROPE_INTERLEAVED)};
}

// [y, h, inv_rms] of velograd_rmsnorm_rope_fwd.
Tensors norm_rope(const at::Tensor& x, const OptTensor& residual, const OptTensor& weight,
                  double eps, double base, double min_mean_sq) {
  const int32_t code = dtype_code(x.scalar_type());
  if (code < 0 || x.dim() < 2 || !plain(x) || !like(residual, x) || x.size(-1) % 2 != 0) return {};
  const int32_t wcode = weight_code(weight, x);
  if (wcode < 0) return {};
  const int64_t d = x.size(-1), rows = x.numel() / d;
  at::Tensor y = at::empty(x.sizes(), x.options());
  at::Tensor h = residual.has_value() ? at::empty(x.sizes(), x.options()) : x;
  at::Tensor inv = row_stat(x);
  check(velograd_rmsnorm_rope_fwd(x.data_ptr(), ptr(residual), ptr(weight), y.data_ptr(),
                                  residual.has_value() ? h.data_ptr() : nullptr,
                                  inv.data_ptr<float>(), rows, d, d, d, d, d, x.size(-2), code,
                                  wcode, (float)eps, (float)min_mean_sq, (float)base,
                                  stream_of(x)),
        "velograd_rmsnorm_rope_fwd");
  return {y, h, inv};
}

// [dx, dweight] of velograd_rmsnorm_rope_bwd.
Tensors norm_rope_backward(const at::Tensor& g, const at::Tensor& h, const OptTensor& weight,
                           const at::Tensor& inv_rms, double base) {
  const int32_t code = dtype_code(g.scalar_type());
  if (code < 0 || g.dim() < 2 || !plain(g) || !like(h, g) || g.size(-1) % 2 != 0) return {};
  const int64_t d = g.size(-1), rows = g.numel() / d;
  const int32_t wcode = weight_code(weight, g);
  if (wcode < 0 || !stat_ok(inv_rms, g, rows)) return {};
  BwdBuffers b(g, weight, rows, d);
  check(velograd_rmsnorm_rope_bwd(g.data_ptr(), h.data_ptr(), ptr(weight),
                                  inv_rms.data_ptr<float>(), b.dx.data_ptr(), b.dw(), b.scratch(),
                                  (size_t)b.ws_bytes, rows, d, d, d, d, g.size(-2), code, wcode,
                                  (float)base, stream_of(g)),
        "velograd_rmsnorm_rope_bwd");
  return {b.dx, b.dweight};
}

// The interpreter lock given up for a scope (pybind11's own guard looks its internals up as well, a
// tenth of a microsecond a call).
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  Unlocked() = default;
  Unlocked(const Unlocked&) = delete;
  Unlocked& operator=(const Unlocked&) = delete;
  ~Unlocked() { PyEval_RestoreThread(state); }
};

}  // namespace

PYBIND11_MODULE(_fastpath, m) {
  m.doc() = "C++ fast path of the kernels' common calls, for launch-bound sizes";
  // Allocation and launch run without the interpreter lock, as torch's own calls do: either may
  // wait (for memory, for room in the queue), and other Python threads go on meanwhile.
  using NoGil = pybind11::call_guard<Unlocked>;
  m.def("forward", &forward, NoGil(),
        "forward(x, residual, weight, eps, min_mean_sq) -> [y, h, inv_rms]", pybind11::arg("x"),
        pybind11::arg("residual"), pybind11::arg("weight"), pybind11::arg("eps"),
        pybind11::arg("min_mean_sq"));
  m.def("forward_quantised", &forward_quantised, NoGil(), pybind11::arg("x"),
        pybind11::arg("residual"), pybind11::arg("weight"), pybind11::arg("eps"),
        pybind11::arg("mx_format"));
  m.def("backward", &backward, NoGil(), pybind11::arg("grad_out"), pybind11::arg("saved"),
        pybind11::arg("weight"), pybind11::arg("inv_rms"), pybind11::arg("saved_is_h"),
        pybind11::arg("dresidual_out"), pybind11::arg("grad_h"));
  m.def("rope", &rope, NoGil(), pybind11::arg("q"), pybind11::arg("k"),
        pybind11::arg("head_dim"), pybind11::arg("theta"), pybind11::arg("inverse"));
  m.def("rope_interleaved", &rope_interleaved, NoGil(), pybind11::arg("x"),
        pybind11::arg("base"), pybind11::arg("inverse"));
  m.def("norm_rope", &norm_rope, NoGil(), pybind11::arg("x"), pybind11::arg("residual"),
        pybind11::arg("weight"), pybind11::arg("eps"), pybind11::arg("base"),
        pybind11::arg("min_mean_sq"));
  m.def("norm_rope_backward", &norm_rope_backward, NoGil(), pybind11::arg("grad_y"),
        pybind11::arg("h"), pybind11::arg("weight"), pybind11::arg("inv_rms"),
        pybind11::arg("base"));
}
