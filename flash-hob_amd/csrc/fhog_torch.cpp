// The host side of the PyTorch entry points in native code: argument checks, output and workspace allocation and the
// autograd chain around the C ABI of libfhog_hip.so (include/fhog_hip.h). A call that is anything but well formed is declined
// (None, or no tensors), and the Python wrappers then find out what is wrong with it and say so; they also take what needs
// the workspace afterwards (row statistics, single passes).
//
// Why native: on short sequences the GPU finishes before Python has prepared the next launch. Host time per call, the Python
// wrappers -> here (same machine): flash_bwdbwd 56 -> 14 us; attention() differentiated twice 208 -> 154 us, of which some 100 are
// torch's own two calls of autograd.grad. On fresh tensors, where the Python nodes also hand the interpreter lock back and forth
// between the caller's and autograd's threads, that program went from 393 to 149 us on 2 x 256 bf16 rows.
#include <ATen/ATen.h>
#include <ATen/TracerMode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/utils/pybind.h>

#include <cmath>
#include <optional>
#include <tuple>

#include "fhog_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::tensor_list;

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return FHOG_DTYPE_BF16;
    case at::kHalf: return FHOG_DTYPE_FP16;
    case at::kFloat: return FHOG_DTYPE_FP32;
    default: return -1;
  }
}

// (batch, N, d) or (B, H, N, d) as the library sees it: batch = B * H slices sb elements apart, rows sn elements apart
struct Layout {
  int64_t batch = 0, n = 0, d = 0, sb = 0, sn = 0;
  bool direct = false;   // usable where it lies: contiguous rows, 16-byte multiples, slices that do not overlap
  bool rows = false;     // contiguous rows, and (B, H) is one dimension of evenly spaced slices
};

Layout layout_of(const Tensor& t) {
  Layout l;
  const auto s = t.sizes(), st = t.strides();
  const int64_t dim = t.dim();
  if (dim != 3 && dim != 4) return l;
  l.n = s[dim - 2], l.d = s[dim - 1], l.sn = st[dim - 2];
  l.batch = dim == 3 ? s[0] : s[0] * s[1];
  const int64_t vec = 16 / t.element_size();
  l.rows = st[dim - 1] == 1;
  if (dim == 3 || s[1] == 1) l.sb = st[0];
  else l.sb = st[1], l.rows = l.rows && (s[0] == 1 || st[0] == s[1] * st[1]);
  if (l.batch == 1) l.sb = l.n * l.sn;   // never used to address anything
  l.direct = l.rows && l.sn >= l.d && l.sn % vec == 0 && l.sb % vec == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 && (l.batch == 1 || l.sb >= l.n * l.sn);
  return l;
}

// Tensors of one group share shape, type, device, batch stride and row stride; copied into contiguous ones if they do not.
// strict: rows that are contiguous but not 16-byte multiples apart are declined instead (the first-order entry points
// have always left those to their callers).
template <size_t N>
struct Group {
  std::array<Tensor, N> t;
  Layout l;
  // shapes, types and devices have to agree with the first tensor
  bool set(const std::array<const Tensor*, N>& in, bool strict) {
    bool same = true;
    for (size_t i = 0; i < N; i++) {
      if (!in[i]->defined() || !in[i]->is_cuda() || in[i]->scalar_type() != in[0]->scalar_type() || in[i]->device() != in[0]->device())
        return false;
      t[i] = *in[i];
      Layout x = layout_of(t[i]);
      if (strict && !x.direct) {
        if (x.rows) return false;
        t[i] = t[i].contiguous();
        x = layout_of(t[i]);
      }
      if (i == 0) l = x;
      if (x.n != l.n || x.d != l.d || x.batch != l.batch || x.batch == 0) return false;
      same = same && x.direct && x.sb == l.sb && x.sn == l.sn;
    }
    if (!same) {
      for (auto& x : t) x = x.contiguous();
      l = layout_of(t[0]);
      for (auto& x : t)
        if (!layout_of(x).direct) return false;
    }
    return true;
  }
  void* ptr(size_t i) const { return t[i].data_ptr(); }
  Tensor like() const { return at::empty_strided(t[0].sizes(), t[0].strides(), t[0].options()); }
};

// What autograd hands over, packed. contiguous() passes over the stride of a dimension of one (a single query that came back
// through (B, 1, H, d)) and over the address, both of which the kernels look at.
Tensor packed(const Tensor& t) {
  const Tensor c = t.contiguous();
  return layout_of(c).direct ? c : c.clone(at::MemoryFormat::Contiguous);
}

// What a saved-tensor hook gave back may lie anywhere; where it lies as it was saved nothing is copied.
Tensor unpacked(const Tensor& t) { return layout_of(t).direct ? t : packed(t); }
Tensor unpacked_lse(const Tensor& L) {
  return reinterpret_cast<uintptr_t>(L.data_ptr()) % 16 == 0 ? L : L.clone(at::MemoryFormat::Contiguous);
}

Tensor as_lse(const Tensor& L) { return L.scalar_type() == at::kFloat && L.is_contiguous() ? L : L.to(at::kFloat).contiguous(); }
Tensor workspace(int64_t bytes, const Tensor& like) { return at::empty({(bytes + 3) / 4}, like.options().dtype(at::kFloat)); }
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

struct Mask {
  int32_t causal;
  int64_t window;
};

bool mask_applies(const Mask& m, int64_t n_q, int64_t n_k) {
  if (m.causal < FHOG_MASK_NONE || m.causal > FHOG_MASK_BOTTOM_RIGHT || m.window < 0 || m.window > INT32_MAX) return false;
  if (m.causal == FHOG_MASK_NONE) return m.window == 0;
  return m.causal == FHOG_MASK_TOP_LEFT ? n_q == n_k : n_k >= n_q;
}

template <size_t NQ, size_t NK>
bool attn_args(fhog_attn_args& a, const Group<NQ>& q, const Group<NK>& k, double scale, const Mask& m) {
  if (k.l.batch != q.l.batch || k.l.d != q.l.d || k.t[0].scalar_type() != q.t[0].scalar_type() || k.t[0].device() != q.t[0].device() ||
      !mask_applies(m, q.l.n, k.l.n))
    return false;
  a = {};
  a.q = q.ptr(0), a.k = k.ptr(0), a.v = k.ptr(1);
  a.batch = q.l.batch, a.n_q = q.l.n, a.n_k = k.l.n, a.d = q.l.d;
  a.stride_qb = q.l.sb, a.stride_qn = q.l.sn, a.stride_kb = k.l.sb, a.stride_kn = k.l.sn;
  a.scale = (float)scale, a.dtype = dtype_code(q.t[0].scalar_type()), a.causal = m.causal, a.window = (int32_t)m.window;
  return a.dtype >= 0;
}

using Forward = std::optional<std::tuple<Tensor, Tensor>>;
Forward forward(const Tensor& q_, const Tensor& k_, const Tensor& v_, double scale, const Mask& m) {
  Group<1> q;
  Group<2> k;
  fhog_attn_args a;
  if (!q.set({&q_}, true) || !k.set({&k_, &v_}, true) || !attn_args(a, q, k, scale, m)) return std::nullopt;
  const c10::DeviceGuard guard(q_.device());
  Tensor o = q.like();
  Tensor lse = at::empty(q_.sizes().slice(0, q_.dim() - 1), q_.options().dtype(at::kFloat));
  a.o = o.data_ptr(), a.lse = (float*)lse.data_ptr();
  if (fhog_attn_validate(&a, 0) != FHOG_OK) return std::nullopt;
  TORCH_CHECK(fhog_attn_fwd(&a, stream_of(q_)) == FHOG_OK, "fhog_attn_fwd: ", fhog_last_error());
  return std::make_tuple(o, lse);
}

using Backward = std::optional<std::tuple<Tensor, Tensor, Tensor>>;
Backward backward(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& o_, const Tensor& do_, const Tensor& L, double scale,
                  const Mask& m, bool strict) {
  Group<3> q;
  Group<2> k;
  fhog_attn_args a;
  if (!q.set({&q_, &o_, &do_}, strict) || !k.set({&k_, &v_}, strict) || !attn_args(a, q, k, scale, m)) return std::nullopt;
  if (!L.is_cuda() || L.device() != q_.device() || L.numel() != a.batch * a.n_q) return std::nullopt;
  const c10::DeviceGuard guard(q_.device());
  const Tensor lse = as_lse(L), ws = workspace(a.batch * a.n_q * 4, q_);
  Tensor dq = q.like(), dk = k.like(), dv = k.like();
  a.o = q.ptr(1), a.dO = q.ptr(2), a.lse = (float*)lse.data_ptr(), a.ws = (float*)ws.data_ptr();
  a.dq = dq.data_ptr(), a.dk = dk.data_ptr(), a.dv = dv.data_ptr();
  if (fhog_attn_validate(&a, 1) != FHOG_OK) return std::nullopt;
  TORCH_CHECK(fhog_attn_bwd(&a, stream_of(q_)) == FHOG_OK, "fhog_attn_bwd: ", fhog_last_error());
  return std::make_tuple(dq, dk, dv);
}

using DoubleBackward = std::optional<std::tuple<Tensor, Tensor, Tensor, Tensor>>;
DoubleBackward double_backward(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& o_, const Tensor& do_, const Tensor& ddq_,
                               const Tensor& ddk_, const Tensor& ddv_, const Tensor& L, double scale, const Mask& m, int impl, int schedule,
                               bool split) {
  Group<4> q, k;
  if (!q.set({&q_, &o_, &do_, &ddq_}, false) || !k.set({&k_, &v_, &ddk_, &ddv_}, false)) return std::nullopt;
  if (k.l.batch != q.l.batch || k.l.d != q.l.d || k_.scalar_type() != q_.scalar_type() || k_.device() != q_.device() ||
      !mask_applies(m, q.l.n, k.l.n) || !L.is_cuda() || L.device() != q_.device() || L.numel() != q.l.batch * q.l.n)
    return std::nullopt;
  fhog_bwdbwd_args a = {};
  a.dtype = dtype_code(q_.scalar_type());
  if (a.dtype < 0) return std::nullopt;
  const c10::DeviceGuard guard(q_.device());
  const Tensor lse = as_lse(L);
  Tensor dq2 = q.like(), ddo = q.like(), dk2 = k.like(), dv2 = k.like();
  a.q = q.ptr(0), a.o = q.ptr(1), a.dO = q.ptr(2), a.ddq = q.ptr(3);
  a.k = k.ptr(0), a.v = k.ptr(1), a.ddk = k.ptr(2), a.ddv = k.ptr(3);
  a.lse = (const float*)lse.data_ptr();
  a.dq2 = dq2.data_ptr(), a.dk2 = dk2.data_ptr(), a.dv2 = dv2.data_ptr(), a.ddo = ddo.data_ptr();
  a.batch = q.l.batch, a.n_q = q.l.n, a.n_k = k.l.n, a.d = q.l.d;
  a.stride_qb = q.l.sb, a.stride_qn = q.l.sn, a.stride_kb = k.l.sb, a.stride_kn = k.l.sn;
  a.scale = (float)scale, a.causal = m.causal, a.window = m.window, a.impl = impl, a.schedule = schedule;
  a.ws = (float*)q.ptr(0);   // any valid pointer: the hint is computed on the host
  const size_t hint = fhog_bwdbwd_workspace_hint(&a);
  if (hint == 0) return std::nullopt;   // not valid
  const int64_t bytes = split ? (int64_t)hint : 3 * a.batch * a.n_q * 4;
  const Tensor ws = workspace(bytes, q_);
  a.ws = (float*)ws.data_ptr(), a.ws_bytes = bytes;
  TORCH_CHECK(fhog_bwdbwd(&a, stream_of(q_)) == FHOG_OK, "fhog_bwdbwd: ", fhog_last_error());
  return std::make_tuple(dq2, dk2, dv2, ddo);
}

// ---- autograd: attention -> first backward -> double-backward (the chain of the Python classes in attention.py) ------
double scale_of(const Tensor& q) { return 1.0 / std::sqrt((double)q.size(-1)); }

struct FirstBackward : torch::autograd::Function<FirstBackward> {
  static tensor_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& grad,
                             const Tensor& L, int64_t causal, int64_t window, int64_t schedule) {
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({q, k, v, o, grad, L});
    ctx->saved_data["arg"] = std::vector<int64_t>{causal, window, schedule};
    const auto r = backward_(q, k, v, o, grad, L, causal, window);
    return {std::get<0>(r), std::get<1>(r), std::get<2>(r)};
  }
  static std::tuple<Tensor, Tensor, Tensor> backward_(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& grad,
                                                      const Tensor& L, int64_t causal, int64_t window) {
    const auto r = ::backward(unpacked(q), unpacked(k), unpacked(v), unpacked(o), grad, unpacked_lse(L), scale_of(q), Mask{(int32_t)causal, window}, false);
    TORCH_CHECK(r, "fhog: first-order backward: ", fhog_last_error());
    return *r;
  }
  static tensor_list backward(AutogradContext* ctx, tensor_list g) {
    tensor_list out(9);
    if (!g[0].defined() && !g[1].defined() && !g[2].defined()) return out;
    const auto s = ctx->get_saved_variables();
    const auto arg = ctx->saved_data["arg"].toIntVector();
    const bool differentiable = at::GradMode::is_enabled() && ((g[0].defined() && g[0].requires_grad()) || (g[1].defined() && g[1].requires_grad()) ||
                                                               (g[2].defined() && g[2].requires_grad()));
    {
      const at::NoGradGuard no_grad;
      const auto dir = [&](size_t i) { return g[i].defined() ? packed(g[i]) : at::zeros_like(s[i]); };
      const auto r = double_backward(unpacked(s[0]), unpacked(s[1]), unpacked(s[2]), unpacked(s[3]), unpacked(s[4]), dir(0), dir(1), dir(2),
                                     unpacked_lse(s[5]), scale_of(s[0]), Mask{(int32_t)arg[0], arg[1]}, FHOG_IMPL_AUTO, (int)arg[2], true);
      TORCH_CHECK(r, "fhog: double-backward: ", fhog_last_error());
      // O and L are caches of (q, k, v): the four results are already total derivatives
      out[0] = std::get<0>(*r), out[1] = std::get<1>(*r), out[2] = std::get<2>(*r), out[4] = std::get<3>(*r);
    }
    if (differentiable) {   // third derivatives do not exist: say so when they are asked for
      tensor_list v = {out[0].detach().requires_grad_(), out[1].detach().requires_grad_(), out[2].detach().requires_grad_(), out[4].detach().requires_grad_()};
      const auto err = std::make_shared<torch::autograd::DelayedError>("trying to differentiate twice the double-backward of fhog.attention", 4);
      v = err->apply(std::move(v));
      out[0] = v[0], out[1] = v[1], out[2] = v[2], out[4] = v[3];
    }
    return out;
  }
};

struct Attention : torch::autograd::Function<Attention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, int64_t causal, int64_t window, int64_t schedule) {
    // The graph of the first backward reaches this node a second time through the saved O, whose gradient FirstBackward
    // does not have: without work to do, and not to be filled in with zeros
    ctx->set_materialize_grads(false);
    const auto r = ::forward(q, k, v, scale_of(q), Mask{(int32_t)causal, window});
    TORCH_CHECK(r, "fhog: forward: ", fhog_last_error());
    ctx->save_for_backward({q, k, v, std::get<0>(*r), std::get<1>(*r)});
    ctx->saved_data["arg"] = std::vector<int64_t>{causal, window, schedule};
    return std::get<0>(*r);
  }
  static tensor_list backward(AutogradContext* ctx, tensor_list g) {
    tensor_list out(6);
    if (!g[0].defined()) return out;
    const auto s = ctx->get_saved_variables();
    const auto arg = ctx->saved_data["arg"].toIntVector();
    const auto r = FirstBackward::apply(s[0], s[1], s[2], s[3], packed(g[0]), s[4], arg[0], arg[1], arg[2]);
    out[0] = r[0], out[1] = r[1], out[2] = r[2];
    return out;
  }
};

// What attention() takes here: what ::forward takes, checked before a node of the graph exists
std::optional<Tensor> attention(const Tensor& q, const Tensor& k, const Tensor& v, int64_t causal, int64_t window, int64_t schedule) {
  // torch.jit.trace records a Python node as a call of it; of a native one it would record the allocations and miss the launches
  if (at::tracer::impl::is_dispatch_enabled()) return std::nullopt;
  // torch.func transforms: the Python nodes say that they have no rule for them
  if (c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode)) return std::nullopt;
  for (const Tensor* t : {&q, &k, &v}) {
    const int64_t dim = t->dim();
    // tensors that dispatch to Python (fake ones among them) have no memory to launch on
    if (t->unsafeGetTensorImpl()->is_python_dispatch()) return std::nullopt;
    if (!t->is_cuda() || t->device() != q.device() || t->scalar_type() != q.scalar_type() || (dim != 3 && dim != 4) || dim != q.dim()) return std::nullopt;
    for (int64_t i = 0; i < dim; i++)
      if (i != dim - 2 && t->size(i) != q.size(i)) return std::nullopt;
    const Layout l = layout_of(*t);
    if (l.rows && !l.direct) return std::nullopt;
  }
  const int64_t d = q.size(-1), n_q = q.size(-2), n_k = k.size(-2);
  if (dtype_code(q.scalar_type()) < 0 || (d != 32 && d != 64 && d != 128) || v.size(-2) != n_k || q.numel() == 0 || k.numel() == 0 ||
      q.numel() / d >= INT32_MAX || q.numel() / d / n_q > 65535 || n_q > (1 << 24) || n_k > (1 << 24) ||
      !mask_applies(Mask{(int32_t)causal, window}, n_q, n_k) || schedule < FHOG_SCHEDULE_FOUR_PASS || schedule > FHOG_SCHEDULE_THREE_SWEEP)
    return std::nullopt;
  return Attention::apply(q, k, v, causal, window, schedule);
}

}  // namespace

PYBIND11_MODULE(_fhog_torch, m) {
  namespace py = pybind11;
  const auto free_lock = py::call_guard<py::gil_scoped_release>();
  m.def("forward", [](const Tensor& q, const Tensor& k, const Tensor& v, double scale, int causal, int64_t window) {
    const at::NoGradGuard no_grad;
    return forward(q, k, v, scale, Mask{causal, window});
  }, free_lock);
  m.def("backward", [](const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& g, const Tensor& L, double scale, int causal,
                       int64_t window) {
    const at::NoGradGuard no_grad;
    return backward(q, k, v, o, g, L, scale, Mask{causal, window}, true);
  }, free_lock);
  m.def("double_backward", [](const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& g, const Tensor& ddq, const Tensor& ddk,
                              const Tensor& ddv, const Tensor& L, double scale, int causal, int64_t window, int impl, int schedule, bool split) {
    const at::NoGradGuard no_grad;
    return double_backward(q, k, v, o, g, ddq, ddk, ddv, L, scale, Mask{causal, window}, impl, schedule, split);
  }, free_lock);
  m.def("attention", &attention, free_lock);
}
