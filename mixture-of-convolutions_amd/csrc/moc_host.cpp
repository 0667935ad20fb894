// Host side of the MoC calls that a program makes per step: the layer and the
// functional op as autograd nodes, the forward with a state, and the decode
// step, each one call from Python.  What they launch and return is what the
// Python functions of moc/api.py and moc/ops.py do (which stay for every call
// that one of these hands back as not its own: other dtypes and shapes, tensor
// subclasses, tracing, function transforms, forward-mode differentiation).
//
// Why: a step of a small layer spent most of its time in the interpreter: checks,
// argument conversion and allocations in Python, and a backward that waits for
// the interpreter lock on autograd's own thread.  Us a call, Python functions ->
// here: training step B 3 T 1021 D 1130 138 to 165 (by box) -> 92 (53 of it
// kernels), fp32 B 2 T 512 D 256 170 -> 95; 777-token prefill 31 -> 17.6; decode step
// 10.5 -> 7.6, fp32 25.6 -> 11.4.
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/extension.h>

#include "../../include/moc_hip.h"

namespace {

using at::Tensor;
using c10::DispatchKey;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

int dtype_code(at::ScalarType t) { return t == at::kFloat ? 0 : (t == at::kBFloat16 ? 1 : -1); }

// A dense GPU tensor of its own: no wrapper or transform of one, no dual number.
bool plain(const Tensor& t) {
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.is_neg() || t.is_conj()) return false;
  static const c10::DispatchKeySet wrapped({DispatchKey::Python, DispatchKey::PythonTLSSnapshot,
                                            DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper,
                                            DispatchKey::Batched, DispatchKey::Functionalize});
  return !t.key_set().has_any(wrapped) && t.has_storage() && !t._fw_grad(0).defined();
}

// No tracer, dispatch mode or function transform is watching this thread.
bool unwatched() {
  using c10::impl::tls_is_dispatch_key_included;
  return !tls_is_dispatch_key_included(DispatchKey::Python) &&
         !tls_is_dispatch_key_included(DispatchKey::Tracer) &&
         !tls_is_dispatch_key_included(DispatchKey::Functionalize) &&
         !tls_is_dispatch_key_included(DispatchKey::FuncTorchDynamicLayerFrontMode);
}

bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t != nullptr && t->requires_grad()) return true;
  return false;
}

void check(int rc, const char* what) {
  if (rc != 0) TORCH_CHECK(false, what, " failed (status ", rc, "): ", moc_last_error());
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor bytes(size_t n, const Tensor& like) {
  return at::empty({static_cast<int64_t>(n > 0 ? n : 1)}, like.options().dtype(at::kByte));
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// A layer call's sizes and codes.  Fixed-length x [B, T, D] or packed x [N, D]
// with cu.
struct Call {
  int act, route;  // route: 1 softmax, 2 exp (layer); 0 weights given (func)
  int dt;
  int64_t N, T, D, K, S, Z;
  Tensor cu;       // undefined: fixed length
  const void* cu_ptr() const { return ptr(cu); }
  int cu64() const { return cu.defined() && cu.scalar_type() == at::kLong; }
  int64_t n_seqs() const { return cu.defined() ? cu.numel() - 1 : 0; }
  int64_t seq_len() const { return cu.defined() ? 0 : T; }
};

// Fills the sizes that x, the basis and the packed offsets give; false where
// the call is not one of these (the Python path then names what is wrong).
bool sizes(Call& c, const Tensor& x, const Tensor& basis, const OptTensor& cu) {
  c.dt = dtype_code(x.scalar_type());
  if (c.dt < 0 || basis.scalar_type() != x.scalar_type() || basis.dim() != 3) return false;
  c.K = basis.size(0), c.S = basis.size(1), c.D = basis.size(2);
  if (x.dim() != (cu.has_value() ? 2 : 3) || x.size(-1) != c.D) return false;
  if (x.numel() == 0 || basis.numel() == 0) return false;
  c.N = x.numel() / c.D;
  c.T = cu.has_value() ? 0 : x.size(1);
  if (cu.has_value()) {
    if (!plain(*cu) || cu->device() != x.device() || cu->dim() != 1 || cu->numel() < 2) return false;
    if (cu->scalar_type() != at::kInt && cu->scalar_type() != at::kLong) return false;
    c.cu = cu->contiguous();
  }
  return basis.device() == x.device();
}

// The router's sizes; whether its kernels take them (as ops.router_supported and
// ops.router_f32_supported say).
bool router_ok(Call& c, const Tensor& x, const Tensor& z, const Tensor& router) {
  if (z.scalar_type() != x.scalar_type() || router.scalar_type() != x.scalar_type()) return false;
  if (z.device() != x.device() || router.device() != x.device()) return false;
  if (router.dim() != 2 || router.size(0) != c.K || z.dim() != x.dim()) return false;
  c.Z = router.size(1);
  if (z.size(-1) != c.Z || z.numel() == 0) return false;
  for (int64_t i = 0; i + 1 < z.dim(); ++i)
    if (z.size(i) != x.size(i)) return false;
  if (c.K > 32) return false;
  if (c.dt == 1) return moc_router_supported(c.N, c.Z, c.K, 1) != 0;
  return !at::autocast::is_autocast_enabled(at::kCUDA) && moc_router_f32_supported(c.N, c.Z, c.K) != 0;
}

// softmax / exp (or the logits: route 0) of z . router^T
Tensor run_router(const Call& c, const Tensor& z, const Tensor& router, int route) {
  auto shape = z.sizes().vec();
  shape.back() = c.K;
  Tensor out = at::empty(shape, z.options());
  if (c.dt == 0)
    check(moc_router_f32_forward(ptr(z), ptr(router), ptr(out), c.N, c.Z, c.K, route, stream_of(z)),
          "moc_router_f32_forward");
  else if (route == 0)
    check(moc_router_forward(ptr(z), ptr(router), ptr(out), c.N, c.Z, c.K, 1, stream_of(z)),
          "moc_router_forward");
  else
    check(moc_router_forward_routed(ptr(z), ptr(router), ptr(out), c.N, c.Z, c.K, 1, route, stream_of(z)),
          "moc_router_forward");
  return out;
}

// moc_forward on weights of the given routing code
Tensor run_forward(const Call& c, const Tensor& x, const Tensor& a, const Tensor& basis, int routing) {
  Tensor y = at::empty_like(x);
  Tensor ws = bytes(moc_forward_workspace_bytes(c.N, c.D, c.K, c.S, c.dt, routing), x);
  check(moc_forward(ptr(x), ptr(a), ptr(basis), ptr(y), c.cu_ptr(), c.cu64(), c.n_seqs(), c.N, c.seq_len(),
                    c.D, c.K, c.S, c.dt, c.dt, c.dt, c.act, routing, ptr(ws), ws.numel(), stream_of(x)),
        "moc_forward");
  return y;
}

// dy as the kernels take it (ops.dy_operand): rows D apart, one broadcast row (0)
// or one broadcast element (-1)
Tensor dy_operand(const Tensor& dy, at::ScalarType dt, int64_t& stride) {
  const auto st = dy.strides();
  const int64_t D = dy.size(-1);
  bool lead0 = true;
  for (size_t i = 0; i + 1 < st.size(); ++i) lead0 = lead0 && st[i] == 0;
  if (dy.numel() > 1 && lead0 && st.back() == 0) {
    stride = -1;
    return dy.as_strided({1}, {1}, dy.storage_offset()).to(dt);
  }
  if (dy.dim() >= 2 && dy.numel() > D && lead0) {
    stride = 0;
    return dy.as_strided({D}, {st.back()}, dy.storage_offset()).to(dt).contiguous();
  }
  stride = D;
  return dy.contiguous().to(dt);
}

struct Grads {
  Tensor dx, da, db;
};
Grads run_backward(const Call& c, const Tensor& x, const Tensor& a, const Tensor& basis, const Tensor& dy,
                   bool need_x, int routing) {
  int64_t stride;
  const Tensor dyo = dy_operand(dy, x.scalar_type(), stride);
  Grads g{need_x ? at::empty_like(x) : Tensor(), at::empty_like(a), at::empty_like(basis)};
  Tensor ws = bytes(moc_backward_workspace_bytes(c.N, c.D, c.K, c.S, c.dt, routing), x);
  check(moc_backward(ptr(x), ptr(a), ptr(basis), ptr(dyo), stride, ptr(g.dx), ptr(g.da), ptr(g.db), c.cu_ptr(),
                     c.cu64(), c.n_seqs(), c.N, c.seq_len(), c.D, c.K, c.S, c.dt, c.dt, c.dt, c.act, routing,
                     ptr(ws), ws.numel(), stream_of(x)),
        "moc_backward");
  return g;
}

// The nodes are differentiable once: with a graph asked for, their results
// raise when they are differentiated again.
variable_list once(variable_list out, const variable_list& grads) {
  bool any = false;
  for (const auto& g : grads) any = any || (g.defined() && g.requires_grad());
  if (!any) return out;
  variable_list defined;
  for (auto& t : out)
    if (t.defined()) defined.push_back(t.detach().set_requires_grad(true));
  auto err = std::make_shared<torch::autograd::DelayedError>(
      "trying to differentiate twice a function that was marked with @once_differentiable",
      static_cast<int64_t>(defined.size()));
  variable_list wrapped = (*err)(std::move(defined));
  size_t i = 0;
  for (auto& t : out)
    if (t.defined()) t = wrapped[i++];
  return out;
}

void keep(AutogradContext* ctx, const Call& c) {
  ctx->saved_data["c"] = std::vector<int64_t>{c.act, c.route, c.dt, c.N, c.T, c.D, c.K, c.S, c.Z};
}
Call kept(AutogradContext* ctx, const Tensor& cu) {
  const auto v = ctx->saved_data["c"].toIntVector();
  return Call{static_cast<int>(v[0]), static_cast<int>(v[1]), static_cast<int>(v[2]), v[3], v[4], v[5], v[6],
              v[7], v[8], cu};
}

// MoC.forward as one node (api._MoCLayerFunction)
struct LayerFn : public torch::autograd::Function<LayerFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x0, const Tensor& z0, const Tensor& r0,
                        const Tensor& b0, const Call* c) {
    const Tensor x = x0.contiguous(), z = z0.contiguous(), r = r0.contiguous(), b = b0.contiguous();
    const Tensor w = run_router(*c, z, r, c->route);
    Tensor y = run_forward(*c, x, w, b, c->route + 2);
    ctx->save_for_backward({x, w, b, z0, r0, c->cu});
    keep(ctx, *c);
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &w = saved[1], &b = saved[2];
    const Call c = kept(ctx, saved[5]);
    const bool need[3] = {ctx->needs_input_grad(0), ctx->needs_input_grad(1), ctx->needs_input_grad(2)};
    variable_list out(5);
    {
      at::NoGradGuard ng;
      const c10::DeviceGuard dg(x.device());
      const Grads g = run_backward(c, x, w, b, grads[0], need[0], c.route + 2);
      out[0] = g.dx;
      out[3] = g.db;
      if (need[1] || need[2]) {
        const Tensor z = saved[3].contiguous(), r = saved[4].contiguous();
        if (need[1]) out[1] = at::empty_like(z);
        if (need[2]) out[2] = at::empty_like(r);
        const bool f32 = c.dt == 0;
        const size_t n = !need[2] ? 0
                         : f32    ? moc_router_f32_backward_workspace_bytes(c.N, c.Z, c.K)
                                  : moc_router_backward_workspace_bytes(c.N, c.Z, c.K, 1);
        Tensor ws = n > 0 ? bytes(n, x) : Tensor();
        check(f32 ? moc_router_f32_backward(ptr(z), ptr(r), ptr(g.da), ptr(out[1]), ptr(out[2]), c.N, c.Z, c.K,
                                            ptr(ws), n, stream_of(x))
                  : moc_router_backward(ptr(z), ptr(r), ptr(g.da), ptr(out[1]), ptr(out[2]), c.N, c.Z, c.K, 1,
                                        ptr(ws), n, stream_of(x)),
              "moc_router_backward");
      }
    }
    return at::GradMode::is_enabled() ? once(std::move(out), grads) : out;
  }
};

// moc_triton on routing weights as one node (api._MoCFunction)
struct FuncFn : public torch::autograd::Function<FuncFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x0, const Tensor& a0, const Tensor& b0,
                        const Call* c) {
    const Tensor x = x0.contiguous(), a = a0.contiguous(), b = b0.contiguous();
    Tensor y = run_forward(*c, x, a, b, 0);
    ctx->save_for_backward({x, a, b, c->cu});
    keep(ctx, *c);
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Call c = kept(ctx, saved[3]);
    variable_list out(4);
    const bool need_x = ctx->needs_input_grad(0);
    {
      at::NoGradGuard ng;
      const c10::DeviceGuard dg(saved[0].device());
      const Grads g = run_backward(c, saved[0], saved[1], saved[2], grads[0], need_x, 0);
      out[0] = g.dx;
      out[1] = g.da;
      out[2] = g.db;
    }
    return at::GradMode::is_enabled() ? once(std::move(out), grads) : out;
  }
};

// y of MoC.forward without a cache, or nothing: not a call of this path
OptTensor layer(const Tensor& x, const Tensor& z, const Tensor& router, const Tensor& basis, int act, int route,
                const OptTensor& cu) {
  if (!unwatched() || !plain(x) || !plain(z) || !plain(router) || !plain(basis)) return std::nullopt;
  Call c{act, route};
  const c10::DeviceGuard dg(x.device());
  if (!sizes(c, x, basis, cu) || !router_ok(c, x, z, router)) return std::nullopt;
  if (wants_grad({&x, &z, &router, &basis})) return LayerFn::apply(x, z, router, basis, &c);
  at::NoGradGuard ng;
  return run_forward(c, x.contiguous(), run_router(c, z.contiguous(), router.contiguous(), route),
                     basis.contiguous(), route + 2);
}

// y of moc_triton without a cache, or nothing
OptTensor func(const Tensor& x, const Tensor& alpha, const Tensor& basis, int act, const OptTensor& cu) {
  if (!unwatched() || !plain(x) || !plain(alpha) || !plain(basis)) return std::nullopt;
  Call c{act, 0};
  const c10::DeviceGuard dg(x.device());
  if (!sizes(c, x, basis, cu) || alpha.scalar_type() != x.scalar_type() || alpha.device() != x.device() ||
      alpha.dim() != x.dim() || alpha.size(-1) != c.K || alpha.numel() != c.N * c.K)
    return std::nullopt;
  for (int64_t i = 0; i + 1 < x.dim(); ++i)
    if (alpha.size(i) != x.size(i)) return std::nullopt;
  if (wants_grad({&x, &alpha, &basis})) return FuncFn::apply(x, alpha, basis, &c);
  at::NoGradGuard ng;
  return run_forward(c, x.contiguous(), alpha.contiguous(), basis.contiguous(), 0);
}

// Whether a prompt's state is cheaper written by the forward launch than as a copy of
// its last rows after the plain forward.  It saves a launch and a slow transposed copy
// (bf16, 8 x 1024 tokens, D 2048, 16 routes, 4 taps: 27 -> 22 us), but the kernel with
// a cache to read walks a sequence's first S - 1 rows one tap at a time (8 taps, 8 x 3
// tokens: 6.3 us plain, 18.9), and in fp32 its larger tile costs more than the copy
// from about 2^22 elements on with more than 3 taps or 16 routes (8 x 2048 tokens, D
// 4096, 4 taps, 16 routes 126 -> 141; 6 taps, 32 routes 256 -> 309; 3 x 300 tokens, D
// 1544, 4 taps 12 -> 10).
bool state_in_forward(const Call& c) {
  if (c.T < c.S - 1) return false;
  return c.dt == 1 || c.N * c.D <= (int64_t(1) << 22) || (c.S <= 3 && c.K <= 16);
}

// (y, state or None) of MoC.forward with a cache or a final state, fixed length:
// one token per sequence and a cache: the decode step, in place on the cache
// (not differentiable); else without gradients only.  Nothing: not a call of
// this path
std::optional<std::tuple<Tensor, OptTensor>> stateful(const Tensor& x, const Tensor& z, const Tensor& router,
                                                      const Tensor& basis, const OptTensor& cache, int act,
                                                      int route, bool want) {
  if (!unwatched() || !plain(x) || !plain(z) || !plain(router) || !plain(basis)) return std::nullopt;
  Call c{act, route};
  const c10::DeviceGuard dg(x.device());
  if (!sizes(c, x, basis, std::nullopt) || z.dim() != 3) return std::nullopt;
  const int64_t B = x.size(0);
  if (cache.has_value()) {
    if (!plain(*cache) || cache->device() != x.device() || cache->scalar_type() != x.scalar_type() ||
        cache->dim() != 3 || cache->size(0) != B || cache->size(1) != c.D || cache->size(2) != c.S)
      return std::nullopt;
  }
  if (!router_ok(c, x, z, router)) return std::nullopt;
  if (cache.has_value() && c.T == 1) {
    const bool one = c.dt == 1 && cache->is_contiguous() && moc_decode_step_supported(B, c.Z, c.D, c.K, c.S);
    if (!one && c.dt == 1) return std::nullopt;
    at::NoGradGuard ng;
    const Tensor xc = x.contiguous(), zc = z.contiguous(), rc = router.contiguous(), bc = basis.contiguous();
    Tensor y = at::empty_like(xc);
    if (one) {
      check(moc_decode_step(ptr(zc), ptr(rc), ptr(xc), ptr(bc), ptr(*cache), ptr(y), B, c.Z, c.D, c.K, c.S, act,
                            route, stream_of(x)),
            "moc_decode_step");
    } else {
      const Tensor lg = run_router(c, zc, rc, 0);
      check(moc_update(ptr(xc), ptr(lg), ptr(bc), ptr(*cache), cache->stride(0), cache->stride(1),
                       cache->stride(2), ptr(y), B, c.D, c.K, c.S, c.dt, c.dt, c.dt, act, route, stream_of(x)),
            "moc_update");
    }
    return std::make_tuple(y, want ? cache : OptTensor());
  }
  if (wants_grad({&x, &z, &router, &basis, cache.has_value() ? &*cache : nullptr})) return std::nullopt;
  if (!moc_prefill_supported(B, c.T, c.D, c.K, c.S, c.dt, cache.has_value())) return std::nullopt;
  if (!cache.has_value() && !state_in_forward(c)) return std::nullopt;
  at::NoGradGuard ng;
  const Tensor xc = x.contiguous(), bc = basis.contiguous();
  const Tensor w = run_router(c, z.contiguous(), router.contiguous(), route);
  const Tensor hist = cache.has_value() ? cache->contiguous() : Tensor();
  Tensor y = at::empty_like(xc), fin;
  if (want) fin = at::empty({B, c.D, c.S}, x.options());
  Tensor ws = bytes(moc_forward_workspace_bytes(c.N, c.D, c.K, c.S, c.dt, route + 2), x);
  check(moc_forward_prefill(ptr(xc), ptr(w), ptr(bc), ptr(y), ptr(hist), ptr(fin), B, c.T, c.D, c.K, c.S, c.dt,
                            c.dt, c.dt, act, route + 2, ptr(ws), ws.numel(), stream_of(x)),
        "moc_forward_prefill");
  return std::make_tuple(y, want ? OptTensor(fin) : OptTensor());
}

// the nodes' Python type, under the name of the Python function they stand for
template <typename F>
void name_node(const char* name) {
  static PyTypeObject type{};
  torch::autograd::_initFunctionPyTypeObject(type, name, nullptr, nullptr);
  torch::autograd::registerCppFunction(typeid(torch::autograd::CppNode<F>), &type);
}

// A call's tensor arguments as Python hands them over.  Only torch.Tensor and
// torch.nn.Parameter themselves are taken: a subclass, with or without a dispatch
// key of its own, keeps its result type and its __torch_function__ in the Python
// functions, and what is no tensor its error there.  The calls then run without the
// interpreter lock: an allocation may wait for the device and a launch for space in
// the queue, and other threads' work goes on meanwhile (saved-tensor hooks take the
// lock themselves).
struct Args {
  bool own = true;
  Tensor operator()(py::handle h) {
    own = own && THPVariable_CheckExact(h.ptr());
    return own ? THPVariable_Unpack(h.ptr()) : Tensor();
  }
  OptTensor opt(py::handle h) { return h.is_none() ? OptTensor() : OptTensor((*this)(h)); }
};

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  name_node<LayerFn>("_MoCLayerFunctionBackward");
  name_node<FuncFn>("_MoCFunctionBackward");
  m.def("layer", [](py::handle x, py::handle z, py::handle router, py::handle basis, int act, int route,
                    py::handle cu) -> OptTensor {
    Args a;
    const Tensor tx = a(x), tz = a(z), tr = a(router), tb = a(basis);
    const OptTensor tc = a.opt(cu);
    if (!a.own) return std::nullopt;
    const py::gil_scoped_release unlocked;
    return layer(tx, tz, tr, tb, act, route, tc);
  });
  m.def("func", [](py::handle x, py::handle alpha, py::handle basis, int act, py::handle cu) -> OptTensor {
    Args a;
    const Tensor tx = a(x), ta = a(alpha), tb = a(basis);
    const OptTensor tc = a.opt(cu);
    if (!a.own) return std::nullopt;
    const py::gil_scoped_release unlocked;
    return func(tx, ta, tb, act, tc);
  });
  m.def("stateful", [](py::handle x, py::handle z, py::handle router, py::handle basis, py::handle cache, int act,
                       int route, bool want) -> std::optional<std::tuple<Tensor, OptTensor>> {
    Args a;
    const Tensor tx = a(x), tz = a(z), tr = a(router), tb = a(basis);
    const OptTensor tc = a.opt(cache);
    if (!a.own) return std::nullopt;
    const py::gil_scoped_release unlocked;
    return stateful(tx, tz, tr, tb, tc, act, route, want);
  });
}
