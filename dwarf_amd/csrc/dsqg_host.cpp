// Native host layer of the eager public functions (dwarf_amd/api.py): argument checks, the C ABI's
// argument blocks, output and workspace allocation and autograd, in C++.
//
// The kernels of a training step take a few tens to two hundred microseconds; the same steps
// through Python objects (ctypes blocks, a Python autograd function whose backward runs on the
// engine's thread) took 220-350 us of host time per forward + backward on the MI355X host, and
// bounded every call but the largest.  Traced code (torch.compile, export, fake tensors) sees the
// custom ops of dwarf_amd/ops.py instead.
//
// The entry points of libdsqg_hip.so arrive as addresses from the loader (dwarf_amd/_lib.py), so
// the library that was checked there is the one called here.  Nothing is kept between calls.
#include <ATen/autocast_mode.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <array>
#include <optional>

#include "../../include/dsqg.h"

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

struct Api {
  decltype(&dsqg_status_string) status_string = nullptr;
  decltype(&dsqg_fwd) fwd = nullptr;
  decltype(&dsqg_bwd_workspace_size) bwd_workspace_size = nullptr;
  decltype(&dsqg_bwd) bwd = nullptr;
  decltype(&dsqg_decode_step) decode_step = nullptr;
  decltype(&dsqg_kv_inject) kv_inject = nullptr;
  decltype(&dsqg_ring_load) ring_load = nullptr;
  decltype(&dsqg_pool_gate_workspace_size) pool_workspace_size = nullptr;
  decltype(&dsqg_pool_gate_fwd) pool_fwd = nullptr;
  decltype(&dsqg_pool_gate_bwd) pool_bwd = nullptr;
  decltype(&dsqg_linear_wgrad_workspace_size) linear_workspace_size = nullptr;
  decltype(&dsqg_linear_wgrad) linear_wgrad = nullptr;
  PyObject* library_error = nullptr;  // dwarf_amd._lib.DSQGLibraryError
} api;

// ---- Errors (Python exceptions; the backward runs without the GIL). --------------------------

[[noreturn]] void raise(PyObject* type, const std::string& msg) {
  py::gil_scoped_acquire gil;
  PyErr_SetString(type, msg.c_str());
  throw py::error_already_set();
}

template <typename... A>
void require(bool ok, const A&... msg) {
  if (!ok) raise(PyExc_AssertionError, c10::str(msg...));
}

void check(int status, const char* what) {
  if (status != DSQG_OK)
    raise(api.library_error, c10::str(what, " failed: status ", status, " (", api.status_string(status), ")"));
}

// Python's spelling of a shape, for the assertion messages.
std::string shape_str(c10::IntArrayRef s) {
  std::string r = "(";
  for (size_t i = 0; i < s.size(); ++i) r += (i ? ", " : "") + std::to_string(s[i]);
  return r + (s.size() == 1 ? ",)" : ")");
}

c10::Device require_gpu(std::initializer_list<const Tensor*> ts) {
  std::optional<c10::Device> dev;
  for (const Tensor* t : ts) {
    if (!t->defined()) continue;
    if (!t->is_cuda())
      raise(PyExc_RuntimeError, c10::str("dwarf_amd DSQG ops need tensors on a ROCm GPU, got device ", t->device(),
                                         "; there is no CPU implementation"));
    if (!dev) dev = t->device();
    else if (*dev != t->device())
      raise(PyExc_RuntimeError, c10::str("tensors on different devices: ", *dev, " and ", t->device()));
  }
  return *dev;
}

dsqg_stream_t stream_of(const c10::Device& dev) {
  return reinterpret_cast<dsqg_stream_t>(c10::hip::getCurrentHIPStream(dev.index()).stream());
}

// ---- Offset tables. ----------------------------------------------------------------------------

struct Table : torch::CustomClassHolder {
  int J = 0;
  int NS = 0;  // taps beyond the dense window 0, 1, .., W (W <= 32)
  int32_t offsets[DSQG_MAX_OFFSETS] = {};
};
using TablePtr = c10::intrusive_ptr<Table>;

// A sequence of ints, strictly increasing from 0 (offsets.validate's rule and message).
TablePtr make_table(const py::object& seq) {
  TablePtr t = c10::make_intrusive<Table>();
  std::vector<long long> v;
  for (const py::handle& item : seq) {
    if (PyLong_CheckExact(item.ptr())) v.push_back(item.cast<long long>());
    else v.push_back(py::int_(py::reinterpret_borrow<py::object>(item)).cast<long long>());
  }
  bool ok = !v.empty() && v[0] == 0;
  for (size_t j = 1; ok && j < v.size(); ++j) ok = v[j] > v[j - 1];
  if (!ok) {
    py::tuple offs(v.size());
    for (size_t j = 0; j < v.size(); ++j) offs[j] = v[j];
    raise(PyExc_AssertionError, "offsets must be strictly increasing and start at 0: " + py::str(offs).cast<std::string>());
  }
  if (v.size() > DSQG_MAX_OFFSETS)
    raise(PyExc_ValueError, c10::str("offset table must have 1..", DSQG_MAX_OFFSETS, " entries, got ", v.size()));
  t->J = (int)v.size();
  for (int j = 0; j < t->J; ++j)
    t->offsets[j] = (int32_t)std::min<long long>(v[j], std::numeric_limits<int32_t>::max());
  int W = 0;
  while (W + 1 < t->J && W + 1 <= 32 && t->offsets[W + 1] == W + 1) ++W;
  t->NS = t->J - W - 1;
  return t;
}

void fill_shape(dsqg_shape& s, at::ScalarType dt, int64_t B, int64_t H, int64_t N, int64_t D, const Table& t) {
  s.dtype = dt == at::kFloat ? DSQG_F32 : DSQG_BF16;
  s.B = (int32_t)B; s.H = (int32_t)H; s.N = (int32_t)N; s.D = (int32_t)D; s.J = t.J;
  std::copy(std::begin(t.offsets), std::end(t.offsets), s.offsets);
}

// ---- Tensors as the kernels take them. -----------------------------------------------------------

void* ptr(const Tensor& t) { return !t.defined() || t.numel() == 0 ? nullptr : t.data_ptr(); }

// t if the kernels can read it in place (unit inner stride, 16-byte aligned rows), else a copy.
Tensor rows_ready(const Tensor& t) {
  if (t.numel() == 0) return t;
  const int64_t es = t.element_size(), d = t.dim();
  bool ok = t.stride(d - 1) == 1 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  for (int64_t i = 0; ok && i < d - 1; ++i) ok = t.stride(i) >= 0 && (t.stride(i) * es) % 16 == 0;
  return ok ? t : t.contiguous();
}

// fp32, contiguous and 16-byte aligned (the kernels read scale_embed as 16-byte pieces).
Tensor param(const Tensor& t) {
  if (!t.defined()) return t;
  if (t.scalar_type() == at::kFloat && t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0)
    return t;
  return t.detach().to(at::kFloat).clone(at::MemoryFormat::Contiguous);
}

void set_strides(int64_t (&dst)[4], const Tensor& t) {
  for (int i = 0; i < 4; ++i) dst[i] = t.stride(i);
}

// One of q, k, v (part 0, 1, 2) as a [B,H,N,HD] view of qkv [B,N,3*H*HD].
Tensor head_view(const Tensor& qkv, int64_t H, int64_t part) {
  const int64_t E = qkv.size(2) / 3, HD = E / H, sc = qkv.stride(2);
  return qkv.as_strided({qkv.size(0), H, qkv.size(1), HD}, {qkv.stride(0), HD * sc, qkv.stride(1), sc},
                        qkv.storage_offset() + part * E * sc);
}

struct Params {
  Tensor pb, se, sg, ig;  // undefined when absent
};

// ---- Forward. --------------------------------------------------------------------------------------

struct FwdOut {
  Tensor out, lse, alpha_lr;
};

FwdOut run_fwd(const Tensor& q0, const Tensor& k0, const Tensor& v0, const Params& P, const Table& t) {
  const c10::Device dev = require_gpu({&q0, &k0, &v0, &P.pb, &P.se, &P.sg, &P.ig});
  const auto dt = q0.scalar_type();
  require((dt == at::kFloat || dt == at::kBFloat16) && k0.scalar_type() == dt && v0.scalar_type() == dt,
          "q/k/v must share dtype float32 or bfloat16, got ", dt, "/", k0.scalar_type(), "/", v0.scalar_type());
  const c10::OptionalDeviceGuard guard(dev);
  const int64_t B = q0.size(0), H = q0.size(1), N = q0.size(2), D = q0.size(3);
  const Tensor q = rows_ready(q0), k = rows_ready(k0), v = rows_ready(v0);
  const Tensor pb = param(P.pb), se = param(P.se), sg = param(P.sg), ig = param(P.ig);
  const auto f32 = q.options().dtype(at::kFloat);
  FwdOut r;
  // Token-major storage: the callers' head merge is a view.
  r.out = at::empty_strided({B, H, N, D}, {N * H * D, D, H * D, 1}, q.options());
  r.lse = at::empty({B, H, N}, f32);
  if (dt == at::kBFloat16 && t.NS > 0) r.alpha_lr = at::empty({B, H, t.NS, N}, f32);
  else r.alpha_lr = at::empty({0}, f32);
  dsqg_fwd_args a = {};
  fill_shape(a.shape, dt, B, H, N, D, t);
  a.q = ptr(q); set_strides(a.q_stride, q);
  a.k = ptr(k); set_strides(a.k_stride, k);
  a.v = ptr(v); set_strides(a.v_stride, v);
  a.pos_bias = static_cast<const float*>(ptr(pb));
  a.scale_embed = static_cast<const float*>(ptr(se));
  a.score_gain = static_cast<const float*>(ptr(sg));
  a.if_gain = static_cast<const float*>(ptr(ig));
  a.out = ptr(r.out); set_strides(a.out_stride, r.out);
  a.lse = static_cast<float*>(ptr(r.lse));
  a.alpha_lr = static_cast<float*>(ptr(r.alpha_lr));
  check(api.fwd(&a, stream_of(dev)), "dsqg_fwd");
  return r;
}

// ---- Backward. ---------------------------------------------------------------------------------------

struct Grads {
  Tensor dq, dk, dv, dpb, dse, dsg, dig;  // dq, dk, dv allocated by the caller or here
};

void run_bwd(Grads& G, const Tensor& q0, const Tensor& k0, const Tensor& v0, const Tensor& dout0, const Tensor& lse0,
             const Tensor& alpha0, const Params& P, const Table& t, bool need_dse, bool need_dsg, bool need_dig) {
  const c10::Device dev = require_gpu({&q0, &k0, &v0, &dout0, &lse0, &P.pb, &P.se, &P.sg, &P.ig});
  const c10::OptionalDeviceGuard guard(dev);
  const auto dt = q0.scalar_type();
  const int64_t B = q0.size(0), H = q0.size(1), N = q0.size(2), D = q0.size(3);
  const Tensor q = rows_ready(q0), k = rows_ready(k0), v = rows_ready(v0), dout = rows_ready(dout0.to(dt));
  const Tensor lse = lse0.contiguous(), alpha = alpha0.contiguous();
  const Tensor pb = param(P.pb), se = param(P.se), sg = param(P.sg), ig = param(P.ig);
  const auto f32 = q.options().dtype(at::kFloat);
  if (!G.dq.defined()) {
    G.dq = at::empty({B, H, N, D}, q.options());
    G.dk = at::empty({B, H, N, D}, q.options());
    G.dv = at::empty({B, H, N, D}, q.options());
  }
  G.dpb = at::empty({t.J, H}, f32);
  if (need_dse) G.dse = at::empty({t.J, D}, f32);
  if (need_dsg) G.dsg = at::empty({H, t.J}, f32);
  if (need_dig) G.dig = at::empty({H}, f32);
  dsqg_bwd_args a = {};
  fill_shape(a.shape, dt, B, H, N, D, t);
  a.q = ptr(q); set_strides(a.q_stride, q);
  a.k = ptr(k); set_strides(a.k_stride, k);
  a.v = ptr(v); set_strides(a.v_stride, v);
  a.dout = ptr(dout); set_strides(a.dout_stride, dout);
  a.lse = static_cast<const float*>(ptr(lse));
  a.alpha_lr = static_cast<const float*>(ptr(alpha));
  a.pos_bias = static_cast<const float*>(ptr(pb));
  a.scale_embed = static_cast<const float*>(ptr(se));
  a.score_gain = static_cast<const float*>(ptr(sg));
  a.if_gain = static_cast<const float*>(ptr(ig));
  a.dq = ptr(G.dq); set_strides(a.dq_stride, G.dq);
  a.dk = ptr(G.dk); set_strides(a.dk_stride, G.dk);
  a.dv = ptr(G.dv); set_strides(a.dv_stride, G.dv);
  a.dpos_bias = static_cast<float*>(ptr(G.dpb));
  a.dscale_embed = static_cast<float*>(ptr(G.dse));
  a.dscore_gain = static_cast<float*>(ptr(G.dsg));
  a.dif_gain = static_cast<float*>(ptr(G.dig));
  size_t nbytes = 0;
  check(api.bwd_workspace_size(&a, &nbytes), "dsqg_bwd_workspace_size");
  const Tensor ws = at::empty({std::max<int64_t>((int64_t)nbytes, 1)}, q.options().dtype(at::kByte));
  a.workspace = ws.data_ptr();
  a.workspace_bytes = nbytes;
  check(api.bwd(&a, stream_of(dev)), "dsqg_bwd");
}

// ---- Autograd. ------------------------------------------------------------------------------------------

// Which of an autograd function's arguments, in their order, need a gradient (absent ones do not;
// the context counts only the tensors that are there).
struct Needs {
  std::array<bool, 8> need{};
  Needs(AutogradContext* ctx, std::initializer_list<bool> present) {
    size_t edge = 0, i = 0;
    for (bool p : present) need[i++] = p && ctx->needs_input_grad(edge++);
  }
};

OptTensor opt(const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; }
Tensor undef(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }

// The attention functions return lse and alpha_lr beside out, whose gradients never exist: left to
// autograd, each backward would fill a zero tensor for both (two launches, up to alpha_lr's size).
// Gradients arrive as they are instead, and only out's is made up where it is absent.  Forward +
// backward through the public call: B4 H8 N2047 D80 92 -> 81 us, B8 H12 N2048 D64 127 -> 121.
Tensor dout_of(const variable_list& g, const Tensor& q) { return g[0].defined() ? g[0] : at::zeros(q.sizes(), q.options()); }

Table& table_of(AutogradContext* ctx) {
  return *c10::static_intrusive_pointer_cast<Table>(ctx->saved_data["table"].toCapsule());
}

struct AttentionFunction : torch::autograd::Function<AttentionFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                               const Tensor& pb, const OptTensor& se, const OptTensor& sg, const OptTensor& ig,
                               const TablePtr& t) {
    const FwdOut r = run_fwd(q, k, v, {pb, undef(se), undef(sg), undef(ig)}, *t);
    ctx->save_for_backward({q, k, v, r.lse, r.alpha_lr, pb, undef(se), undef(sg), undef(ig)});
    ctx->saved_data["table"] = c10::IValue::make_capsule(t);
    ctx->mark_non_differentiable({r.lse, r.alpha_lr});
    ctx->set_materialize_grads(false);
    return {r.out, r.lse, r.alpha_lr};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const variable_list s = ctx->get_saved_variables();
    const Params P{s[5], s[6], s[7], s[8]};
    const Needs n(ctx, {true, true, true, true, P.se.defined(), P.sg.defined(), P.ig.defined()});
    Grads G;
    run_bwd(G, s[0], s[1], s[2], dout_of(g, s[0]), s[3], s[4], P, table_of(ctx), n.need[4], n.need[5], n.need[6]);
    return {G.dq, G.dk, G.dv, G.dpb, G.dse, G.dsg, G.dig, Tensor()};
  }
};

// q, k, v as the head views of one projection output; its gradient is one tensor.
struct AttentionQkvFunction : torch::autograd::Function<AttentionQkvFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& pb, const OptTensor& se,
                               const OptTensor& sg, const OptTensor& ig, int64_t H, const TablePtr& t) {
    const FwdOut r = run_fwd(head_view(qkv, H, 0), head_view(qkv, H, 1), head_view(qkv, H, 2),
                             {pb, undef(se), undef(sg), undef(ig)}, *t);
    ctx->save_for_backward({qkv, r.lse, r.alpha_lr, pb, undef(se), undef(sg), undef(ig)});
    ctx->saved_data["table"] = c10::IValue::make_capsule(t);
    ctx->saved_data["H"] = H;
    ctx->mark_non_differentiable({r.lse, r.alpha_lr});
    ctx->set_materialize_grads(false);
    return {r.out, r.lse, r.alpha_lr};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const variable_list s = ctx->get_saved_variables();
    const int64_t H = ctx->saved_data["H"].toInt();
    const Params P{s[3], s[4], s[5], s[6]};
    const Needs n(ctx, {true, true, P.se.defined(), P.sg.defined(), P.ig.defined()});
    const Tensor dqkv = at::empty_like(s[0], at::MemoryFormat::Contiguous);
    Grads G;
    G.dq = head_view(dqkv, H, 0); G.dk = head_view(dqkv, H, 1); G.dv = head_view(dqkv, H, 2);
    const Tensor q = head_view(s[0], H, 0);
    run_bwd(G, q, head_view(s[0], H, 1), head_view(s[0], H, 2), dout_of(g, q), s[1], s[2], P, table_of(ctx), n.need[2],
            n.need[3], n.need[4]);
    return {dqkv, G.dpb, G.dse, G.dsg, G.dig, Tensor(), Tensor()};
  }
};

// The attended operands of a K/V injection: q, K + k_delta and V + v_delta as [B,H,N,HD] views, in
// the compute type dt.
struct Injected {
  Tensor q, k, v;
};

Injected inject(const Tensor& qkv, const Tensor& kd, const Tensor& vd, int64_t H, at::ScalarType dt) {
  const int64_t B = qkv.size(0), N = qkv.size(1), E = qkv.size(2) / 3, HD = E / H;
  const bool cast = qkv.scalar_type() != dt;
  auto aligned = [](const Tensor& t) {
    bool ok = t.stride(t.dim() - 1) == 1 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
    for (int64_t i = 0; ok && i < t.dim() - 1; ++i) ok = t.stride(i) >= 0 && t.stride(i) * t.element_size() % 16 == 0;
    return ok;
  };
  // What the kernel takes; anything else is the casts and adds one by one.
  if (qkv.numel() == 0 || HD % 8 != 0 || E * qkv.element_size() % 16 != 0 || kd.scalar_type() != qkv.scalar_type() ||
      vd.scalar_type() != qkv.scalar_type() || !kd.is_cuda() || !vd.is_cuda() || !qkv.is_cuda() ||
      kd.device() != qkv.device() || vd.device() != qkv.device() || (cast && qkv.scalar_type() != at::kHalf) ||
      kd.is_neg() || vd.is_neg() || !aligned(qkv) || !aligned(kd) || !aligned(vd)) {
    const Tensor x = qkv.to(dt);
    return {head_view(x, H, 0), head_view(x, H, 1) + kd.to(dt), head_view(x, H, 2) + vd.to(dt)};
  }
  const c10::OptionalDeviceGuard guard(qkv.device());
  const int64_t parts = cast ? 3 : 2;  // q is read from qkv itself where the types agree
  const Tensor eff = at::empty({B, N, parts * E}, qkv.options().dtype(dt));
  auto view = [&](int64_t part) {
    return eff.as_strided({B, H, N, HD}, {N * parts * E, HD, parts * E, 1}, part * E);
  };
  Injected r{cast ? view(0) : head_view(qkv, H, 0), view(parts - 2), view(parts - 1)};
  auto code = [](at::ScalarType t) { return t == at::kFloat ? DSQG_F32 : t == at::kBFloat16 ? DSQG_BF16 : DSQG_F16; };
  dsqg_kv_inject_args a = {};
  a.B = (int32_t)B; a.H = (int32_t)H; a.N = (int32_t)N; a.D = (int32_t)HD;
  a.qkv_dtype = a.delta_dtype = code(qkv.scalar_type());
  a.out_dtype = code(dt);
  a.qkv = qkv.data_ptr(); a.qkv_stride[0] = qkv.stride(0); a.qkv_stride[1] = qkv.stride(1);
  a.k_delta = kd.data_ptr(); a.v_delta = vd.data_ptr();
  for (int i = 0; i < 3; ++i) { a.k_delta_stride[i] = kd.stride(i); a.v_delta_stride[i] = vd.stride(i); }
  a.q_out = cast ? r.q.data_ptr() : nullptr;
  a.k_out = r.k.data_ptr(); a.v_out = r.v.data_ptr();
  a.out_stride[0] = N * parts * E; a.out_stride[1] = parts * E;
  check(api.kv_inject(&a, stream_of(qkv.device())), "dsqg_kv_inject");
  return r;
}

// The same with a K/V injection: K + k_delta and V + v_delta are attended, and the K and V slices
// of d(qkv) are also the deltas' gradients.  Takes qkv in its own type (dt: the compute type).
struct AttentionQkvKvFunction : torch::autograd::Function<AttentionQkvKvFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& kd, const Tensor& vd,
                               const Tensor& pb, const OptTensor& se, const OptTensor& sg, const OptTensor& ig,
                               int64_t H, at::ScalarType dt, const TablePtr& t) {
    require_gpu({&qkv, &kd, &vd});
    const Injected x = inject(qkv, kd, vd, H, dt);
    const FwdOut r = run_fwd(x.q, x.k, x.v, {pb, undef(se), undef(sg), undef(ig)}, *t);
    ctx->save_for_backward({x.q, x.k, x.v, r.lse, r.alpha_lr, pb, undef(se), undef(sg), undef(ig)});
    ctx->saved_data["table"] = c10::IValue::make_capsule(t);
    ctx->saved_data["types"] = std::vector<int64_t>{(int64_t)qkv.scalar_type(), (int64_t)kd.scalar_type(),
                                                    (int64_t)vd.scalar_type()};
    ctx->mark_non_differentiable({r.lse, r.alpha_lr});
    ctx->set_materialize_grads(false);
    return {r.out, r.lse, r.alpha_lr};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const variable_list s = ctx->get_saved_variables();
    const std::vector<int64_t> types = ctx->saved_data["types"].toIntVector();
    const Params P{s[5], s[6], s[7], s[8]};
    const Needs n(ctx, {true, true, true, true, P.se.defined(), P.sg.defined(), P.ig.defined()});
    const int64_t B = s[0].size(0), H = s[0].size(1), N = s[0].size(2), HD = s[0].size(3);
    const Tensor dqkv = at::empty({B, N, 3 * H * HD}, s[0].options());
    Grads G;
    G.dq = head_view(dqkv, H, 0); G.dk = head_view(dqkv, H, 1); G.dv = head_view(dqkv, H, 2);
    run_bwd(G, s[0], s[1], s[2], dout_of(g, s[0]), s[3], s[4], P, table_of(ctx), n.need[4], n.need[5], n.need[6]);
    // One cast of the whole gradient; a delta of qkv's type takes its slice of the result.
    const Tensor dx = dqkv.to((at::ScalarType)types[0]);
    auto delta = [&](int part) {
      return types[part] == types[0] ? head_view(dx, H, part) : head_view(dqkv, H, part).to((at::ScalarType)types[part]);
    };
    return {dx, delta(1), delta(2), G.dpb, G.dse, G.dsg, G.dig, Tensor(), Tensor(), Tensor()};
  }
};

// ---- Public attention calls. ---------------------------------------------------------------------------------

// The per-tap and per-head parameters for H heads of HD over the table t (the kernels index them by these).
void check_params(const Params& P, int64_t H, int64_t HD, const Table& t) {
  const int64_t J = t.J;
  auto expect = [](const Tensor& x, c10::IntArrayRef s, const char* name) {
    if (x.defined() && x.sizes() != s) require(false, name, " must be ", shape_str(s), ", got ", shape_str(x.sizes()));
  };
  expect(P.pb, {J, H}, "pos_bias");
  expect(P.se, {J, HD}, "scale_embed");
  expect(P.sg, {H, J}, "score_gain");
  expect(P.ig, {H}, "if_gain");
}

void check_shapes(const Tensor& q, const Tensor& k, const Tensor& v, const Params& P, const Table& t) {
  require(q.dim() == 4, "q must be [B,H,N,HD], got ", shape_str(q.sizes()));
  require(k.sizes() == q.sizes() && v.sizes() == q.sizes(), "q, k, v must have the same shape");
  check_params(P, q.size(1), q.size(3), t);
}

Params float_params(const Tensor& pb, const OptTensor& se, const OptTensor& sg, const OptTensor& ig) {
  auto f = [](const Tensor& t) { return t.defined() ? t.to(at::kFloat) : t; };
  return {f(pb), f(undef(se)), f(undef(sg)), f(undef(ig))};
}

bool kernel_dtype(at::ScalarType dt) { return dt == at::kFloat || dt == at::kBFloat16; }

// (out, lse) with the dtype rules of the public functions.
std::tuple<Tensor, Tensor> attention(const Tensor& q0, const Tensor& k0, const Tensor& v0, const Tensor& pb,
                                     const OptTensor& se, const OptTensor& sg, const OptTensor& ig,
                                     const py::object& offsets) {
  const TablePtr t = make_table(offsets);
  py::gil_scoped_release nogil;
  check_shapes(q0, k0, v0, {pb, undef(se), undef(sg), undef(ig)}, *t);
  const auto orig = q0.scalar_type();
  const auto dt = kernel_dtype(orig) ? orig : at::kBFloat16;
  const Params P = float_params(pb, se, sg, ig);
  const variable_list r = AttentionFunction::apply(q0.to(dt), k0.to(dt), v0.to(dt), P.pb, opt(P.se), opt(P.sg),
                                                   opt(P.ig), t);
  return {r[0].to(orig), r[1]};
}

Tensor attention_qkv(const Tensor& qkv0, int64_t H, const Tensor& pb, const OptTensor& se, const OptTensor& sg,
                     const OptTensor& ig, const py::object& offsets, const OptTensor& kd, const OptTensor& vd) {
  const TablePtr t = make_table(offsets);
  py::gil_scoped_release nogil;
  const int64_t E3 = qkv0.size(2);
  require(H > 0 && E3 % (3 * H) == 0, "qkv last dim ", E3, " is not 3 * num_heads * head_dim");
  const std::vector<int64_t> heads{qkv0.size(0), H, qkv0.size(1), E3 / (3 * H)};
  check_params({pb, undef(se), undef(sg), undef(ig)}, H, heads[3], *t);
  const auto orig = qkv0.scalar_type();
  const auto dt = kernel_dtype(orig) ? orig : at::kBFloat16;
  const Params P = float_params(pb, se, sg, ig);
  variable_list r;
  if (!kd.has_value()) {
    r = AttentionQkvFunction::apply(qkv0.to(dt), P.pb, opt(P.se), opt(P.sg), opt(P.ig), H, t);
  } else {
    require(kd->sizes() == c10::IntArrayRef(heads) && vd->sizes() == c10::IntArrayRef(heads),
            "kv_inject deltas must be torch.Size([", heads[0], ", ", heads[1], ", ", heads[2], ", ", heads[3], "])");
    r = AttentionQkvKvFunction::apply(qkv0, *kd, *vd, P.pb, opt(P.se), opt(P.sg), opt(P.ig), H, dt, t);
  }
  return r[0].to(orig);
}

// ---- Decode step. ----------------------------------------------------------------------------------------------

Tensor decode(const Tensor& q0, const Tensor& k0, const Tensor& v0, const Tensor& k_ring, const Tensor& v_ring,
              const Tensor& pos0, const Tensor& pb0, const OptTensor& se0, const OptTensor& sg0,
              const OptTensor& ig0, const py::object& offsets) {
  const TablePtr t = make_table(offsets);
  py::gil_scoped_release nogil;
  require(k_ring.dim() == 4, "k_ring must be [B,H,S,D], got ", shape_str(k_ring.sizes()));
  check_params({pb0, undef(se0), undef(sg0), undef(ig0)}, k_ring.size(1), k_ring.size(3), *t);
  // (The kernel reads stored values: lazily negated operands are resolved, as the op's dispatch does.)
  auto ready = [](const Tensor& x) { return x.is_neg() ? x.resolve_neg().contiguous() : x.contiguous(); };
  auto f32 = [&](const Tensor& x) { return x.defined() ? ready(x.detach().to(at::kFloat)) : x; };
  const Tensor q = ready(q0), k = ready(k0), v = ready(v0);
  const Tensor pos = pos0.to(at::kLong).contiguous();
  const Tensor pb = f32(pb0), se = f32(undef(se0)), sg = f32(undef(sg0)), ig = f32(undef(ig0));
  const Tensor out = at::empty_like(q);
  const c10::Device dev = require_gpu({&q, &k, &v, &k_ring, &v_ring, &pos, &pb, &se, &sg, &ig, &out});
  const c10::OptionalDeviceGuard guard(dev);
  const int64_t B = k_ring.size(0), H = k_ring.size(1), S = k_ring.size(2), D = k_ring.size(3);
  const auto dt = q.scalar_type();
  require(kernel_dtype(dt) && k.scalar_type() == dt && v.scalar_type() == dt && k_ring.scalar_type() == dt &&
              v_ring.scalar_type() == dt, "q, k_new, v_new, rings and out must share dtype float32 or bfloat16");
  auto expect = [](const Tensor& x, std::vector<int64_t> s, const char* name) {
    if (x.sizes() != c10::IntArrayRef(s) || !x.is_contiguous())
      require(false, name, " must be a contiguous ", shape_str(s), " tensor, got ", shape_str(x.sizes()),
              " (contiguous=", x.is_contiguous() ? "True" : "False", ")");
  };
  expect(q, {B, H, D}, "q");
  expect(k, {B, H, D}, "k_new");
  expect(v, {B, H, D}, "v_new");
  expect(v_ring, {B, H, S, D}, "v_ring");
  require(k_ring.is_contiguous(), "k_ring must be contiguous");
  require(pos.dim() == 1 && pos.size(0) == B, "pos must be a contiguous int64 [B] tensor");
  dsqg_decode_args a = {};
  fill_shape(a.shape, dt, B, H, 0, D, *t);
  a.S = (int32_t)S;
  a.q = ptr(q); a.k_new = ptr(k); a.v_new = ptr(v);
  a.k_ring = ptr(k_ring); a.v_ring = ptr(v_ring);
  a.pos = static_cast<const int64_t*>(ptr(pos));
  a.pos_bias = static_cast<const float*>(ptr(pb));
  a.scale_embed = static_cast<const float*>(ptr(se));
  a.score_gain = static_cast<const float*>(ptr(sg));
  a.if_gain = static_cast<const float*>(ptr(ig));
  a.out = ptr(out);
  check(api.decode_step(&a, stream_of(dev)), "dsqg_decode_step");
  // The rings were written in place.
  for (const Tensor* r : {&k_ring, &v_ring})
    if (!r->is_inference()) r->unsafeGetTensorImpl()->bump_version();
  return out;
}

// Loads k, v [B,H,N,D] into the rings; false (nothing done) where the kernel does not take these
// tensors as they are: other shapes, types, layouts or devices, and whatever the indexed writes
// refuse or see more in than the stored values (a ring that records gradients or is an inference
// tensor outside inference mode, functorch wrappers, tangents, lazy negation).
bool ring_load(const Tensor& k, const Tensor& v, const Tensor& k_ring, const Tensor& v_ring, const Tensor& pos) {
  py::gil_scoped_release nogil;
  const auto dt = k_ring.scalar_type();
  if (!k_ring.is_cuda() || k.dim() != 4 || k_ring.dim() != 4 || v.sizes() != k.sizes() || v_ring.sizes() != k_ring.sizes() ||
      v_ring.scalar_type() != dt ||
      k.size(0) != k_ring.size(0) || k.size(1) != k_ring.size(1) || k.size(3) != k_ring.size(3) ||
      (dt != at::kFloat && dt != at::kBFloat16 && dt != at::kHalf) || pos.scalar_type() != at::kLong || pos.dim() != 1 ||
      pos.size(0) != k.size(0) || !pos.is_contiguous() || !k_ring.is_contiguous() || !v_ring.is_contiguous() || k.numel() == 0)
    return false;
  const int64_t es = k.element_size();
  for (const Tensor* t : {&k, &v}) {
    if (t->scalar_type() != dt || t->stride(3) != 1) return false;
    for (int i = 0; i < 3; ++i)
      if (t->stride(i) < 0 || t->stride(i) * es % 16 != 0) return false;
  }
  const bool grad = at::GradMode::is_enabled(), inference = c10::InferenceMode::is_enabled();
  for (const Tensor* t : {&k, &v, &k_ring, &v_ring, &pos})
    if (t->device() != k_ring.device() || t->key_set().has(c10::DispatchKey::Python) || !t->has_storage() || t->is_neg() ||
        (grad && t->requires_grad()) || t->_fw_grad(0).defined())
      return false;
  for (const Tensor* r : {&k_ring, &v_ring, &pos})
    if (r->is_inference() && !inference) return false;
  for (const Tensor* t : {&k, &v, &k_ring, &v_ring})
    if (reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 != 0) return false;
  if (k.size(3) * es % 16 != 0 || k.size(0) * k.size(1) > 65535) return false;
  const c10::OptionalDeviceGuard guard(k_ring.device());
  dsqg_ring_load_args a = {};
  a.dtype = dt == at::kFloat ? DSQG_F32 : dt == at::kBFloat16 ? DSQG_BF16 : DSQG_F16;
  a.B = (int32_t)k.size(0); a.H = (int32_t)k.size(1); a.N = (int32_t)k.size(2); a.D = (int32_t)k.size(3);
  a.S = (int32_t)k_ring.size(2);
  a.k = k.data_ptr(); a.v = v.data_ptr();
  for (int i = 0; i < 3; ++i) { a.k_stride[i] = k.stride(i); a.v_stride[i] = v.stride(i); }
  a.k_ring = k_ring.data_ptr(); a.v_ring = v_ring.data_ptr();
  a.pos = static_cast<int64_t*>(pos.data_ptr());
  const int status = api.ring_load(&a, stream_of(k_ring.device()));
  if (status == DSQG_EUNSUPPORTED) return false;
  check(status, "dsqg_ring_load");
  for (const Tensor* r : {&k_ring, &v_ring, &pos})
    if (!r->is_inference()) r->unsafeGetTensorImpl()->bump_version();
  return true;
}

// ---- Causal-mean pool with a sigmoid gate. ---------------------------------------------------------------------

int pool_code(at::ScalarType dt) { return dt == at::kFloat ? DSQG_F32 : dt == at::kBFloat16 ? DSQG_BF16 : DSQG_F16; }

Tensor pool_ready(const Tensor& t, const Tensor& like, const char* name) {
  const int64_t B = like.size(0), N = like.size(1), C = like.size(2);
  if (t.sizes() != like.sizes())
    require(false, name, " must be [", B, ",", N, ",", C, "], got ", shape_str(t.sizes()));
  const auto dt = t.scalar_type();
  require(dt == at::kFloat || dt == at::kBFloat16 || dt == at::kHalf, name,
          " must be float32, bfloat16 or float16, got ", dt);
  return rows_ready(t.numel() && t.stride(1) < C ? t.contiguous() : t);  // overlapping rows: copy
}

Tensor pool_workspace(const Tensor& x, bool backward) {
  size_t n = 0;
  check(api.pool_workspace_size((int32_t)x.size(0), (int32_t)x.size(1), (int32_t)x.size(2), backward, &n),
        "dsqg_pool_gate_workspace_size");
  return at::empty({std::max<int64_t>((int64_t)n, 1)}, x.options().dtype(at::kByte));
}

void set_strides(int64_t (&dst)[2], const Tensor& t) { dst[0] = t.stride(0); dst[1] = t.stride(1); }

struct PoolFunction : torch::autograd::Function<PoolFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x0, const Tensor& g0) {
    const c10::Device dev = require_gpu({&x0, &g0});
    const c10::OptionalDeviceGuard guard(dev);
    const Tensor x = pool_ready(x0, x0, "x"), g = pool_ready(g0, x0, "gate_pre"), ws = pool_workspace(x, false);
    const Tensor out = at::empty(x.sizes(), x.options().dtype(at::promote_types(x.scalar_type(), g.scalar_type())));
    dsqg_pool_gate_fwd_args a = {};
    a.B = (int32_t)x.size(0); a.N = (int32_t)x.size(1); a.C = (int32_t)x.size(2);
    a.x_dtype = pool_code(x.scalar_type()); a.gate_dtype = pool_code(g.scalar_type());
    a.out_dtype = pool_code(out.scalar_type());
    a.x = ptr(x); set_strides(a.x_stride, x);
    a.gate_pre = ptr(g); set_strides(a.gate_stride, g);
    a.out = ptr(out); set_strides(a.out_stride, out);
    a.workspace = ws.data_ptr(); a.workspace_bytes = (size_t)ws.numel();
    check(api.pool_fwd(&a, stream_of(dev)), "dsqg_pool_gate_fwd");
    ctx->save_for_backward({x0, g0});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list s = ctx->get_saved_variables();
    const bool need_dx = ctx->needs_input_grad(0), need_dg = ctx->needs_input_grad(1);
    if (!need_dx && !need_dg) return {Tensor(), Tensor()};
    const c10::Device dev = require_gpu({&s[0], &s[1], &grads[0]});
    const c10::OptionalDeviceGuard guard(dev);
    const Tensor x = pool_ready(s[0], s[0], "x"), g = pool_ready(s[1], s[0], "gate_pre");
    const Tensor dy = pool_ready(grads[0], s[0], "dout"), ws = pool_workspace(x, true);
    Tensor dx, dg;
    dsqg_pool_gate_bwd_args a = {};
    a.B = (int32_t)x.size(0); a.N = (int32_t)x.size(1); a.C = (int32_t)x.size(2);
    a.x_dtype = pool_code(x.scalar_type()); a.gate_dtype = pool_code(g.scalar_type());
    a.dout_dtype = pool_code(dy.scalar_type());
    a.x = ptr(x); set_strides(a.x_stride, x);
    a.gate_pre = ptr(g); set_strides(a.gate_stride, g);
    a.dout = ptr(dy); set_strides(a.dout_stride, dy);
    if (need_dx) {
      dx = at::empty(x.sizes(), x.options());
      a.dx = ptr(dx); set_strides(a.dx_stride, dx);
    }
    if (need_dg) {
      dg = at::empty(x.sizes(), g.options());
      a.dgate_pre = ptr(dg); set_strides(a.dgate_stride, dg);
    }
    a.workspace = ws.data_ptr(); a.workspace_bytes = (size_t)ws.numel();
    check(api.pool_bwd(&a, stream_of(dev)), "dsqg_pool_gate_bwd");
    return {dx, dg};
  }
};

Tensor pool_gate(const Tensor& x, const Tensor& g) {
  py::gil_scoped_release nogil;
  return PoolFunction::apply(x, g);
}

// ---- Linear layers: the library's products, and dW and db from one kernel pair. -----------------------------------

// Whether the weight gradient goes to dsqg_linear_wgrad: 16-bit operands of aligned widths, and an
// output small enough that the library's tiling of it alone leaves most of the chip idle.  Against
// its product and column sum, both callers' host time included (us, either type), by O x I and rows:
//                 512      2048      4096       16384      32768       65536
//   256 x 256   9 / 29   10 / 27   11 / 41    18 / 114    17 / 139    24 / 242
//   768 x 768  12 / 27   20 / 29   24 / 46    45 / 114    79 / 212   145 / 308
//  1024 x 2048 20 / 27   25 / 34   37 / 55   112 / 145   214 / 321   500 / 573
//  1536 x 1536 21 / 29   29 / 42   44 / 64   144 / 178   277 / 330   562 / 596
//  3072 x 768  21 / 27   29 / 42   44 / 60   143 / 178   277 / 327   571 / 514
//  1792 x 1792 24 / 29   32 / 44   51 / 64   162 / 176   312 / 345   621 / 660
//  2048 x 2048 25 / 27   40 / 44   65 / 62   215 / 180   468 / 318   965 / 604
// The library's time depends on the shape where the two are close, so the lines lie inside: up to
// 2^21 outputs, where every measured row count wins by an eighth or more, and up to 3072 x 768, the
// widest layer of the reference's models, for the rows at which every such shape wins by a seventh.
bool use_wgrad(at::ScalarType dt, int64_t T, int64_t O, int64_t I) {
  if ((dt != at::kHalf && dt != at::kBFloat16) || T < 1 || O < 1 || O % 8 != 0 || I % 8 != 0) return false;
  if ((T + 128) * std::max(O, I) * 2 >= (1ll << 31)) return false;
  return O * I <= (1ll << 21) || (O * I <= 3072 * 768 && T <= 16384);
}

// [T, C] rows the kernel reads in place (unit column stride, 16-byte aligned rows that do not
// overlap), else a copy.
Tensor wgrad_rows(const Tensor& t) {
  const bool ok = t.stride(1) == 1 && t.stride(0) >= t.size(1) && t.stride(0) % 8 == 0 &&
                  (t.size(0) + 128) * t.stride(0) * 2 < (1ll << 31) && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  return ok ? t : t.clone(at::MemoryFormat::Contiguous);
}

void linear_wgrad(const Tensor& dy0, const Tensor& x0, at::ScalarType out, bool need_db, Tensor& dw, Tensor& db) {
  const c10::Device dev = require_gpu({&dy0, &x0});
  const c10::OptionalDeviceGuard guard(dev);
  const Tensor dy = wgrad_rows(dy0.resolve_neg()), x = wgrad_rows(x0);
  dw = at::empty({dy.size(1), x.size(1)}, x.options().dtype(out));
  if (need_db) db = at::empty({dy.size(1)}, x.options().dtype(out));
  dsqg_linear_wgrad_args a = {};
  a.T = (int32_t)dy.size(0); a.O = (int32_t)dy.size(1); a.I = (int32_t)x.size(1);
  a.dtype = pool_code(x.scalar_type());
  a.out_dtype = pool_code(out);
  a.dy = dy.data_ptr(); a.dy_stride = dy.stride(0);
  a.x = x.data_ptr(); a.x_stride = x.stride(0);
  a.dw = dw.data_ptr();
  a.db = need_db ? db.data_ptr() : nullptr;
  size_t nbytes = 0;
  check(api.linear_workspace_size(&a, &nbytes), "dsqg_linear_wgrad_workspace_size");
  const Tensor ws = at::empty({(int64_t)nbytes}, x.options().dtype(at::kByte));
  a.workspace = ws.data_ptr(); a.workspace_bytes = nbytes;
  check(api.linear_wgrad(&a, stream_of(dev)), "dsqg_linear_wgrad");
}

// w with the history of a cast of w0.
struct CastOf : torch::autograd::Function<CastOf> {
  static Tensor forward(AutogradContext* ctx, const Tensor& w0, const Tensor& w) {
    ctx->saved_data["type"] = (int64_t)w0.scalar_type();
    return w;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    return {g[0].to((at::ScalarType)ctx->saved_data["type"].toInt()), Tensor()};
  }
};

// x in the compute type; w in it too, or the float32 leaf parameter that autocast would cast: the
// cast happens here, its gradient and b0's come out of the kernel in float32, and only the copy is
// saved (the parameter may change before the backward, as under nn.Linear).  A weight with a history
// of its own comes as its cast w and, for the float32 gradient, as w0.  (A cast recorded for every
// weight costs the block of eight layers 100 us of host time a step.)  Under create_graph the
// gradients are themselves differentiated: plain products of the inputs, the weight's through its cast.
struct LinearFunction : torch::autograd::Function<LinearFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, const OptTensor& w0, const OptTensor& b0) {
    const auto dt = x.scalar_type();
    const Tensor wc = w.to(dt);
    ctx->save_for_backward({x, x.requires_grad() ? wc : Tensor()});  // (the weight serves dx alone)
    ctx->saved_data["type"] = (int64_t)(w0 ? *w0 : w).scalar_type();
    ctx->saved_data["cast"] = w0.has_value();
    if (w.scalar_type() != dt) ctx->saved_data["leaf"] = w;
    ctx->saved_data["bias"] = b0.has_value();
    return at::linear(x, wc, b0 ? OptTensor(b0->to(dt)) : OptTensor());
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const variable_list s = ctx->get_saved_variables();
    const bool cast = ctx->saved_data["cast"].toBool();
    const Needs n(ctx, {true, true, cast, ctx->saved_data["bias"].toBool()});
    const Tensor &x = s[0], &w = s[1], &dy = g[0];
    const int64_t O = dy.size(-1), I = x.size(-1);
    const auto out = (at::ScalarType)ctx->saved_data["type"].toInt();
    const bool plain = at::GradMode::is_enabled(), need_dw = n.need[1] || n.need[2];
    Tensor dx, dw, db;
    if (n.need[0]) {
      const auto leaf = ctx->saved_data.find("leaf");
      dx = at::matmul(dy, plain && leaf != ctx->saved_data.end() ? CastOf::apply(leaf->second.toTensor(), w) : w);
    }
    if (need_dw || n.need[3]) {
      const Tensor dy2 = dy.reshape({-1, O});
      if (need_dw && !plain && dy.scalar_type() == x.scalar_type() && use_wgrad(x.scalar_type(), dy2.size(0), O, I)) {
        linear_wgrad(dy2, x.reshape({-1, I}), out, n.need[3], dw, db);
      } else {
        if (need_dw) dw = dy2.t().mm(x.reshape({-1, I}));
        if (n.need[3]) db = dy2.sum(0).to(out);
      }
    }
    if (cast && plain) return {dx, dw, Tensor(), db};
    if (dw.defined()) dw = dw.to(out);
    return cast ? variable_list{dx, Tensor(), dw, db} : variable_list{dx, dw, Tensor(), db};
  }
};

// F.linear on GPU tensors.  Under autocast the operands take the types F.linear's would; anything
// but 16-bit training on plain tensors is F.linear itself.
Tensor linear(const Tensor& x0, const Tensor& w0, const OptTensor& b0) {
  py::gil_scoped_release nogil;
  auto plain = [](const Tensor& t) {
    return t.is_cuda() && t.layout() == at::kStrided && !t.is_neg() && !t.key_set().has(c10::DispatchKey::Python);
  };
  if (!at::GradMode::is_enabled() || !w0.requires_grad() || !plain(x0) || !plain(w0) || (b0 && !plain(*b0)) ||
      x0.dim() < 2 || w0.dim() != 2 || x0.numel() == 0 || (b0 && b0->scalar_type() != w0.scalar_type()))
    return at::linear(x0, w0, b0);
  const bool autocast = at::autocast::is_autocast_enabled(at::kCUDA);
  const auto dt = autocast ? at::autocast::get_autocast_dtype(at::kCUDA) : x0.scalar_type();
  const auto wt = w0.scalar_type();
  const bool types_ok = autocast ? (wt == at::kFloat || wt == dt) && (x0.scalar_type() == at::kFloat || kernel_dtype(x0.scalar_type()) ||
                                                                      x0.scalar_type() == at::kHalf)
                                 : wt == dt;
  if (!types_ok || x0.size(-1) != w0.size(1) || !use_wgrad(dt, x0.numel() / x0.size(-1), w0.size(0), w0.size(1)))
    return at::linear(x0, w0, b0);
  const Tensor x = autocast ? at::autocast::cached_cast(dt, x0, at::kCUDA) : x0;
  if (wt == dt || w0.is_leaf()) return LinearFunction::apply(x, w0, OptTensor(), b0);
  return LinearFunction::apply(x, w0.to(dt), OptTensor(w0), b0);
}

void init(const py::dict& addresses, const py::object& library_error) {
  auto get = [&](auto& fn, const char* name) {
    fn = reinterpret_cast<std::decay_t<decltype(fn)>>(addresses[name].cast<uintptr_t>());
  };
  get(api.status_string, "dsqg_status_string");
  get(api.fwd, "dsqg_fwd");
  get(api.bwd_workspace_size, "dsqg_bwd_workspace_size");
  get(api.bwd, "dsqg_bwd");
  get(api.decode_step, "dsqg_decode_step");
  get(api.kv_inject, "dsqg_kv_inject");
  get(api.ring_load, "dsqg_ring_load");
  get(api.pool_workspace_size, "dsqg_pool_gate_workspace_size");
  get(api.pool_fwd, "dsqg_pool_gate_fwd");
  get(api.pool_bwd, "dsqg_pool_gate_bwd");
  get(api.linear_workspace_size, "dsqg_linear_wgrad_workspace_size");
  get(api.linear_wgrad, "dsqg_linear_wgrad");
  api.library_error = library_error.inc_ref().ptr();  // lives as long as the process
}

}  // namespace

PYBIND11_MODULE(_dsqg_host, m) {
  m.doc() = "Native host layer of dwarf_amd's eager public functions.";
  m.attr("abi_version") = DSQG_ABI_VERSION;  // of the argument blocks compiled in here
  m.def("init", &init);
  m.def("attention", &attention);
  m.def("attention_qkv", &attention_qkv);
  m.def("decode", &decode);
  m.def("ring_load", &ring_load);
  m.def("pool_gate", &pool_gate);
  m.def("linear", &linear);
}
