// The operator's host path between torch tensors and the C ABI (include/trifast_hip.h), as
// a Python extension module (trifast_amd._host): argument checks, layouts, output and
// workspace allocation, the launches, and the autograd node around them.
//
// What bounds small calls is the host: at n = 256 the kernels of a training step take about
// 0.12 ms, and the same steps in Python (stride arrays, ctypes marshalling, autograd nodes
// whose backward has to take the interpreter lock in the engine's thread) took 0.25 ms; at
// n = 32 0.24 ms around 0.08 ms of kernels.  Here a call is some tens of microseconds and the
// backward runs without the interpreter.
//
// Everything that is not an ordinary eager call on plain GPU tensors (tracing, transforms,
// autocast, other devices, wrong shapes) is declined (attention() returns None): the caller
// then goes through the registered operators, which trace, transform or raise.
//
// Tiles are chosen in Python (trifast_amd/tuner.py); a choice is remembered here per shape
// until forget_tiles().
#include <torch/extension.h>

#include <ATen/FuncTorchTLS.h>
#include <ATen/TracerMode.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <cctype>
#include <cstdlib>
#include <mutex>
#include <string>
#include <tuple>
#include <unordered_map>

#include "../../include/trifast_hip.h"

namespace py = pybind11;
using at::Tensor;

// A tensor as Python gives it: `overrides` for a subclass other than Parameter, which may have a
// __torch_function__ of its own that the registered operators call and the native path would pass by.
struct PyTensor {
  Tensor t;
  bool overrides = false;
};
template <>
struct py::detail::type_caster<PyTensor> {
  PYBIND11_TYPE_CASTER(PyTensor, const_name("torch.Tensor"));
  bool load(handle src, bool convert) {
    make_caster<Tensor> tensor;
    if (!tensor.load(src, convert)) return false;
    value.t = std::move(cast_op<Tensor&>(tensor));
    value.overrides = !THPVariable_CheckTypeExact(Py_TYPE(src.ptr()));
    return true;
  }
};

namespace {

void check(int rc, const char* what) {
  if (rc == 0) return;
  const std::string msg = std::string(what) + " failed (" + std::to_string(rc) + "): " + trifast_last_error();
  if (rc < 0) throw py::value_error(msg);
  throw std::runtime_error(msg);
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return TRIFAST_F32;
    case at::kBFloat16: return TRIFAST_BF16;
    case at::kHalf: return TRIFAST_F16;
    default: return -1;
  }
}

// element strides as the C ABI takes them; the stride of a size-1 dim is never used for
// addressing and is reported as 0
struct Strides {
  int64_t s[5];
  explicit Strides(const Tensor& t) {
    const auto sz = t.sizes(), st = t.strides();
    for (size_t x = 0; x < sz.size(); ++x) s[x] = sz[x] == 1 ? 0 : st[x];
  }
  operator const int64_t*() const { return s; }
};

// q-like tensors: rows of d contiguous elements, 16-byte aligned, less than 2^24 bytes apart along j
bool rows_ok(const Tensor& t) {
  const Strides st(t);
  const int64_t es = t.element_size(), vec = 16 / es;
  if (st.s[4] != 1 || st.s[3] < 0 || st.s[3] * es >= (int64_t(1) << 24)) return false;
  for (int x = 0; x < 4; ++x)
    if (st.s[x] % vec != 0) return false;
  return true;
}

// (as trifast_amd.torch._vector_ready: transposed views are read in place, the rest is copied)
Tensor vector_ready(const Tensor& t) {
  return rows_ok(t) && reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0 ? t : t.contiguous();
}

// An upstream gradient that is one [d] row expanded over b, h, i, j is read through zero
// strides: nothing of q's size is materialised.
Tensor broadcast_rows(const Tensor& t) {
  const Strides st(t);
  if (st.s[0] || st.s[1] || st.s[2] || st.s[3]) return t;
  return t.select(0, 0).select(0, 0).select(0, 0).select(0, 0).contiguous().expand(t.sizes());
}

// Gradient buffer of input t, in t's layout where the kernels can write it.
Tensor grad_like(const Tensor& t) {
  if ((t.dim() == 4 || rows_ok(t)) && t.is_non_overlapping_and_dense()) return at::empty_strided(t.sizes(), t.strides(), t.options());
  return at::empty(t.sizes(), t.options());
}

hipStream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor workspace(int64_t bytes, const Tensor& like) {
  return at::empty({std::max<int64_t>(bytes, 256)}, like.options().dtype(at::kByte));
}

// ---- tile choice ------------------------------------------------------------------------

bool env_true(const char* name, bool otherwise) {
  const char* v = std::getenv(name);
  if (!v) return otherwise;
  std::string s(v);
  for (char& ch : s) ch = (char)std::tolower((unsigned char)ch);
  return s == "1" || s == "true" || s == "yes" || s == "on";
}

using Tiles = std::array<int, 3>;
std::mutex g_tiles_mutex;
std::unordered_map<uint64_t, Tiles> g_tiles;
constexpr size_t kMaxTiles = 4096;

// (heap-held: destroyed never, so not after the interpreter)
struct Choosers { py::object fwd, bwd; };
Choosers* g_choosers = nullptr;

struct Shape {
  int64_t b, h, n, d;
  int code;
};

uint64_t tiles_key(const Shape& s, bool bwd, bool tuned) {
  return (uint64_t)s.n | (uint64_t)s.h << 17 | (uint64_t)s.d << 37 | (uint64_t)s.code << 46 | (uint64_t)bwd << 49 | (uint64_t)tuned << 50;
}

template <typename Choose>
Tiles tiles_for(const Shape& s, bool bwd, Choose choose) {
  const bool force = env_true("TRIFAST_FORCE_TUNE", false);
  const uint64_t key = tiles_key(s, bwd, env_true("TRIFAST_AUTOTUNE", true));
  if (!force) {
    std::lock_guard<std::mutex> lock(g_tiles_mutex);
    const auto it = g_tiles.find(key);
    if (it != g_tiles.end()) return it->second;
  }
  Tiles tiles{-1, -1, -1};
  bool keep = false;
  {
    py::gil_scoped_acquire gil;
    TORCH_CHECK(g_choosers, "trifast: no tile chooser registered");
    std::tie(tiles, keep) = choose();
  }
  if (keep) {
    std::lock_guard<std::mutex> lock(g_tiles_mutex);
    if (force || g_tiles.size() >= kMaxTiles) g_tiles.clear();  // (a forced choice may stand for other shapes too)
    g_tiles[key] = tiles;
  }
  return tiles;
}

// ---- the operator -----------------------------------------------------------------------

Shape shape_of(const Tensor& q) {
  return Shape{q.size(0), q.size(1), q.size(2), q.size(4), dtype_code(q.scalar_type())};
}

// Every requirement trifast_amd.torch._check_inputs states, without the messages.
bool inputs_ok(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& b, const Tensor& mask) {
  if (q.dim() != 5 || q.size(2) != q.size(3) || dtype_code(q.scalar_type()) < 0) return false;
  if (k.sizes() != q.sizes() || v.sizes() != q.sizes()) return false;
  const int64_t bs = q.size(0), h = q.size(1), n = q.size(2);
  if (b.dim() != 4 || b.size(0) != bs || b.size(1) != h || b.size(2) != n || b.size(3) != n) return false;
  if (mask.dim() != 3 || mask.size(0) != bs || mask.size(1) != n || mask.size(2) != n || mask.scalar_type() != at::kBool) return false;
  const auto t = q.scalar_type();
  if (k.scalar_type() != t || v.scalar_type() != t || b.scalar_type() != t || !q.is_cuda()) return false;
  const auto dev = q.device();
  return k.device() == dev && v.device() == dev && b.device() == dev && mask.device() == dev && q.numel() > 0;
}

struct Forward { Tensor o, lse, ws; };

// train: f.ws is for the backward of the step (the pre-passes' results: b h n^2 elements and one bit
// per mask byte)
Forward forward(Tensor q, Tensor k, Tensor v, const Tensor& b, const Tensor& mask, bool train = false) {
  const c10::DeviceGuard guard(q.device());
  const Shape s = shape_of(q);
  const Tiles tiles = tiles_for(s, false, [&] { return g_choosers->fwd(q, k, v, b, mask).cast<std::tuple<Tiles, bool>>(); });
  Forward f;
  f.o = at::empty(q.sizes(), q.options().memory_format(at::MemoryFormat::Contiguous));
  f.lse = at::empty({s.b, s.h, s.n, s.n}, q.options().dtype(at::kFloat));
  f.ws = workspace((train ? trifast_train_workspace_bytes : trifast_fwd_workspace_bytes)(s.b, s.h, s.n, s.d, s.code), q);
  q = vector_ready(q), k = vector_ready(k), v = vector_ready(v);
  check((train ? trifast_fwd_train : trifast_fwd)(f.o.mutable_data_ptr(), f.lse.mutable_data_ptr<float>(), q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(),
                    b.const_data_ptr(), static_cast<const uint8_t*>(mask.const_data_ptr()), s.b, s.h, s.n, s.d, s.code, Strides(q), Strides(k),
                    Strides(v), Strides(b), Strides(mask), tiles[0], f.ws.mutable_data_ptr(), f.ws.numel(), stream_of(q)),
        "trifast_fwd");
  return f;
}

// The upstream gradient as numbers in memory: autograd may hand a node a lazily negated view, or a
// zero tensor without any.
Tensor materialized(const Tensor& g) {
  if (g._is_zerotensor()) return at::zeros(g.sizes(), g.options());
  return g.is_neg() ? g.resolve_neg() : g;
}

using Grads = std::array<Tensor, 4>;

Grads backward(Tensor dout, Tensor q, Tensor k, Tensor v, const Tensor& b, Tensor o, Tensor lse, const Tensor& mask, const Tensor& saved = Tensor()) {
  const c10::DeviceGuard guard(q.device());
  const Shape s = shape_of(q);
  dout = materialized(dout);
  if (dout.scalar_type() != q.scalar_type()) dout = dout.to(q.scalar_type());
  dout = vector_ready(broadcast_rows(dout));
  o = o.contiguous();
  lse = lse.contiguous();
  const Tiles tiles = tiles_for(s, true, [&] { return g_choosers->bwd(dout, q, k, v, b, o, lse, mask).cast<std::tuple<Tiles, bool>>(); });
  Grads g{grad_like(q), grad_like(k), grad_like(v), grad_like(b)};  // (the layout of the caller's tensors, not of a vector-ready copy)
  q = vector_ready(q), k = vector_ready(k), v = vector_ready(v);
  Tensor ws = workspace(trifast_bwd_workspace_bytes(s.b, s.h, s.n, s.d, s.code), q);
  auto run = [&](auto... args) { return saved.defined() ? trifast_bwd_train(saved.const_data_ptr(), args...) : trifast_bwd(args...); };
  check(run(g[0].mutable_data_ptr(), g[1].mutable_data_ptr(), g[2].mutable_data_ptr(), g[3].mutable_data_ptr(), dout.const_data_ptr(),
                    q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), b.const_data_ptr(), static_cast<const uint8_t*>(mask.const_data_ptr()),
                    o.const_data_ptr(), lse.const_data_ptr<float>(), s.b, s.h, s.n, s.d, s.code, Strides(dout).s, Strides(q).s, Strides(k).s, Strides(v).s,
                    Strides(b).s, Strides(mask).s, Strides(g[0]).s, Strides(g[1]).s, Strides(g[2]).s, Strides(g[3]).s, tiles.data(), ws.mutable_data_ptr(),
                    ws.numel(), stream_of(q)),
        "trifast_bwd");
  return g;
}

// (the views that turn the ending-node problem into the starting-node one)
Tensor swap_pair(const Tensor& t, bool ending) {
  if (!ending || !t.defined()) return t;
  return t.dim() == 5 ? t.transpose(2, 3) : t.transpose(-1, -2);
}

// The gradients of a backward that ran the kernels.  They have no graph: where the caller asked for
// one (create_graph turns grad mode on in the backward) they come from a node over the tensors they
// were made of that raises when it is differentiated: a penalty on a gradient is not silently a constant.
torch::autograd::variable_list once_differentiable(torch::autograd::variable_list grads, const torch::autograd::variable_list& saved, const Tensor& dout,
                                                   const char* what) {
  if (!at::GradMode::is_enabled()) return grads;
  const size_t n = grads.size();
  grads.push_back(dout);
  for (const Tensor& t : saved)
    if (t.defined() && t.requires_grad()) grads.push_back(t);
  torch::autograd::DelayedError raises(std::string("trifast: the backward of ") + what + " has no second derivative", static_cast<int>(grads.size()));
  grads = raises(std::move(grads));
  grads.resize(n);
  return grads;
}

struct Attention : torch::autograd::Function<Attention> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& b,
                        const Tensor& mask, bool ending) {
    at::AutoDispatchBelowADInplaceOrView below;
    Forward f = ::forward(swap_pair(q, ending), swap_pair(k, ending), swap_pair(v, ending), swap_pair(b, ending), swap_pair(mask, ending), true);
    Tensor out = swap_pair(f.o, ending);
    ctx->save_for_backward({q, k, v, b, mask, out, f.lse, f.ws});
    ctx->saved_data["ending"] = ending;
    ctx->set_materialize_grads(false);
    return out;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const bool ending = ctx->saved_data["ending"].toBool();
    torch::autograd::variable_list out(6);
    if (!grads[0].defined()) return out;
    {
      at::AutoDispatchBelowADInplaceOrView below;
      auto t = [&](int x) { return swap_pair(saved[x], ending); };
      const Grads g = ::backward(swap_pair(grads[0], ending), t(0), t(1), t(2), t(3), t(5), saved[6], t(4), saved[7]);
      for (int i = 0; i < 4; ++i) out[i] = swap_pair(g[i], ending);
    }
    return once_differentiable(std::move(out), saved, grads[0], "triangle attention");
  }
};

// Ordinary eager execution: no function transforms, no dispatch modes, no autocast, no tracer (which
// would record the allocations made here and none of the launches), plain tensors without a forward-mode tangent (the kernels have no rule for it, and the launches here would drop it).
bool plain_eager(std::initializer_list<const Tensor*> tensors) {
  using c10::DispatchKey;
  if (at::autocast::is_autocast_enabled(at::kCUDA) || at::tracer::impl::is_dispatch_enabled()) return false;
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  if (tls.included_.has(DispatchKey::Python) || tls.included_.has(DispatchKey::FuncTorchDynamicLayerFrontMode)) return false;
  if (c10::impl::TorchDispatchModeTLS::stack_len() > 0) return false;
  // (lazily negated or conjugated tensors and zero tensors: their memory does not hold their numbers)
  constexpr c10::DispatchKeySet kOther({DispatchKey::Python, DispatchKey::FuncTorchGradWrapper, DispatchKey::FuncTorchBatched, DispatchKey::Negative,
                                        DispatchKey::Conjugate, DispatchKey::ZeroTensor});
  for (const Tensor* t : tensors)
    if (!t->defined() || t->key_set().has_any(kOther) || t->layout() != at::kStrided || t->_fw_grad(/*level=*/0).defined()) return false;
  return true;
}

bool wants_grad(std::initializer_list<const Tensor*> tensors) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : tensors)
    if (t->requires_grad()) return true;
  return false;
}

// The operator on plain tensors; none where the call has to take another path.
std::optional<Tensor> attention(const PyTensor& q_, const PyTensor& k_, const PyTensor& v_, const PyTensor& b_, const PyTensor& mask_, bool ending) {
  if (q_.overrides || k_.overrides || v_.overrides || b_.overrides || mask_.overrides) return std::nullopt;
  const Tensor &q = q_.t, &k = k_.t, &v = v_.t, &b = b_.t, &mask = mask_.t;
  if (!plain_eager({&q, &k, &v, &b, &mask}) || !inputs_ok(q, k, v, b, mask)) return std::nullopt;
  if (wants_grad({&q, &k, &v, &b})) return Attention::apply(q, k, v, b, mask, ending);
  at::AutoDispatchBelowADInplaceOrView below;
  return swap_pair(
      ::forward(swap_pair(q, ending), swap_pair(k, ending), swap_pair(v, ending), swap_pair(b, ending), swap_pair(mask, ending)).o, ending);
}

// ---- the gated block --------------------------------------------------------------------
//
// trifast_amd.nn.TriangleAttention as one node: the projections, the operator, and the gated output
// layer.  Everything between x and the output lies in the order the operator works in (for the
// ending node: the pair-transposed one), so the operator always reads and writes contiguous rows;
// the kernels that read x and dout or write dx and the output map their rows.

// A dense tensor whose first byte is 16-byte aligned
Tensor dense(const Tensor& t) {
  Tensor c = t.contiguous();
  return reinterpret_cast<uintptr_t>(c.const_data_ptr()) % 16 == 0 ? c : c.clone();
}

struct BlockShape {
  int64_t b, n, c, h, d;
  bool ending;
  int code;
  BlockShape(const Tensor& x, int64_t h_, int64_t d_, bool ending_)
      : n(x.size(-2)), c(x.size(-1)), h(h_), d(d_), ending(ending_), code(dtype_code(x.scalar_type())) {
    b = n > 0 && c > 0 ? x.numel() / (n * n * c) : 0;
  }
};

// parameters in this order; a missing bias is an undefined tensor
enum { WQ, WK, WV, WB, WG, BG, WO, BO, NPARAMS };
using Params = std::array<Tensor, NPARAMS>;

bool block_ok(const Tensor& x, const Tensor& mask, const Params& p, int64_t h, int64_t d) {
  if (x.dim() < 3 || x.size(-2) != x.size(-3) || !x.is_cuda() || x.numel() == 0 || h < 1) return false;
  if (x.scalar_type() != at::kBFloat16 && x.scalar_type() != at::kHalf) return false;
  const int64_t c = x.size(-1), hd = h * d;
  if (c != 32 && c != 64 && c != 128) return false;
  if (hd != 32 && hd != 64 && hd != 128 && hd != 256) return false;
  if (d != 16 && d != 32 && d != 64 && d != 128) return false;
  if (x.numel() / c >= (int64_t(1) << 31) || x.size(-2) > 65535) return false;
  if (mask.scalar_type() != at::kBool || mask.device() != x.device() || mask.sizes() != x.sizes().slice(0, x.dim() - 1)) return false;
  const int64_t rows[NPARAMS] = {hd, hd, hd, h, hd, hd, c, c}, cols[NPARAMS] = {c, c, c, c, c, 0, hd, 0};
  for (int i = 0; i < NPARAMS; ++i) {
    const Tensor& t = p[i];
    if (!t.defined()) {
      if (cols[i]) return false;
      continue;
    }
    if (t.scalar_type() != x.scalar_type() || t.device() != x.device() || t.dim() != (cols[i] ? 2 : 1) || t.size(0) != rows[i]) return false;
    if (cols[i] && t.size(1) != cols[i]) return false;
  }
  return true;
}

// What the backward needs of a forward besides its inputs, all dense, in the operator's row order
struct BlockState {
  Tensor q, k, v;  // [h, b, n, n, d]
  Tensor bias;     // [b, n, n, h]
  Tensor g;        // [b, n, n, h d]
  Tensor o;        // [b, h, n, n, d]
  Tensor lse;
  Tensor ws;  // of the operator's forward; undefined without a backward
};

Tensor heads_view(const Tensor& t) { return t.permute({1, 0, 2, 3, 4}); }
Tensor bias_view(const Tensor& t) { return t.permute({0, 3, 1, 2}); }
Tensor mask_view(const Tensor& mask, const BlockShape& s) {
  return swap_pair(mask.dim() == 3 ? mask : mask.reshape({s.b, s.n, s.n}), s.ending);
}

std::pair<Tensor, BlockState> block_forward(const Tensor& x_in, const Tensor& mask, const Params& p, int64_t h, int64_t d, bool ending, bool train = false) {
  const c10::DeviceGuard guard(x_in.device());
  const BlockShape s(x_in, h, d, ending);
  const Tensor x = dense(x_in);
  const auto opt = x.options();
  BlockState st;
  st.q = at::empty({h, s.b, s.n, s.n, d}, opt);
  st.k = at::empty({h, s.b, s.n, s.n, d}, opt);
  st.v = at::empty({h, s.b, s.n, s.n, d}, opt);
  st.bias = at::empty({s.b, s.n, s.n, h}, opt);
  st.g = at::empty({s.b, s.n, s.n, h * d}, opt);
  {
    const Tensor w[5] = {dense(p[WQ]), dense(p[WK]), dense(p[WV]), dense(p[WB]), dense(p[WG])};
    const Tensor bg = p[BG].defined() ? p[BG].contiguous() : Tensor();
    const void* ws[5];
    for (int i = 0; i < 5; ++i) ws[i] = w[i].const_data_ptr();
    const void* bs[5] = {nullptr, nullptr, nullptr, nullptr, bg.defined() ? bg.const_data_ptr() : nullptr};
    void* ys[5] = {st.q.mutable_data_ptr(), st.k.mutable_data_ptr(), st.v.mutable_data_ptr(), st.bias.mutable_data_ptr(), st.g.mutable_data_ptr()};
    const int64_t nout[5] = {h * d, h * d, h * d, h, h * d}, hds[5] = {d, d, d, 0, 0};
    check(trifast_block_in_fwd(x.const_data_ptr(), s.b, s.n, s.c, 5, ws, bs, ys, nout, hds, ending, s.code, stream_of(x)), "trifast_block_in_fwd");
  }
  Forward f = forward(heads_view(st.q), heads_view(st.k), heads_view(st.v), bias_view(st.bias), mask_view(mask, s), train);
  if (train) st.ws = std::move(f.ws);
  st.o = std::move(f.o);
  st.lse = std::move(f.lse);
  Tensor y = at::empty(x.sizes(), opt);
  const Tensor wo = dense(p[WO]), bo = p[BO].defined() ? p[BO].contiguous() : Tensor();
  check(trifast_block_out_fwd(y.mutable_data_ptr(), st.o.const_data_ptr(), st.g.const_data_ptr(), wo.const_data_ptr(), bo.defined() ? bo.const_data_ptr() : nullptr,
                              s.b, h, s.n, d, s.c, ending, s.code, stream_of(x)),
        "trifast_block_out_fwd");
  return {std::move(y), std::move(st)};
}

// dx (undefined unless wanted) and the gradients of the parameters (undefined unless wanted)
std::pair<Tensor, Params> block_backward(const Tensor& dy_lazy, const Tensor& x_in, const Tensor& mask, const Params& p, const BlockState& st, int64_t h,
                                         int64_t d, bool ending, bool want_dx, bool want_dw) {
  const c10::DeviceGuard guard(x_in.device());
  const BlockShape s(x_in, h, d, ending);
  const Tensor dy_in = materialized(dy_lazy), x = dense(x_in), dy = dense(dy_in.scalar_type() == x.scalar_type() ? dy_in : dy_in.to(x.scalar_type()));
  const auto opt = x.options();
  hipStream_t stream = stream_of(x);
  const int64_t rows = s.b * s.n * s.n, hd = h * d;
  Params grads;
  if (want_dw)
    for (int i = 0; i < NPARAMS; ++i)
      if (p[i].defined()) grads[i] = at::empty(p[i].sizes(), opt);
  auto out = [](const Tensor& t) { return t.defined() ? t.mutable_data_ptr() : nullptr; };

  Tensor dout_o = at::empty(st.o.sizes(), opt), dg = at::empty(st.g.sizes(), opt);
  {
    const Tensor wo = dense(p[WO]);
    Tensor ws;
    if (want_dw) ws = workspace(trifast_block_dw_workspace_bytes(rows, hd, 1, &s.c), x);
    check(trifast_block_out_bwd(dout_o.mutable_data_ptr(), dg.mutable_data_ptr(), out(grads[WO]), out(grads[BO]), dy.const_data_ptr(), st.o.const_data_ptr(),
                                st.g.const_data_ptr(), wo.const_data_ptr(), s.b, h, s.n, d, s.c, ending, s.code, out(ws), ws.defined() ? ws.numel() : 0, stream),
          "trifast_block_out_bwd");
  }
  const Tensor bias = bias_view(st.bias);
  Grads a = backward(dout_o, heads_view(st.q), heads_view(st.k), heads_view(st.v), bias, st.o, st.lse, mask_view(mask, s), st.ws);
  Tensor dx;
  if (want_dx) dx = at::empty(x.sizes(), opt);
  if (want_dx || want_dw) {
    const Tensor w[5] = {dense(p[WQ]), dense(p[WK]), dense(p[WV]), dense(p[WB]), dense(p[WG])};
    const void* ws[5];
    for (int i = 0; i < 5; ++i) ws[i] = w[i].const_data_ptr();
    // (the gradients have the memory order of q, k, v and the bias: dense [h, rows, d] and [rows, h])
    const void* dys[5] = {a[0].const_data_ptr(), a[1].const_data_ptr(), a[2].const_data_ptr(), a[3].const_data_ptr(), dg.const_data_ptr()};
    void* dws[5] = {out(grads[WQ]), out(grads[WK]), out(grads[WV]), out(grads[WB]), out(grads[WG])};
    void* dbs[5] = {nullptr, nullptr, nullptr, nullptr, out(grads[BG])};
    const int64_t nout[5] = {hd, hd, hd, h, hd}, hds[5] = {d, d, d, 0, 0};
    Tensor wsp;
    if (want_dw) wsp = workspace(trifast_block_dw_workspace_bytes(rows, s.c, 5, nout), x);
    check(trifast_block_in_bwd(out(dx), want_dw ? dws : nullptr, dbs, x.const_data_ptr(), s.b, s.n, s.c, 5, dys, ws, nout, hds, ending, s.code, out(wsp),
                               wsp.defined() ? wsp.numel() : 0, stream),
          "trifast_block_in_bwd");
  }
  return {std::move(dx), std::move(grads)};
}

struct Block : torch::autograd::Function<Block> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& x, const Tensor& mask, const Tensor& wq, const Tensor& wk, const Tensor& wv,
                        const Tensor& wb, const Tensor& wg, const Tensor& bg, const Tensor& wo, const Tensor& bo, int64_t h, int64_t d, bool ending) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Params p{wq, wk, wv, wb, wg, bg, wo, bo};
    auto [y, st] = block_forward(x, mask, p, h, d, ending, true);
    ctx->save_for_backward({x, mask, wq, wk, wv, wb, wg, bg, wo, bo, st.q, st.k, st.v, st.bias, st.g, st.o, st.lse, st.ws});
    bool want_dw = false;
    for (const Tensor& t : p) want_dw = want_dw || (t.defined() && t.requires_grad());
    ctx->saved_data["shape"] = std::vector<int64_t>{h, d, ending, x.requires_grad(), want_dw};
    ctx->set_materialize_grads(false);
    return y;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    torch::autograd::variable_list out(2 + NPARAMS + 3);
    if (!grads[0].defined()) return out;
    const auto t = ctx->get_saved_variables();
    const auto s = ctx->saved_data["shape"].toIntVector();
    {
      at::AutoDispatchBelowADInplaceOrView below;
      const Params p{t[2], t[3], t[4], t[5], t[6], t[7], t[8], t[9]};
      const BlockState st{t[10], t[11], t[12], t[13], t[14], t[15], t[16], t[17]};
      auto [dx, dp] = block_backward(grads[0], t[0], t[1], p, st, s[0], s[1], s[2] != 0, s[3] != 0, s[4] != 0);
      out[0] = dx;
      for (int i = 0; i < NPARAMS; ++i) out[2 + i] = dp[i];
    }
    return once_differentiable(std::move(out), t, grads[0], "the triangle attention block");
  }
};

using OptTensor = std::optional<Tensor>;
Tensor or_undefined(const OptTensor& t) { return t ? *t : Tensor(); }

// The block on plain tensors; none where the call has to take another path.
OptTensor block(const PyTensor& x_, const PyTensor& mask_, const PyTensor& wq, const PyTensor& wk, const PyTensor& wv, const PyTensor& wb, const PyTensor& wg,
                const std::optional<PyTensor>& bg, const PyTensor& wo, const std::optional<PyTensor>& bo, int64_t h, int64_t d, bool ending) {
  for (const PyTensor* t : {&x_, &mask_, &wq, &wk, &wv, &wb, &wg, &wo})
    if (t->overrides) return std::nullopt;
  if ((bg && bg->overrides) || (bo && bo->overrides)) return std::nullopt;
  const Tensor &x = x_.t, &mask = mask_.t;
  const Params p{wq.t, wk.t, wv.t, wb.t, wg.t, bg ? bg->t : Tensor(), wo.t, bo ? bo->t : Tensor()};
  if (!plain_eager({&x, &mask, &p[WQ], &p[WK], &p[WV], &p[WB], &p[WG], &p[WO]}) || !block_ok(x, mask, p, h, d)) return std::nullopt;
  for (int i : {(int)BG, (int)BO})
    if (p[i].defined() && !plain_eager({&p[i]})) return std::nullopt;
  bool grad = wants_grad({&x, &p[WQ], &p[WK], &p[WV], &p[WB], &p[WG], &p[WO]});
  for (int i : {(int)BG, (int)BO}) grad = grad || (p[i].defined() && wants_grad({&p[i]}));
  if (grad) return Block::apply(x, mask, p[WQ], p[WK], p[WV], p[WB], p[WG], p[BG], p[WO], p[BO], h, d, ending);
  at::AutoDispatchBelowADInplaceOrView below;
  return block_forward(x, mask, p, h, d, ending).first;
}

// ---- the output gate on its own ------------------------------------------------------------

struct GateShape {
  int64_t b, h, n, d;
  explicit GateShape(const Tensor& o) : b(1), h(o.size(-4)), n(o.size(-2)), d(o.size(-1)) {
    for (int64_t x = 0; x + 4 < o.dim(); ++x) b *= o.size(x);
  }
};

Tensor gate_forward(const Tensor& o_in, const Tensor& g_in) {
  const c10::DeviceGuard guard(o_in.device());
  const Tensor o = o_in.contiguous(), g = g_in.contiguous();
  const GateShape s(o);
  Tensor y = at::empty_like(g);
  if (y.numel())
    check(trifast_gate_fwd(y.mutable_data_ptr(), o.const_data_ptr(), g.const_data_ptr(), s.b, s.h, s.n, s.d, dtype_code(o.scalar_type()), stream_of(o)),
          "trifast_gate_fwd");
  return y;
}

std::pair<Tensor, Tensor> gate_backward(const Tensor& dy_in, const Tensor& o_in, const Tensor& g_in) {
  const c10::DeviceGuard guard(o_in.device());
  const Tensor dy = materialized(dy_in).contiguous(), o = o_in.contiguous(), g = g_in.contiguous();
  const GateShape s(o);
  Tensor dout = at::empty_like(o), dg = at::empty_like(g);
  if (dy.numel())
    check(trifast_gate_bwd(dout.mutable_data_ptr(), dg.mutable_data_ptr(), dy.const_data_ptr(), o.const_data_ptr(), g.const_data_ptr(), s.b, s.h, s.n, s.d,
                           dtype_code(o.scalar_type()), stream_of(o)),
          "trifast_gate_bwd");
  return {dout, dg};
}

struct Gate : torch::autograd::Function<Gate> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& o, const Tensor& g) {
    at::AutoDispatchBelowADInplaceOrView below;
    ctx->save_for_backward({o, g});
    return gate_forward(o, g);
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto t = ctx->get_saved_variables();
    torch::autograd::variable_list out(2);
    {
      at::AutoDispatchBelowADInplaceOrView below;
      std::tie(out[0], out[1]) = gate_backward(grads[0], t[0], t[1]);
    }
    return once_differentiable(std::move(out), t, grads[0], "the output gate");
  }
};

// (shapes are the caller's to check)
OptTensor gate(const PyTensor& o_, const PyTensor& g_) {
  if (o_.overrides || g_.overrides) return std::nullopt;
  const Tensor &o = o_.t, &g = g_.t;
  if (!plain_eager({&o, &g})) return std::nullopt;
  if (wants_grad({&o, &g})) return Gate::apply(o, g);
  at::AutoDispatchBelowADInplaceOrView below;
  return gate_forward(o, g);
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  using release = py::call_guard<py::gil_scoped_release>;
  m.def("plain_eager", [](const std::vector<Tensor>& tensors) {
    for (const Tensor& t : tensors)
      if (!plain_eager({&t})) return false;
    return true;
  });
  m.def("attention", &attention, release());
  m.def("forward", [](const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& b, const Tensor& mask) {
    Forward f = forward(q, k, v, b, mask);
    return std::make_tuple(f.o, f.lse);
  }, release());
  m.def("backward", [](const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& b, const Tensor& o, const Tensor& lse, const Tensor& mask) {
    return backward(dout, q, k, v, b, o, lse, mask);
  }, release());
  m.def("block", &block, release());
  m.def("block_ok", [](const Tensor& x, const Tensor& mask, const Tensor& wq, const Tensor& wk, const Tensor& wv, const Tensor& wb, const Tensor& wg,
                       const OptTensor& bg, const Tensor& wo, const OptTensor& bo, int64_t h, int64_t d) {
    return block_ok(x, mask, Params{wq, wk, wv, wb, wg, or_undefined(bg), wo, or_undefined(bo)}, h, d);
  });
  m.def("block_forward", [](const Tensor& x, const Tensor& mask, const std::array<OptTensor, NPARAMS>& params, int64_t h, int64_t d, bool ending) {
    Params p;
    for (int i = 0; i < NPARAMS; ++i) p[i] = or_undefined(params[i]);
    auto [y, st] = block_forward(x, mask, p, h, d, ending);
    return std::make_tuple(y, st.q, st.k, st.v, st.bias, st.g, st.o, st.lse);
  }, release());
  m.def("block_backward", [](const Tensor& dy, const Tensor& x, const Tensor& mask, const std::array<OptTensor, NPARAMS>& params,
                             const std::array<Tensor, 7>& state, int64_t h, int64_t d, bool ending) {
    Params p;
    for (int i = 0; i < NPARAMS; ++i) p[i] = or_undefined(params[i]);
    const BlockState st{state[0], state[1], state[2], state[3], state[4], state[5], state[6], Tensor()};
    auto [dx, dp] = block_backward(dy, x, mask, p, st, h, d, ending, true, true);
    std::vector<Tensor> out{dx};
    for (const Tensor& t : dp)
      if (t.defined()) out.push_back(t);
    return out;
  }, release());
  m.def("gate", &gate, release());
  m.def("gate_forward", &gate_forward, release());
  m.def("gate_backward", &gate_backward, release());
  m.def("set_choosers", [](py::object fwd, py::object bwd) {
    if (!g_choosers) g_choosers = new Choosers;
    *g_choosers = Choosers{std::move(fwd), std::move(bwd)};
  });
  m.def("forget_tiles", [] {
    std::lock_guard<std::mutex> lock(g_tiles_mutex);
    g_tiles.clear();
  });
}
