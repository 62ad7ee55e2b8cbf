// Native host path of the PyTorch entry points: the same calls into the C ABI that attention.py makes
// through ctypes (allocation of the outputs, the argument block, the launch), as C++ on ATen
// tensors, with the autograd node in C++ too.
//
// Why: on a short sequence the kernels take 30-100 us and the host path took longer. A Python autograd
// function's backward runs on the engine's device thread, which must first take the interpreter
// lock from the thread that waits for it; a plain backward here never touches the interpreter. Host
// time per call at N=128, ctypes path against this one: forward and backward 165 -> 77 us (an elementwise
// product's takes 59 on the same host: the rest is the engine's thread), a transformers layer
// without gradients 55 -> 19 us, inference 16 -> 8 us.
//
// Arguments arrive checked (attention.py: _check_inputs, _norm_window, ...). Only what depends on
// this call's tensors is decided here, by attention.py's rules: copies of inputs whose layout the
// ABI cannot address, outputs in the input's layout where it can. Nothing is kept between calls.
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/utils/pybind.h>

#include <optional>

#include "gfa.h"

namespace py = pybind11;
using at::Tensor;

namespace {

// The C ABI of the library that the Python binding has loaded, and its exception type.
struct Api {
  decltype(&gfa_fwd) fwd = nullptr;
  decltype(&gfa_bwd) bwd = nullptr;
  decltype(&gfa_bwd_workspace_bytes) workspace_bytes = nullptr;
  decltype(&gfa_segments_from_positions) positions = nullptr;
  decltype(&gfa_last_error) last_error = nullptr;
  PyObject* error_type = nullptr;  // GfaError(status, message); held for the process
} api;

// A non-zero status as the Python binding raises it. Called with or without the interpreter lock;
// python_error carries the exception through the autograd engine's threads.
void check(int status) {
  if (status == 0) return;
  const std::string message = api.last_error();  // this thread's
  py::gil_scoped_acquire gil;
  PyObject* e = PyObject_CallFunction(api.error_type, "is", status, message.c_str());
  if (e != nullptr) {
    PyErr_SetObject(api.error_type, e);
    Py_DECREF(e);
  }
  python_error err;
  err.persist();
  throw err;
}

constexpr int64_t kSliceLimit = 0xFFFFFFFFll;  // attention.py, _layout_ok
constexpr int64_t kTileOverrun = 128;

bool needs_copy(const Tensor& t) {
  const auto s = t.strides();
  if (s[3] != 1) return true;
  for (int i = 0; i < 3; ++i)
    if (s[i] % 8 != 0 || s[i] < 0) return true;
  if (((t.size(2) - 1 + kTileOverrun) * s[2] + t.size(3)) * t.element_size() > kSliceLimit) return true;
  return reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 != 0;
}
Tensor prep(const Tensor& t) {
  if (t.is_neg()) return prep(t.resolve_neg());  // a view that negates on reading
  return needs_copy(t) ? t.contiguous() : t;
}
// An output with t's layout, or contiguous where the ABI cannot address that layout.
Tensor out_like(const Tensor& t) {
  Tensor o = at::empty_like(t);
  return needs_copy(o) ? at::empty(t.sizes(), t.options()) : o;
}

gfa_strides strides_of(const Tensor& t) { return gfa_strides{t.stride(0), t.stride(1), t.stride(2)}; }
int64_t lse_ld(int64_t n) { return (n + 63) / 64 * 64; }
int dtype_of(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? GFA_DTYPE_BF16 : GFA_DTYPE_FP16; }
void* stream_of(const Tensor& t) {
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

struct Options {
  bool causal;
  int64_t window;
  double scale, softcap, dropout_p;
  int64_t seed, block_kv;
  Tensor lo, hi;       // segment tables, or undefined
  bool as_op = false;  // autograd as the registered op's (Attention)
};

// O, and the LSE where asked for, of prepared inputs. Profilers list it, and the backward below, under
// the registered ops' names.
std::pair<Tensor, Tensor> forward_call(const Tensor& q, const Tensor& k, const Tensor& v, const Options& x,
                                       bool store_lse) {
  RECORD_FUNCTION("gfa::attn_fwd", c10::ArrayRef<const c10::IValue>{});
  const c10::DeviceGuard on_device(q.device());
  Tensor o = out_like(q);
  const int64_t ld = lse_ld(q.size(2));
  Tensor lse;
  if (store_lse) lse = at::empty({q.size(0), q.size(1), ld}, q.options().dtype(at::kFloat));
  gfa_fwd_args a{};
  a.q = q.data_ptr();
  a.k = k.data_ptr();
  a.v = v.data_ptr();
  a.o = o.data_ptr();
  a.lse = store_lse ? static_cast<float*>(lse.data_ptr()) : nullptr;
  a.q_strides = strides_of(q);
  a.k_strides = strides_of(k);
  a.v_strides = strides_of(v);
  a.o_strides = strides_of(o);
  a.batch = (int32_t)q.size(0);
  a.heads_q = (int32_t)q.size(1);
  a.heads_kv = (int32_t)k.size(1);
  a.seq_len = (int32_t)q.size(2);
  a.head_dim = (int32_t)q.size(3);
  a.causal = x.causal;
  a.window = (int32_t)x.window;
  a.scale = (float)x.scale;
  a.dtype = dtype_of(q);
  a.block_kv = (int32_t)x.block_kv;
  a.lse_ld = (int32_t)ld;
  a.softcap = (float)x.softcap;
  a.dropout_p = (float)x.dropout_p;
  a.dropout_seed = (uint64_t)x.seed;
  a.stream = stream_of(q);
  if (x.lo.defined()) {
    a.seg_lo = static_cast<const int32_t*>(x.lo.data_ptr());
    a.seg_hi = static_cast<const int32_t*>(x.hi.data_ptr());
  }
  check(api.fwd(&a));
  return {o, lse};
}

// Whether something stands between the engine and the tensors of a backward that a launch on their
// pointers would pass by: compiled autograd's or a subclass's stand-ins for them, batched
// gradients, zeros without memory, a dispatch mode, a trace.
bool watched(const Tensor& t) {
  using c10::DispatchKey;
  constexpr c10::DispatchKeySet keys({DispatchKey::Python, DispatchKey::Functionalize, DispatchKey::FuncTorchBatched,
                                      DispatchKey::FuncTorchGradWrapper, DispatchKey::Batched, DispatchKey::ZeroTensor});
  return t.key_set().has_any(keys);
}
bool watched(const torch::autograd::variable_list& tensors) {
  using c10::DispatchKey;
  for (const auto key : {DispatchKey::Python, DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::Tracer})
    if (c10::impl::tls_is_dispatch_key_included(key)) return true;
  for (const Tensor& t : tensors)
    if (t.defined() && watched(t)) return true;
  return false;
}

// dQ, dK, dV through the registered op gfa::attn_bwd (ops.py).
std::tuple<Tensor, Tensor, Tensor> backward_op(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                                               const Tensor& lse, const Tensor& dout, const Options& x,
                                               const Tensor& seed) {
  using Maybe = std::optional<Tensor>;
  static const auto op =
      c10::Dispatcher::singleton()
          .findSchemaOrThrow("gfa::attn_bwd", "")
          .typed<std::tuple<Tensor, Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                                                    const Tensor&, const Tensor&, bool, c10::SymInt, double,
                                                    const Maybe&, const Maybe&, double, double, const Maybe&)>();
  const auto maybe = [](const Tensor& t) { return t.defined() ? Maybe(t) : Maybe(); };
  return op.call(q, k, v, o, lse, dout, x.causal, x.window, x.scale, maybe(x.lo), maybe(x.hi), x.softcap, x.dropout_p,
                 maybe(seed));
}

// The autograd node of a call. With as_op (the transformers adapter, which is the registered op
// gfa::attn_fwd everywhere else) a backward that itself records a graph (create_graph) calls the
// op gfa::attn_bwd too: its gradients then refuse to be differentiated again, where the launch
// below would give gradients without a graph and drop the second-order terms. Any watched
// backward calls that op as well, so compiled autograd traces it into its one graph.
struct Attention : public torch::autograd::Function<Attention> {
  static constexpr bool is_traceable = true;

  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                        const Options& x) {
    auto [o, lse] = forward_call(prep(q), prep(k), prep(v), x, true);
    torch::autograd::variable_list saved{q, k, v, o, lse};
    if (x.lo.defined()) saved.insert(saved.end(), {x.lo, x.hi});
    // As the op does, a one-element CPU tensor: a compiled backward takes another seed each time.
    if (x.as_op && x.dropout_p > 0.0) saved.push_back(at::full({1}, x.seed, at::kLong));
    ctx->save_for_backward(std::move(saved));
    ctx->saved_data["whole"] = std::vector<int64_t>{x.causal, x.window, x.seed, x.as_op, x.lo.defined()};
    ctx->saved_data["real"] = std::vector<double>{x.scale, x.softcap, x.dropout_p};
    return o;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 const torch::autograd::variable_list& grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &o = saved[3], &lse = saved[4];
    const auto whole = ctx->saved_data["whole"].toIntVector();
    const auto real = ctx->saved_data["real"].toDoubleVector();
    Options x{whole[0] != 0, whole[1], real[0], real[1], real[2], whole[2]};
    x.as_op = whole[3] != 0;
    if (whole[4] != 0) {
      x.lo = saved[5];
      x.hi = saved[6];
    }
    Tensor seed;
    if (x.dropout_p > 0.0 && x.as_op) seed = saved.back();
    if ((x.as_op && at::GradMode::is_enabled()) || watched(grads) || watched(saved)) {
      if (x.dropout_p > 0.0 && !x.as_op) seed = at::full({1}, x.seed, at::kLong);
      auto [dq, dk, dv] = backward_op(saved[0], saved[1], saved[2], o, lse, grads[0], x, seed);
      return {dq, dk, dv, Tensor()};
    }
    RECORD_FUNCTION("gfa::attn_bwd", c10::ArrayRef<const c10::IValue>{});
    if (seed.defined()) x.seed = seed.item<int64_t>();
    const Tensor q = prep(saved[0]), k = prep(saved[1]), v = prep(saved[2]);
    const c10::DeviceGuard on_device(q.device());
    Tensor dout = prep(grads[0]);
    if (dout.scalar_type() != q.scalar_type()) dout = dout.to(q.scalar_type());
    Tensor dq = out_like(q), dk = out_like(k), dv = out_like(v);
    Tensor delta = at::empty(lse.sizes(), lse.options());
    gfa_bwd_args a{};
    a.q = q.data_ptr();
    a.k = k.data_ptr();
    a.v = v.data_ptr();
    a.o = o.data_ptr();
    a.dout = dout.data_ptr();
    a.lse = static_cast<const float*>(lse.data_ptr());
    a.delta = static_cast<float*>(delta.data_ptr());
    a.dq = dq.data_ptr();
    a.dk = dk.data_ptr();
    a.dv = dv.data_ptr();
    a.q_strides = strides_of(q);
    a.k_strides = strides_of(k);
    a.v_strides = strides_of(v);
    a.o_strides = strides_of(o);
    a.do_strides = strides_of(dout);
    a.dq_strides = strides_of(dq);
    a.dk_strides = strides_of(dk);
    a.dv_strides = strides_of(dv);
    a.batch = (int32_t)q.size(0);
    a.heads_q = (int32_t)q.size(1);
    a.heads_kv = (int32_t)k.size(1);
    a.seq_len = (int32_t)q.size(2);
    a.head_dim = (int32_t)q.size(3);
    a.causal = x.causal;
    a.window = (int32_t)x.window;
    a.scale = (float)x.scale;
    a.dtype = dtype_of(q);
    a.lse_ld = (int32_t)lse.size(2);
    a.softcap = (float)x.softcap;
    a.dropout_p = (float)x.dropout_p;
    a.dropout_seed = (uint64_t)x.seed;
    a.stream = stream_of(q);
    if (x.lo.defined()) {
      a.seg_lo = static_cast<const int32_t*>(x.lo.data_ptr());
      a.seg_hi = static_cast<const int32_t*>(x.hi.data_ptr());
    }
    Tensor ws;
    const size_t need = api.workspace_bytes(&a);
    if (need > 0) {
      ws = at::empty({(int64_t)need}, q.options().dtype(at::kByte));
      a.workspace = ws.data_ptr();
      a.workspace_bytes = need;
    }
    check(api.bwd(&a));
    return {dq, dk, dv, Tensor()};
  }
};

template <typename F>
F pointer(uintptr_t p) {
  return reinterpret_cast<F>(p);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.attr("version") = GFA_VERSION;
  m.def("bind", [](uintptr_t fwd, uintptr_t bwd, uintptr_t workspace_bytes, uintptr_t positions, uintptr_t last_error,
                   py::object error_type) {
    api.fwd = pointer<decltype(api.fwd)>(fwd);
    api.bwd = pointer<decltype(api.bwd)>(bwd);
    api.workspace_bytes = pointer<decltype(api.workspace_bytes)>(workspace_bytes);
    api.positions = pointer<decltype(api.positions)>(positions);
    api.last_error = pointer<decltype(api.last_error)>(last_error);
    api.error_type = error_type.release().ptr();
  });
  // Bodies run without the interpreter lock: an allocation or a launch that waits for the driver does
  // not hold up other Python threads (a data loader's, another stream's).
  const auto or_undefined = [](const std::optional<Tensor>& t) { return t ? *t : Tensor(); };
  // O alone, without autograd.
  m.def("infer", torch::wrap_pybind_function_no_gil(
                     [or_undefined](const Tensor& q, const Tensor& k, const Tensor& v, bool causal, int64_t window,
                                    double scale, double softcap, double dropout_p, int64_t seed, int64_t block_kv,
                                    const std::optional<Tensor>& lo, const std::optional<Tensor>& hi) {
                       const Options x{causal, window, scale, softcap, dropout_p, seed, block_kv,
                                       or_undefined(lo), or_undefined(hi)};
                       return forward_call(prep(q), prep(k), prep(v), x, false).first;
                     }));
  // O with autograd.
  m.def("train", torch::wrap_pybind_function_no_gil(
                     [or_undefined](const Tensor& q, const Tensor& k, const Tensor& v, bool causal, int64_t window,
                                    double scale, double softcap, double dropout_p, int64_t seed,
                                    const std::optional<Tensor>& lo, const std::optional<Tensor>& hi, bool as_op) {
                       const Options x{causal, window, scale, softcap, dropout_p, seed, 0,
                                       or_undefined(lo), or_undefined(hi), as_op};
                       return Attention::apply(q, k, v, x);
                     }));
  // (lo, hi) tables, int32 (batch, seq_len), of unit-stride position ids (rows of stride 0 included).
  m.def("positions", torch::wrap_pybind_function_no_gil([](const Tensor& pos) {
          const c10::DeviceGuard guard(pos.device());
          const Tensor t = at::empty({2, pos.size(0), pos.size(1)}, pos.options().dtype(at::kInt));
          const Tensor lo = t.select(0, 0), hi = t.select(0, 1);
          check(api.positions(pos.data_ptr(), 8 * (int32_t)pos.element_size(), pos.stride(0), (int32_t)pos.size(0),
                              (int32_t)pos.size(1), static_cast<int32_t*>(lo.data_ptr()),
                              static_cast<int32_t*>(hi.data_ptr()), stream_of(pos)));
          return std::make_tuple(lo, hi);
        }));
}
