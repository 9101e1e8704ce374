// Host path of the Python API: what a call does between its arguments and its kernel launches
// (output and workspace allocation, the autograd node, the small results that travel back) in one
// native call. A micro-batch's loss stage or a short lm_head step is bound by this work, not by its
// kernels: the loss stage of 32 Ki tokens with its statistics, forward and backward (16 us of kernels),
// takes 94 us where the same sequence in Python (about twenty tensor calls, ctypes argument lists, a
// Python autograd node) and its kernels took 335.
//
// Loaded as areal_amd._host; every kernel behind it is reached through the C ABI of
// libareal_hip.so (include/areal_hip.h).
#include <torch/extension.h>

#include <torch/csrc/Exceptions.h>
#include <ATen/core/CachingHostAllocator.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <cmath>
#include <initializer_list>
#include <optional>
#include <utility>
#include <vector>

#include "../../include/areal_hip.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

PyObject* error_class = nullptr;  // areal_amd._lib.ArealHipError, set by the binding

// Raises areal_amd._lib.ArealHipError, from any thread (the autograd engine's included).
[[noreturn]] void fail(const std::string& message) {
  py::gil_scoped_acquire gil;
  PyErr_SetString(error_class != nullptr ? error_class : PyExc_RuntimeError, message.c_str());
  python_error e;
  e.persist();
  throw e;
}

void check(int rc, const char* what) {
  if (rc == AREAL_OK) return;
  static const char* const names[] = {"ok", "bad argument", "pointer or leading dimension not suitably aligned",
                                      "workspace too small", "kernel launch failed", "unsupported shape"};
  const std::string name = rc <= 0 && rc >= -5 ? names[-rc] : std::to_string(rc);
  fail(std::string(what) + " failed: " + name + " (code " + std::to_string(rc) + ")");
}

// All given tensors have to live on one HIP device.
template <class... T>
void require_gpu(const T&... ts) {
  const Tensor* first = nullptr;
  auto one = [&](const Tensor& t) {
    if (!t.defined()) return;
    if (!t.is_cuda())
      fail("areal_amd kernels run on an MI355X only; got a tensor on " + t.device().str() +
           " (there is no CPU fallback)");
    if (first == nullptr) first = &t;
    else if (t.device() != first->device())
      fail("tensors on different devices: " + first->device().str() + " and " + t.device().str());
  };
  (one(ts), ...);
  if (first == nullptr) fail("no tensor given");
}

// A kernel reads n elements of every array of a call, whatever an array's own size is.
void require_numel(int64_t n, std::initializer_list<std::pair<const char*, const Tensor*>> arrays) {
  for (const auto& [name, t] : arrays)
    if (t->defined() && t->numel() != n)
      fail(std::string(name) + " has " + std::to_string(t->numel()) + " elements, expected " + std::to_string(n));
}

// Autograd nodes have no forward-mode formula and say so; where a call makes no node (nothing asks for a
// gradient), a tangent would be dropped without a word.
void refuse_tangent(const Tensor& t) {
  TORCH_CHECK_NOT_IMPLEMENTED(!t.defined() || !t._fw_grad(/*level=*/0).defined(),
                              "areal_amd: forward-mode AD is not implemented");
}

Tensor or_undefined(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }

areal_stream_t stream_of(const Tensor& t) {
  return (areal_stream_t)c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

Tensor empty(const Tensor& like, at::IntArrayRef shape, at::ScalarType type) {
  return at::empty(shape, like.options().dtype(type).requires_grad(false));
}
Tensor empty_f32(const Tensor& like, int64_t n) { return empty(like, {n}, at::kFloat); }
Tensor workspace(const Tensor& like, size_t bytes) {
  return empty(like, {(int64_t)(bytes > 0 ? bytes : 1)}, at::kByte);
}

template <class T>
T* ptr(const Tensor& t) { return t.defined() ? (T*)t.data_ptr() : nullptr; }

// Flat fp32 / bool / int64 forms of an argument, as the kernels read it (no copy when it is already one).
Tensor flat(const Tensor& t, at::ScalarType type) {
  if (!t.defined()) return t;
  Tensor d = t.requires_grad() ? t.detach() : t;
  if (d.scalar_type() != type) d = type == at::kBool ? d.to(at::kBool) : d.to(type);
  if (!d.is_contiguous()) d = d.contiguous();
  return d.dim() == 1 ? d : d.view({-1});
}

// ---------------------------------------------------------------------------------------
// Small results on their way to the host: the kernels write them into pinned host memory, which is
// filled with a bit pattern no result has before they are launched. Waiting means looking at that
// memory until the pattern is gone (about a microsecond after the kernel's store, where a copy
// queued behind the kernel, its event and the synchronisation take about 15); after 200 us of that
// the host sleeps instead: until the stream is idle, or, where more may be queued before anyone waits,
// until it has passed the point where mark() was called. A result that nobody waits for keeps its
// memory out of the pinned allocator's hands until the stream has passed the point of its
// destruction. In a captured
// graph, which may be replayed after that memory has gone to someone else, the results stay on the
// device (`results`, the graph's own memory) and whoever asks for them first copies them then; that copy
// is what every later reader gets, whatever has been replayed in between.
// ---------------------------------------------------------------------------------------
constexpr uint64_t PENDING = 0x7ff8a5c3d2e1f0b4ull;  // a NaN payload arithmetic does not make

bool capturing() {
  return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
}

// The allocator of pinned memory gives this one to nobody else before the stream has passed the point at which the last
// tensor of it has gone. False if it does not know the memory.
bool hold_until_passed(const Tensor& pinned, const c10::hip::HIPStream& stream) {
  return at::getHostAllocator(at::kCUDA)->record_event(pinned.data_ptr(), pinned.storage().data_ptr().get_context(),
                                                       c10::hip::HIPStreamMasqueradingAsCUDA(stream).unwrap());
}
// For memory that a queued kernel takes addresses or offsets from: behind the launch, which need not wait for it.
void hold_or_wait(const Tensor& pinned, const c10::hip::HIPStream& stream) {
  bool held = false;
  try {
    held = hold_until_passed(pinned, stream);
  } catch (...) {
  }
  if (!held) stream.synchronize();  // or the next pinned allocation could overwrite what the kernel reads
}
// For results that nobody waited for, in destructors: nothing may be thrown.
void keep_until_passed(const Tensor& pinned, const c10::hip::HIPStream& stream) noexcept {
  try {
    (void)hold_until_passed(pinned, stream);
  } catch (...) {
  }
}

// A point of a stream.
struct Mark {
  hipEvent_t event = nullptr;
  Mark() = default;
  Mark(const Mark&) = delete;
  Mark& operator=(const Mark&) = delete;
  ~Mark() {
    if (event != nullptr) (void)hipEventDestroy(event);
  }
  void set(const c10::hip::HIPStream& stream) {
    const c10::hip::HIPGuard guard(stream.device_index());  // an event belongs to the device it is made on
    if (event == nullptr && hipEventCreateWithFlags(&event, hipEventDisableTiming) != hipSuccess) {
      event = nullptr;
      fail("creation of an event failed");
    }
    if (hipEventRecord(event, stream.stream()) != hipSuccess) fail("recording an event failed");
  }
  void wait(const c10::hip::HIPStream& stream) const {  // without a mark: for all of the stream
    if (event == nullptr) stream.synchronize();
    else if (hipEventSynchronize(event) != hipSuccess) fail("waiting for an event failed");
  }
};

// Which statistics a result holds: (row, key, denominator). Made once per kind of call, so that a call converts no strings.
struct StatRows {
  std::vector<std::tuple<int, py::str, py::str>> rows;
};

struct HostResult {
  Tensor host;    // fp64, pinned
  Tensor device;  // the results of a captured call
  c10::hip::HIPStream stream;
  Mark behind;
  bool done = false;

  explicit HostResult(const Tensor& results) : stream(c10::hip::getCurrentHIPStream(results.device().index())) {
    if (capturing()) {
      device = results;
      return;
    }
    const int64_t n = results.numel();
    host = at::empty({n}, at::TensorOptions().dtype(at::kDouble).pinned_memory(true));
    uint64_t* p = (uint64_t*)host.data_ptr();
    for (int64_t i = 0; i < n; ++i) p[i] = PENDING;
    std::atomic_thread_fence(std::memory_order_release);
  }
  ~HostResult() {
    if (!done && host.defined() && !arrived()) keep_until_passed(host, stream);
  }
  double* data() { return (double*)host.data_ptr(); }
  double* target() { return host.defined() ? data() : nullptr; }  // where kernels write the results
  bool arrived() const {
    const volatile uint64_t* p = (const volatile uint64_t*)host.data_ptr();
    for (int64_t i = host.numel() - 1; i >= 0; --i)
      if (p[i] == PENDING) return false;
    std::atomic_thread_fence(std::memory_order_acquire);
    return true;
  }
  void wait() {
    if (done) return;
    py::gil_scoped_release no_gil;
    if (device.defined()) {
      host = device.cpu();
      done = true;
      return;
    }
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
    while (!arrived()) {
      if (std::chrono::steady_clock::now() > until) {
        behind.wait(stream);
        break;
      }
    }
    done = true;
  }
  void mark() {
    if (!device.defined() && !arrived()) behind.set(stream);
  }
  Tensor value() { wait(); return host; }
  // The counters as Python floats. (As a tensor, each of the few numbers that a call looks at cost an indexing and an
  // item(), one to two microseconds apiece while the GPU stands idle.)
  py::list counters() {
    wait();
    py::list out;
    for (int64_t i = 0; i < std::min<int64_t>(host.numel(), 9); ++i) out.append(py::float_(data()[i]));
    return out;
  }
  // {key: {sum, count, avg, min, max, denominator}} of rows `offset + 4 * row` of the result; avg, min and max
  // are None under an empty denominator.
  void fill(py::dict out, const StatRows& stats, int64_t offset) {
    wait();
    static PyObject *k_sum = PyUnicode_InternFromString("sum"), *k_count = PyUnicode_InternFromString("count"),
                    *k_avg = PyUnicode_InternFromString("avg"), *k_min = PyUnicode_InternFromString("min"),
                    *k_max = PyUnicode_InternFromString("max"),
                    *k_den = PyUnicode_InternFromString("denominator");
    const double* h = data() + offset;
    auto set = [](py::dict& d, PyObject* k, const py::object& v) { PyDict_SetItem(d.ptr(), k, v.ptr()); };
    for (const auto& [row, key, den] : stats.rows) {
      const double* r = h + 4 * row;
      const bool empty = r[1] == 0.0;
      py::dict d;
      set(d, k_sum, py::float_(r[0]));
      set(d, k_count, py::float_(r[1]));
      set(d, k_avg, empty ? py::object(py::none()) : py::object(py::float_(r[0] / r[1])));
      set(d, k_min, empty ? py::object(py::none()) : py::object(py::float_(r[2])));
      set(d, k_max, empty ? py::object(py::none()) : py::object(py::float_(r[3])));
      set(d, k_den, den);
      PyDict_SetItem(out.ptr(), key.ptr(), d.ptr());
    }
  }
};
using HostResultPtr = std::shared_ptr<HostResult>;

// ---------------------------------------------------------------------------------------
// Scalar losses: a kernel has written the loss, d(loss sum)/dx per element and the token counts; the
// node multiplies by upstream / count.
// ---------------------------------------------------------------------------------------
struct LossGraph {
  Tensor loss, dsum, counters;
};

struct ScaledLoss : public torch::autograd::Function<ScaledLoss> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const LossGraph* g) {
    ctx->save_for_backward({g->dsum, g->counters});
    ctx->saved_data["shape"] = x.sizes().vec();
    ctx->saved_data["type"] = (int64_t)x.scalar_type();
    return g->loss;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &dsum = saved[0], &counters = saved[1];
    const c10::hip::HIPGuard guard(dsum.device().index());
    const Tensor up = flat(grads[0], at::kFloat);
    Tensor out = at::empty_like(dsum);
    check(areal_actor_loss_grad(ptr<float>(dsum), ptr<float>(up), ptr<double>(counters), ptr<float>(out),
                                dsum.numel(), stream_of(dsum)),
          "areal_actor_loss_grad");
    out = out.view(ctx->saved_data["shape"].toIntVector());
    const auto type = (at::ScalarType)ctx->saved_data["type"].toInt();
    if (type != at::kFloat) out = out.to(type);
    return {out, Tensor()};
  }
};

Tensor attach(const Tensor& x, const Tensor& loss, const Tensor& dsum, const Tensor& counters) {
  if (!dsum.defined()) return loss;
  const LossGraph g{loss, dsum, counters};
  return ScaledLoss::apply(x, &g);
}
bool wants_grad(const Tensor& x) { return x.requires_grad() && at::GradMode::is_enabled(); }

// ---------------------------------------------------------------------------------------
// PPO / CISPO actor loss (areal_actor_loss_call)
// ---------------------------------------------------------------------------------------
// What a call leaves behind besides the loss: nothing per token, the tensors of the reference's
// `stat` dict, those and the further ones grpo_loss_fn logs, or reduced statistics.
enum { OUT_NONE = 0, OUT_STAT = 1, OUT_LOGGED = 2, OUT_REDUCED = 3 };
constexpr int N_STATS = 18;

areal_loss_config loss_config(const std::array<double, 14>& v) {
  areal_loss_config c;
  c.loss_kind = (int)v[0]; c.clip_lo = (float)v[1]; c.clip_hi = (float)v[2]; c.has_c_clip = (int)v[3];
  c.c_clip = (float)v[4]; c.seq_is = (int)v[5]; c.rs_enabled = (int)v[6]; c.rs_seq_level = (int)v[7];
  c.rs_clamp = (int)v[8]; c.rs_metric = (int)v[9]; c.rs_agg = (int)v[10]; c.rs_upper = (float)v[11];
  c.rs_has_lower = (int)v[12]; c.rs_lower = (float)v[13];
  return c;
}

// (loss, {name: per-token tensor}, host result [9 (+ 18 * 4)]). keep_mask: also return the behave mask
// in the modes that would not.
py::tuple actor_loss(const Tensor& logprobs, const Tensor& proximal, const OptTensor& old_logprobs,
                     const Tensor& advantages, const Tensor& loss_mask, const OptTensor& cu_seqlens,
                     const std::array<double, 14>& config, int mode, bool keep_mask, bool nan_if_nonfinite,
                     const OptTensor& entropy, const OptTensor& extra0, const OptTensor& extra1) {
  refuse_tangent(logprobs);
  const areal_loss_config cfg = loss_config(config);
  const Tensor old_arg = or_undefined(old_logprobs);
  require_numel(loss_mask.numel(), {{"logprobs", &logprobs}, {"proximal_logprobs", &proximal},
                                    {"old_logprobs", &old_arg}, {"advantages", &advantages}});
  require_gpu(proximal, loss_mask, logprobs, old_arg, advantages);
  const c10::hip::HIPGuard guard(proximal.device().index());
  const at::IntArrayRef shape = logprobs.sizes();
  const Tensor lp = flat(logprobs, at::kFloat), prox = flat(proximal, at::kFloat),
               old = flat(old_arg, at::kFloat), adv = flat(advantages, at::kFloat),
               mask = flat(loss_mask, at::kBool);
  const int64_t n = mask.numel();
  const bool seq_is = cfg.loss_kind == 0 && cfg.seq_is, rs = cfg.rs_enabled != 0;
  areal_actor_loss_io io{};
  Tensor cu;
  if ((rs && cfg.rs_seq_level) || seq_is) {
    if (shape.size() == 2) {
      io.n_seqs = shape[0];
      io.uniform_len = shape[1];
    } else {
      cu = or_undefined(cu_seqlens).to(lp.device(), at::kInt).contiguous();
      io.n_seqs = cu.numel() - 1;
    }
  }
  const bool grad = wants_grad(logprobs), stats = mode == OUT_REDUCED;
  const bool stat = mode == OUT_STAT || mode == OUT_LOGGED;
  py::dict out;
  auto f32 = [&](const char* name, bool want) {
    if (!want) return (float*)nullptr;
    const Tensor t = empty(lp, {n}, at::kFloat);
    out[name] = shape.size() == 1 ? t : t.view(shape);
    return ptr<float>(t);
  };
  auto u8 = [&](const char* name, bool want) {
    if (!want) return (uint8_t*)nullptr;
    const Tensor t = empty(lp, {n}, at::kBool);
    out[name] = shape.size() == 1 ? t : t.view(shape);
    return ptr<uint8_t>(t);
  };
  const Tensor ent = flat(or_undefined(entropy), at::kFloat), x0 = flat(or_undefined(extra0), at::kFloat),
               x1 = flat(or_undefined(extra1), at::kFloat);
  if (x0.defined() && x0.numel() != n)
    throw py::value_error("extra statistic has " + std::to_string(x0.numel()) + " elements, expected " + std::to_string(n));
  if (x1.defined() && x1.numel() != n)
    throw py::value_error("extra statistic has " + std::to_string(x1.numel()) + " elements, expected " + std::to_string(n));
  if (ent.defined() && ent.numel() != n)
    throw py::value_error("entropy has " + std::to_string(ent.numel()) + " elements, expected " + std::to_string(n));
  const Tensor loss = empty(lp, {}, at::kFloat);
  const Tensor dlp = grad ? empty(lp, {n}, at::kFloat) : Tensor();
  const int64_t n_results = 9 + (stats ? 4 * N_STATS : 0);
  const Tensor results = empty(lp, {n_results}, at::kDouble);
  auto host = std::make_shared<HostResult>(results);
  io.logprobs = ptr<float>(lp); io.proximal_logprobs = ptr<float>(prox); io.old_logprobs = ptr<float>(old);
  io.advantages = ptr<float>(adv); io.loss_mask = ptr<uint8_t>(mask); io.cu_seqlens = ptr<int32_t>(cu);
  io.entropy = ptr<float>(ent); io.extra0 = ptr<float>(x0); io.extra1 = ptr<float>(x1);
  io.n_tokens = n;
  io.loss = ptr<float>(loss); io.dlogprobs = ptr<float>(dlp);
  io.stat_loss = f32("loss", stat);
  io.stat_ratio = f32("importance_weight", stat);
  io.stat_approx_kl = f32("approx_kl", stat);
  io.clip_mask = u8("clip_mask", stat);
  io.dual_clip_mask = u8("dual_clip_mask", stat);
  // the per-sequence ratio aggregates over what rejection sampling left
  io.new_mask = u8("new_mask", rs && seq_is);
  io.behave_imp_weight = f32("behave_imp_weight", rs && (stat || seq_is));
  io.behave_approx_kl = f32("behave_approx_kl", rs && stat);
  io.behave_mask = u8("behave_mask", rs && (stat || keep_mask));
  const bool logged = mode == OUT_LOGGED;
  io.clip_ratio = f32("clip_ratio", logged);
  io.dual_clip_ratio = f32("dual_clip_ratio", logged);
  io.logp_diff = f32("logp_diff", logged);
  io.logp_abs_diff = f32("logp_abs_diff", logged);
  io.behave_filtered_ratio = f32("behave_filtered_ratio", logged && rs);
  io.results = ptr<double>(results);
  io.host_results = host->target();
  io.with_stats = stats;
  io.nan_if_nonfinite = nan_if_nonfinite;
  const size_t bytes = stats ? areal_actor_loss_stats_workspace_bytes(n, io.n_seqs)
                             : areal_actor_loss_workspace_bytes(n, io.n_seqs);
  const Tensor ws = workspace(lp, bytes);
  check(areal_actor_loss_call(&io, &cfg, ptr<void>(ws), bytes, stream_of(lp)), "areal_actor_loss_call");
  return py::make_tuple(attach(logprobs, loss, dlp, results), out, host);
}

// Tokens whose proximal log-prob is not finite, and its statistics under the mask: a host result [9 + 18 * 4]
// of which entry 8 and row 17 are set (for the losses whose own kernels do not read it).
HostResultPtr proximal_stats(const Tensor& proximal, const Tensor& loss_mask) {
  require_numel(loss_mask.numel(), {{"proximal_logprobs", &proximal}});
  require_gpu(proximal, loss_mask);
  const c10::hip::HIPGuard guard(proximal.device().index());
  const Tensor prox = flat(proximal, at::kFloat), mask = flat(loss_mask, at::kBool);
  areal_loss_config cfg{};
  cfg.loss_kind = -1;
  const Tensor results = empty(prox, {9 + 4 * N_STATS}, at::kDouble);
  auto host = std::make_shared<HostResult>(results);
  areal_actor_loss_io io{};
  io.proximal_logprobs = ptr<float>(prox);
  io.loss_mask = ptr<uint8_t>(mask);
  io.n_tokens = mask.numel();
  io.results = ptr<double>(results);
  io.host_results = host->target();
  io.with_stats = 1;
  const size_t bytes = areal_actor_loss_stats_workspace_bytes(io.n_tokens, 0);
  const Tensor ws = workspace(prox, bytes);
  check(areal_actor_loss_call(&io, &cfg, ptr<void>(ws), bytes, stream_of(prox)), "areal_actor_loss_call");
  return host;
}

// ---------------------------------------------------------------------------------------
// SAPO and critic losses
// ---------------------------------------------------------------------------------------
constexpr int N_SAPO_STATS = 13;

py::tuple sapo_loss(const Tensor& logprobs, const Tensor& old_logprobs, const Tensor& advantages,
                    const Tensor& loss_mask, const OptTensor& cu_seqlens, double tau_pos, double tau_neg,
                    bool seq_level, bool reduced, const OptTensor& entropy, const OptTensor& extra0,
                    const OptTensor& extra1) {
  refuse_tangent(logprobs);
  require_numel(loss_mask.numel(), {{"logprobs", &logprobs}, {"old_logprobs", &old_logprobs}, {"advantages", &advantages}});
  require_gpu(logprobs, old_logprobs, advantages, loss_mask);
  const c10::hip::HIPGuard guard(logprobs.device().index());
  const at::IntArrayRef shape = logprobs.sizes();
  const Tensor lp = flat(logprobs, at::kFloat), old = flat(old_logprobs, at::kFloat),
               adv = flat(advantages, at::kFloat), mask = flat(loss_mask, at::kBool);
  const int64_t n = mask.numel();
  Tensor cu;
  int64_t n_seqs = 0, uniform_len = 0;
  if (seq_level) {
    if (shape.size() == 2) {
      n_seqs = shape[0];
      uniform_len = shape[1];
    } else {
      cu = or_undefined(cu_seqlens).to(lp.device(), at::kInt).contiguous();
      n_seqs = cu.numel() - 1;
    }
  }
  const Tensor ent = flat(or_undefined(entropy), at::kFloat), x0 = flat(or_undefined(extra0), at::kFloat),
               x1 = flat(or_undefined(extra1), at::kFloat);
  for (const Tensor* t : {&x0, &x1, &ent})
    if (t->defined() && t->numel() != n)
      throw py::value_error("a statistic rides along with " + std::to_string(t->numel()) + " elements, expected " +
                            std::to_string(n));
  py::dict out;
  auto f32 = [&](const char* name) {
    if (reduced) return (float*)nullptr;
    const Tensor t = empty(lp, {n}, at::kFloat);
    out[name] = shape.size() == 1 ? t : t.view(shape);
    return ptr<float>(t);
  };
  const Tensor loss = empty(lp, {}, at::kFloat);
  const Tensor dsum = wants_grad(logprobs) ? empty(lp, {n}, at::kFloat) : Tensor();
  const int64_t n_results = 8 + (reduced ? 4 * N_SAPO_STATS : 0);
  const Tensor results = empty(lp, {n_results}, at::kDouble);
  float *stat_loss = f32("loss"), *ratio = f32("importance_weight"), *kl = f32("approx_kl"),
        *gate = f32("sapo_soft_gate"), *gp = f32("sapo_scaled_gate_pos"), *gn = f32("sapo_scaled_gate_neg");
  const size_t bytes = areal_aux_loss_workspace_bytes(n, n_seqs);
  const Tensor ws = workspace(lp, bytes);
  check(areal_sapo_loss(ptr<float>(lp), ptr<float>(old), ptr<float>(adv), ptr<uint8_t>(mask), ptr<int32_t>(cu), n,
                        n_seqs, uniform_len, (float)tau_pos, (float)tau_neg, seq_level, ptr<float>(loss),
                        ptr<float>(dsum), stat_loss, ratio, kl, gate, gp, gn, ptr<double>(results), ptr<float>(ent),
                        ptr<float>(x0), ptr<float>(x1), reduced ? ptr<double>(results) + 8 : nullptr, ptr<void>(ws),
                        bytes, stream_of(lp)),
        "areal_sapo_loss");
  HostResultPtr host;
  if (reduced) {
    host = std::make_shared<HostResult>(results);
    if (host->target() != nullptr &&
        hipMemcpyAsync(host->data(), results.data_ptr(), n_results * sizeof(double), hipMemcpyDeviceToHost,
                       (hipStream_t)stream_of(lp)) != hipSuccess)
      fail("copy of the statistics to the host failed");
  }
  return py::make_tuple(attach(logprobs, loss, dsum, results), out, host);
}

py::tuple critic_loss(const Tensor& value, const Tensor& old_value, const Tensor& target_value,
                      const OptTensor& loss_mask, double eps_clip, bool huber) {
  refuse_tangent(value);
  const Tensor mask_arg = or_undefined(loss_mask);
  require_numel(value.numel(), {{"old_value", &old_value}, {"target_value", &target_value}, {"loss_mask", &mask_arg}});
  require_gpu(value, old_value, target_value, mask_arg);
  const c10::hip::HIPGuard guard(value.device().index());
  const Tensor v = flat(value, at::kFloat), old = flat(old_value, at::kFloat), target = flat(target_value, at::kFloat),
               mask = flat(mask_arg, at::kBool);
  const int64_t n = v.numel();
  const Tensor loss = empty(v, {}, at::kFloat), stat_loss = empty(v, value.sizes(), at::kFloat),
               clip = empty(v, value.sizes(), at::kBool), counters = empty(v, {8}, at::kDouble);
  const Tensor dsum = wants_grad(value) ? empty(v, {n}, at::kFloat) : Tensor();
  const size_t bytes = areal_aux_loss_workspace_bytes(n, 0);
  const Tensor ws = workspace(v, bytes);
  check(areal_critic_loss(ptr<float>(v), ptr<float>(old), ptr<float>(target), ptr<uint8_t>(mask), n, (float)eps_clip,
                          huber, ptr<float>(loss), ptr<float>(dsum), ptr<float>(stat_loss), ptr<uint8_t>(clip),
                          ptr<double>(counters), ptr<void>(ws), bytes, stream_of(v)),
        "areal_critic_loss");
  return py::make_tuple(attach(value, loss, dsum, counters), clip, stat_loss);
}

// ---------------------------------------------------------------------------------------
// Fused lm_head (areal_amd/functional/lm_head.py says what the modes are)
// ---------------------------------------------------------------------------------------
int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// Largest token chunk (multiple of 256) whose backward workspace fits `budget`: bf16 dlogits of the chunk
// plus the transposed weight (and, when T is not a multiple of 64, transposed copies of the last chunk's
// hidden states and dlogits).
int64_t default_token_chunk(int64_t T, int64_t H, int64_t V, int64_t budget) {
  const bool ragged = T % 64 != 0;
  const int64_t per_token = 2 * V + 64 + (ragged ? 2 * (V + H) : 0), fixed = 2 * H * (V + 64);
  const int64_t room = budget - fixed;
  int64_t chunk = room > 0 ? room / per_token : 0;
  chunk = std::max<int64_t>(chunk, 256) / 256 * 256;
  return std::min(std::max<int64_t>(chunk, 256), std::max<int64_t>(T, 1));
}

// Whether `bytes` fit 60 % of the device memory the allocator can still hand out: free on the device
// plus what the caching allocator holds but has not given to a tensor. The device is only asked when
// the latter alone does not settle it.
bool fits_memory(int64_t bytes, int device) {
  const auto stats = c10::hip::HIPCachingAllocator::getDeviceStats(device);
  const size_t all = (size_t)c10::CachingAllocator::StatType::AGGREGATE;
  const int64_t held = stats.reserved_bytes[all].current - stats.allocated_bytes[all].current;
  if ((double)bytes <= 0.6 * (double)held) return true;
  size_t free = 0, total = 0;
  if (hipMemGetInfo(&free, &total) != hipSuccess) return false;
  return (double)bytes <= 0.6 * (double)(held + (int64_t)free);
}

struct LMHeadArgs {
  double temperature, logit_scale;
  int64_t token_chunk;  // 0: the default
  int save_probs;       // -1: decide by size
  bool with_moments;
  Tensor accum;         // fp32 accumulator of the weight gradient
  Tensor owner;         // fp32 parameter whose .grad is that accumulator, see LMHeadState
  int64_t save_limit, bwd_budget;
  bool logprobs_only = false;  // no other output (and no backward)
};

// An int that the device makes (`flag`), on its way to the host: in pinned memory, -1 until it has been
// written there. Of a captured call it stays on the device, as HostResult's, and is read anew each time.
struct Status {
  Tensor host, device;
  c10::hip::HIPStream stream;
  Mark behind;
  explicit Status(const Tensor& flag) : stream(c10::hip::getCurrentHIPStream(flag.device().index())) {
    if (capturing()) {
      device = flag;
      return;
    }
    host = at::empty({1}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    *(volatile int*)host.data_ptr() = -1;
    std::atomic_thread_fence(std::memory_order_release);
  }
  ~Status() {
    if (host.defined() && !known()) keep_until_passed(host, stream);
  }
  int* target() const { return host.defined() ? (int*)host.data_ptr() : nullptr; }  // where kernels write it
  int read() const { return *(volatile int*)host.data_ptr(); }
  bool known() const { return host.defined() && read() >= 0; }
  int wait() {
    if (known()) return read();
    py::gil_scoped_release no_gil;
    if (device.defined()) return device.cpu().item<int>();
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
    while (read() < 0)
      if (std::chrono::steady_clock::now() > until) {
        behind.wait(stream);
        break;
      }
    return read();
  }
  void mark() {
    if (host.defined() && !known()) behind.set(stream);
  }
};

// State of one forward for its backward. The exponentials are consumed by the first backward (it
// rewrites entries of them in place); a second one recomputes.
// owner: the fp32 master of `weight`. Its .grad is looked up when the backward runs: an existing one is
// added to by the contraction (behind it, if its strides are not the kernels'), a missing one is
// allocated and stored to (not cleared first and then read back: 3 x 4 bytes per weight less).
struct LMHeadState {
  Tensor probs, probs_ref, probs_status, label_logprobs, bias, accum, owner;
  std::shared_ptr<Status> status;
  double temperature = 1.0, logit_scale = 1.0;
  int64_t token_chunk = 0, bwd_budget = 0;
  std::vector<int64_t> hidden_shape;
  at::ScalarType weight_type = at::kBFloat16, bias_type = at::kFloat;
};

variable_list lm_head_forward(const Tensor& hidden, const Tensor& weight, const Tensor& bias, const Tensor& labels,
                              const LMHeadArgs& a, bool needs_grad, std::shared_ptr<LMHeadState>* state,
                              variable_list* saved) {
  const int64_t H = hidden.size(-1), V = weight.size(0);
  const Tensor h2 = (hidden.dim() == 2 ? hidden : hidden.reshape({-1, H})).contiguous(), w = weight.contiguous();
  const Tensor lab = flat(labels, at::kLong);
  const Tensor bias_f = bias.defined() ? bias.detach().to(at::kFloat).contiguous() : Tensor();
  const int64_t T = h2.size(0);
  variable_list outs(6);
  for (int i = 0; i < (a.logprobs_only ? 1 : a.with_moments ? 6 : 4); ++i) outs[i] = empty(h2, labels.sizes(), at::kFloat);
  const int64_t need = 2 * round_up(T, 128) * round_up(V, 64);
  const bool save = needs_grad && T > 0 &&
                    (a.save_probs >= 0 ? a.save_probs != 0
                                       : need <= a.save_limit && fits_memory(need, h2.device().index()));
  // row_max, sum_exp [T] (and the copy of the log-probabilities and the row references) in one allocation
  const int64_t Tp = round_up(T, 64);
  Tensor rows, row_max, sum_exp;
  if (!a.logprobs_only) {
    rows = empty_f32(h2, Tp * (save ? 4 : 2));
    row_max = rows.narrow(0, 0, T);
    sum_exp = rows.narrow(0, Tp, T);
  }
  Tensor probs, probs_ref, probs_status, lp_copy;
  std::shared_ptr<Status> status;
  if (save) {
    probs = empty(h2, {round_up(T, 128), round_up(V, 64)}, at::kBFloat16);
    lp_copy = rows.narrow(0, 2 * Tp, T);
    probs_ref = rows.narrow(0, 3 * Tp, T);
    probs_status = empty(h2, {1}, at::kInt);
    status = std::make_shared<Status>(probs_status);
  }
  if (T > 0) {
    const size_t bytes = areal_lmhead_fwd_workspace_bytes(T, H, V);
    const Tensor ws = workspace(h2, bytes);
    check(areal_lmhead_fwd_ex(ptr<void>(h2), ptr<void>(w), ptr<float>(bias_f), ptr<int64_t>(lab), T, H, V,
                              (float)(1.0 / a.temperature), (float)a.logit_scale, ptr<float>(outs[0]),
                              ptr<float>(outs[1]), ptr<float>(outs[2]), ptr<float>(outs[3]), ptr<float>(outs[4]),
                              ptr<float>(outs[5]), ptr<float>(row_max), ptr<float>(sum_exp), ptr<void>(probs),
                              save ? (size_t)need : 0, ptr<float>(probs_ref), ptr<int>(probs_status),
                              ptr<float>(lp_copy), save ? status->target() : nullptr, ptr<void>(ws), bytes,
                              stream_of(h2)),
          "areal_lmhead_fwd");
  }
  if (state != nullptr) {
    auto st = std::make_shared<LMHeadState>();
    st->probs = probs; st->probs_ref = probs_ref; st->probs_status = probs_status; st->label_logprobs = lp_copy;
    st->bias = bias_f; st->accum = a.accum; st->owner = a.owner; st->status = status;
    st->temperature = a.temperature; st->logit_scale = a.logit_scale; st->token_chunk = a.token_chunk;
    st->bwd_budget = a.bwd_budget;
    st->hidden_shape = hidden.sizes().vec();
    st->weight_type = weight.scalar_type();
    if (bias.defined()) st->bias_type = bias.scalar_type();
    *state = st;
    *saved = {h2, w, lab, row_max, sum_exp};
  }
  return outs;
}

// (dHidden, dWeight, dBias), each absent when it is not wanted. want_*: whose gradient autograd asks for.
std::vector<OptTensor> lm_head_backward(const std::shared_ptr<LMHeadState>& st, const variable_list& saved,
                                        const Tensor& grad, bool want_h, bool want_w, bool need_b) {
  bool need_h = want_h, need_w = want_w;
  // dWeight goes straight into the caller's fp32 accumulator when one was given: the contraction's
  // epilogue adds to it and no gradient is returned for the weight
  Tensor accum = st->accum;
  bool add = accum.defined();
  Tensor strided;  // a .grad of the owner that the kernels cannot write to: theirs is added to it at the end
  if (st->owner.defined()) {
    accum = st->owner.grad();
    if (accum.defined() && !(accum.layout() == at::kStrided && accum.scalar_type() == at::kFloat &&
                             accum.device() == saved[1].device() && accum.sizes() == saved[1].sizes() &&
                             accum.is_contiguous()))
      std::swap(strided, accum);
    add = accum.defined();
  }
  if (add || st->owner.defined()) need_w = true;
  std::vector<OptTensor> none(3);
  if (!(need_h || need_w || need_b)) return none;
  const Tensor &h2 = saved[0], &w = saved[1], &lab = saved[2], &row_max = saved[3], &sum_exp = saved[4];
  const c10::hip::HIPGuard guard(h2.device().index());
  const int64_t T = h2.size(0), H = h2.size(1), V = w.size(0);
  if (st->probs.defined()) {
    if (!st->status->known() && capturing())
      fail("this lm_head backward reads a result of its forward on the host and cannot be captured: use save_probs=False");
    st->status->mark();  // what is queued below is not to be waited for
  }
  const Tensor g = flat(grad, at::kFloat);
  // the kernels need one of dHidden / dWeight as an output; a bias-only request computes dHidden
  need_h = need_h || (need_b && !need_w);
  const Tensor dh = need_h ? at::empty_like(h2) : Tensor();
  if (st->owner.defined() && !add) accum = empty(h2, {V, H}, at::kFloat);
  // (the kernels add to the bias gradient as well when they add to the weight's)
  const Tensor db32 = need_b ? (add ? at::zeros({V}, h2.options().dtype(at::kFloat)) : empty_f32(h2, V)) : Tensor();
  Tensor probs = st->probs;
  const Tensor probs_ref = st->probs_ref;
  const float inv_t = (float)(1.0 / st->temperature), scale = (float)st->logit_scale;
  // A contraction over the whole batch can store dWeight in bf16 itself: the saved mode always, the
  // recompute mode when one token chunk covers the batch. Several chunks accumulate in fp32 and cast.
  const int64_t chunk = T > 0 ? (st->token_chunk > 0 ? st->token_chunk
                                                     : default_token_chunk(T, H, V, st->bwd_budget))
                              : 1;
  const bool bf16_out = !accum.defined() && T > 0 && st->weight_type == at::kBFloat16;
  bool direct = bf16_out && (probs.defined() || chunk >= T);
  Tensor dw_direct = need_w && direct ? empty(h2, {V, H}, at::kBFloat16) : Tensor();
  Tensor dw32 = accum;
  if (!accum.defined() && need_w && !direct) dw32 = empty(h2, {V, H}, at::kFloat);
  const Tensor probs_status = st->probs_status, label_logprobs = st->label_logprobs;
  st->probs = st->probs_ref = st->probs_status = Tensor();
  bool recompute = !probs.defined();
  const int mode = add ? 1 : 0;
  if (T == 0) {
    recompute = false;
    if (dw32.defined() && !add) dw32.zero_();
    if (db32.defined()) db32.zero_();
  } else if (probs.defined()) {
    // Queued before the host knows whether every row's saved exponentials were in range: the kernels
    // read that status on the device and return at once if it is set.
    const size_t bytes = areal_lmhead_bwd_saved_workspace_bytes(T, H, V);
    const Tensor ws = workspace(h2, bytes);
    check(areal_lmhead_bwd_saved(ptr<void>(h2), ptr<void>(w), ptr<int64_t>(lab), ptr<float>(row_max),
                                 ptr<float>(sum_exp), ptr<float>(label_logprobs), ptr<float>(g), T, H, V, inv_t, scale,
                                 ptr<void>(probs), (size_t)probs.numel() * 2, ptr<float>(probs_ref),
                                 ptr<int>(probs_status), ptr<void>(dh),
                                 need_w ? ptr<void>(direct ? dw_direct : dw32) : nullptr, direct ? 2 : mode,
                                 ptr<float>(db32), ptr<void>(ws), bytes, stream_of(h2)),
          "areal_lmhead_bwd_saved");
    // The status travelled to pinned memory with the forward's last kernel. Looking at it now, with the
    // launches above already queued, idles nothing, and waits for the forward (and what was queued up to
    // this call) alone; if it was set (a row's maximum far above its estimate) those launches did nothing
    // and the recompute mode runs.
    if (st->status->wait() != 0) {
      recompute = true;
      probs = Tensor();  // (up to 40 GiB, the recompute's workspace up to 24: not both at a time)
      if (need_w && direct && chunk < T) {
        direct = false;
        dw_direct = Tensor();
        dw32 = empty(h2, {V, H}, at::kFloat);
      }
    }
  }
  if (recompute) {
    const size_t bytes = areal_lmhead_bwd_workspace_bytes(T, H, V, chunk);
    const Tensor ws = workspace(h2, bytes);
    check(areal_lmhead_bwd(ptr<void>(h2), ptr<void>(w), ptr<float>(st->bias), ptr<int64_t>(lab), ptr<float>(row_max),
                           ptr<float>(sum_exp), ptr<float>(g), T, H, V, inv_t, scale, ptr<void>(dh),
                           need_w ? ptr<void>(direct ? dw_direct : dw32) : nullptr, ptr<float>(db32),
                           direct ? 2 : mode, chunk, ptr<void>(ws), bytes, stream_of(h2)),
          "areal_lmhead_bwd");
  }
  Tensor dw = dw_direct;
  if (dw32.defined() && !accum.defined()) {
    if (st->weight_type == at::kFloat) {
      dw = dw32;
    } else {
      dw = empty(h2, {V, H}, st->weight_type);
      check(areal_cast_f32_to_bf16(ptr<float>(dw32), ptr<void>(dw), dw32.numel(), stream_of(h2)),
            "areal_cast_f32_to_bf16");
    }
  }
  // with every launch queued: an error above leaves the owner's .grad as it was
  if (strided.defined()) {
    const at::NoGradGuard no_grad;
    strided.add_(accum);
  } else if (st->owner.defined() && !add) {
    st->owner.mutable_grad() = accum;
  }
  if (want_h) none[0] = dh.view(st->hidden_shape);
  if (dw.defined()) none[1] = dw;
  if (db32.defined()) none[2] = db32.to(st->bias_type);
  return none;
}

// (six per-token outputs, tensors to save, state); without needs_grad only the outputs.
py::tuple lm_head(const Tensor& hidden, const Tensor& weight, const OptTensor& bias_arg, const Tensor& labels,
                  double temperature, double logit_scale, int64_t token_chunk, int save_probs, bool with_moments,
                  const OptTensor& accum, const OptTensor& owner, int64_t save_limit, int64_t bwd_budget,
                  bool build_graph, bool needs_grad, bool logprobs_only) {
  const Tensor bias = or_undefined(bias_arg);
  for (const Tensor* t : {&hidden, &weight, &bias}) refuse_tangent(*t);
  require_gpu(hidden, weight, labels, bias);
  const c10::hip::HIPGuard guard(hidden.device().index());
  const LMHeadArgs a{temperature, logit_scale, token_chunk, save_probs, with_moments, or_undefined(accum),
                     or_undefined(owner), save_limit, bwd_budget, logprobs_only && !needs_grad && !build_graph};
  std::shared_ptr<LMHeadState> state;
  variable_list saved;
  const variable_list outs = lm_head_forward(hidden, weight, bias, labels, a, needs_grad,
                                             build_graph ? &state : nullptr, &saved);
  py::tuple r(6);
  for (int i = 0; i < 6; ++i) r[i] = outs[i].defined() ? py::cast(outs[i]) : py::none();
  return build_graph ? py::make_tuple(r, saved, state) : r;
}

// ---------------------------------------------------------------------------------------
// Logits-in path
// ---------------------------------------------------------------------------------------
struct Logits : public torch::autograd::Function<Logits> {
  static variable_list forward(AutogradContext* ctx, const Tensor& logits, const Tensor& labels, double temperature,
                               bool with_entropy, bool needs_grad) {
    const int64_t V = logits.size(-1);
    Tensor rows = logits.scalar_type() == at::kFloat || logits.scalar_type() == at::kBFloat16 ? logits
                                                                                            : logits.to(at::kFloat);
    rows = rows.dim() == 2 ? rows : rows.reshape({-1, V});
    if (rows.stride(-1) != 1 || (rows.size(0) > 1 && rows.stride(0) < V)) rows = rows.contiguous();
    const int64_t T = rows.size(0);
    const Tensor lab = flat(labels, at::kLong);
    const Tensor lp = empty(rows, labels.sizes(), at::kFloat);
    const Tensor ent = with_entropy ? empty(rows, labels.sizes(), at::kFloat) : Tensor();
    const Tensor lse2 = needs_grad ? empty_f32(rows, T) : Tensor();
    check(areal_logits_logprobs_entropy_fwd(ptr<void>(rows), rows.scalar_type() == at::kBFloat16 ? 1 : 0,
                                            T > 1 ? rows.stride(0) : V, ptr<int64_t>(lab), T, V,
                                            (float)(1.0 / temperature), ptr<float>(lp), ptr<float>(ent),
                                            ptr<float>(lse2), stream_of(rows)),
          "areal_logits_logprobs_entropy_fwd");
    ctx->save_for_backward({rows, lab, lse2, ent});
    ctx->saved_data["temperature"] = temperature;
    ctx->saved_data["shape"] = logits.sizes().vec();
    ctx->saved_data["type"] = (int64_t)logits.scalar_type();
    ctx->set_materialize_grads(false);
    if (with_entropy) return {lp, ent};
    return {lp};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list r(5);
    const Tensor glp_arg = grads[0], gen_arg = grads.size() > 1 ? grads[1] : Tensor();
    if (!glp_arg.defined() && !gen_arg.defined()) return r;
    const auto saved = ctx->get_saved_variables();
    const Tensor &rows = saved[0], &lab = saved[1], &lse2 = saved[2], &ent = saved[3];
    const c10::hip::HIPGuard guard(rows.device().index());
    const int64_t T = rows.size(0), V = rows.size(1);
    const Tensor glp = flat(glp_arg, at::kFloat), gen = flat(gen_arg, at::kFloat);
    Tensor d = empty(rows, {T, V}, rows.scalar_type());
    check(areal_logits_logprobs_entropy_bwd(ptr<void>(rows), rows.scalar_type() == at::kBFloat16 ? 1 : 0,
                                            T > 1 ? rows.stride(0) : V, ptr<int64_t>(lab), T, V,
                                            (float)(1.0 / ctx->saved_data["temperature"].toDouble()), ptr<float>(lse2),
                                            ptr<float>(ent), ptr<float>(glp), ptr<float>(gen), ptr<void>(d), V,
                                            stream_of(rows)),
          "areal_logits_logprobs_entropy_bwd");
    d = d.view(ctx->saved_data["shape"].toIntVector());
    const auto type = (at::ScalarType)ctx->saved_data["type"].toInt();
    r[0] = d.scalar_type() == type ? d : d.to(type);
    return r;
  }
};

variable_list logits_logprobs(const Tensor& logits, const Tensor& labels, double temperature, bool with_entropy) {
  require_gpu(logits, labels);
  const c10::hip::HIPGuard guard(logits.device().index());
  return Logits::apply(logits, labels, temperature, with_entropy, wants_grad(logits));
}

// ---------------------------------------------------------------------------------------
// Advantages
// ---------------------------------------------------------------------------------------
// What a group normalisation needs besides its data: (group offsets [G + 1], rows per group [G], longest
// group, tail group, mean level, deviation level, leave one out, unbiased, eps).
using NormTables = std::tuple<Tensor, Tensor, int64_t, int, int, int, int, int, double>;

Tensor bytes_of(const Tensor& t, int64_t bs, int64_t L) {  // a mask as [bs, L] bytes
  Tensor r = t.scalar_type() == at::kBool ? t : t.ne(0);
  if (r.dim() != 2 || r.size(0) != bs || r.size(1) != L) r = r.reshape({bs, L});
  return r.contiguous();
}
bool in_place_ok(const Tensor& t) { return t.scalar_type() == at::kFloat && t.is_contiguous() && !t.requires_grad(); }

Tensor f32(const Tensor& t) {
  if (!t.defined()) return t;
  return (t.scalar_type() == at::kFloat ? t : t.to(at::kFloat)).contiguous();
}

// Reward scores and their normalisation, then areal_advantage_prep, over bs rows. `score`: the scores themselves when
// `scored`, else the raw rewards. Returns (loss mask, old log-probs, kl rewards, total rewards, kl rewards
// for GAE, outcome rewards (both turn mode only), no-eos mask, and with `gae` = (values, discount, lambda, normalisation
// of the advantages) where one launch does it all: advantages, returns and their row sums, or no sums where
// the advantages came out normalised).
using GaeOptions = std::tuple<OptTensor, double, double, std::optional<NormTables>>;
py::tuple advantage_prep(const Tensor& score, bool scored, double bias, double scaling, double clip,
                         const std::optional<NormTables>& norm, const Tensor& loss_mask, const Tensor& attention_mask,
                         const Tensor& logp_src, const OptTensor& ref_logp, bool recompute, int estimator, bool clamp,
                         bool no_eos_zero, double kl_ctl, bool turn_mode, int64_t bs,
                         const std::optional<GaeOptions>& gae) {
  const int64_t L = logp_src.size(-1);
  const Tensor ref_arg = or_undefined(ref_logp);
  require_numel(bs, {{"rewards", &score}});
  require_numel(bs * L, {{"logprobs", &logp_src}, {"loss_mask", &loss_mask}, {"attention_mask", &attention_mask},
                         {"ref_logp", &ref_arg}});
  require_gpu(logp_src, loss_mask, attention_mask, score, ref_arg);
  const c10::hip::HIPGuard guard(logp_src.device().index());
  const areal_stream_t stream = stream_of(logp_src);
  Tensor sc = score.scalar_type() == at::kFloat ? score : score.to(at::kFloat);
  sc = sc.contiguous();
  Tensor logp = logp_src.requires_grad() ? logp_src.detach() : logp_src;
  const bool src_ok = in_place_ok(logp_src);
  if (logp.dim() != 2) logp = logp.reshape({bs, L});
  if (!in_place_ok(logp)) logp = logp.to(at::kFloat).contiguous();
  const Tensor old = recompute && src_ok ? logp : empty(logp, {bs, L}, at::kFloat);
  Tensor ref = ref_arg;
  const bool ref_in_place = ref.defined() && in_place_ok(ref);
  if (ref.defined()) ref = ref_in_place ? ref.reshape({bs, L}) : ref.detach().to(at::kFloat).contiguous().reshape({bs, L});
  const Tensor lm = empty(logp, {bs, L}, at::kFloat), kl = empty(logp, {bs, L}, at::kFloat),
               tot = empty(logp, {bs, L}, at::kFloat);
  const Tensor seqlens = empty(logp, {bs}, at::kLong), no_eos = empty(logp, {bs}, at::kBool);
  const Tensor lmb = bytes_of(loss_mask, bs, L), amb = bytes_of(attention_mask, bs, L);
  auto opt = [](const Tensor& t) { return t.defined() ? OptTensor(t) : OptTensor(); };
  auto norm_args = [&](auto&& call) {
    if (!norm.has_value()) return call(nullptr, nullptr, 0, -1, 0, 0, 0, 0.0);
    const auto& [off, rows, longest, tail, mean_level, std_level, loo, unbiased, eps] = *norm;
    return call(ptr<int64_t>(off), ptr<int64_t>(rows), rows.numel(), tail, mean_level, std_level, unbiased, eps);
  };
  auto shape_scores = [&] {
    const Tensor shaped = empty_f32(sc, bs);
    check(norm_args([&](const int64_t* off, const int64_t* rows, int64_t n, int tail, int mean_level, int std_level,
                        int unbiased, double eps) {
            return areal_reward_scores(ptr<float>(sc), bs, (float)bias, (float)scaling, (float)clip, off, rows, n, tail,
                                       mean_level, std_level, unbiased, eps, ptr<float>(shaped), stream);
          }),
          "areal_reward_scores");
    sc = shaped;
    scored = true;
  };
  // (a score that is not one per row, or values of another size, are for the calls that look at them)
  if (gae.has_value() && !turn_mode && bs > 0 && L > 0) {
    const Tensor v = f32(or_undefined(std::get<0>(*gae)));
    if (!v.defined() || (v.device() == lm.device() && v.sizes() == lm.sizes())) {
      const Tensor adv = at::empty_like(lm), ret = at::empty_like(lm);
      Tensor sums;
      auto launch = [&](auto entry, auto... behind) {
        return norm_args([&](const int64_t* off, const int64_t* rows, int64_t n, int tail, int mean_level,
                             int std_level, int unbiased, double eps) {
          return entry(ptr<float>(sc), scored ? 0 : norm.has_value() ? 2 : 1, (float)bias, (float)scaling, (float)clip,
                       off, rows, n, tail, mean_level, std_level, unbiased, eps, ptr<uint8_t>(lmb), ptr<uint8_t>(amb),
                       ptr<float>(logp), ptr<float>(ref), ptr<float>(v), bs, L, recompute ? 0 : 1, estimator, clamp,
                       no_eos_zero, ref_in_place, (float)kl_ctl, (float)std::get<1>(*gae), (float)std::get<2>(*gae),
                       ptr<float>(lm), ptr<float>(old), ptr<float>(kl), ptr<float>(tot), ptr<int64_t>(seqlens),
                       ptr<uint8_t>(no_eos), ptr<float>(adv), ptr<float>(ret), behind..., stream);
        });
      };
      auto one_launch = [&] {
        const auto& adv_norm = std::get<3>(*gae);
        if (adv_norm.has_value()) {
          const auto& [off, rows, longest, tail, mean_level, std_level, loo, unbiased, eps] = *adv_norm;
          const areal_group_norm_spec spec{ptr<int64_t>(off), rows.numel(), longest / L, tail, mean_level, std_level,
                                           loo, unbiased, -1, eps};
          const size_t bytes = areal_advantages_normalized_workspace_bytes(bs);
          const Tensor ws = workspace(lm, bytes);
          const int rc = launch(areal_advantages_normalized, &spec, ptr<void>(ws), bytes);
          if (rc != AREAL_ERR_UNSUPPORTED) return rc;
        }
        sums = empty(lm, {5, bs}, at::kDouble);
        const int rc = launch(areal_advantages_row_stats, ptr<double>(sums));
        if (rc != AREAL_OK) sums = Tensor();
        return rc;
      };
      int rc = one_launch();
      if (rc == AREAL_ERR_UNSUPPORTED && !scored) {  // it may take the scores ready-made
        shape_scores();
        rc = one_launch();
      }
      if (rc != AREAL_ERR_UNSUPPORTED) {
        check(rc, "areal_advantages_row_stats");
        return py::make_tuple(lm, old.view(logp_src.sizes()), kl, tot, OptTensor(), OptTensor(), no_eos,
                              py::make_tuple(adv, ret, opt(sums)));
      }
    }
  }
  if (!scored) shape_scores();
  const Tensor gkl = turn_mode ? empty(logp, {bs, L}, at::kFloat) : Tensor(),
               outcome = turn_mode ? empty(logp, {bs, L}, at::kFloat) : Tensor();
  check(areal_advantage_prep(ptr<uint8_t>(lmb), ptr<uint8_t>(amb), ptr<float>(logp), ptr<float>(ref), ptr<float>(sc), bs,
                             L, recompute ? 0 : 1, estimator, clamp, no_eos_zero, ref_in_place, (float)kl_ctl,
                             ptr<float>(lm), ptr<float>(old), ptr<float>(kl), ptr<float>(gkl), ptr<float>(outcome),
                             ptr<float>(tot), ptr<int64_t>(seqlens), ptr<uint8_t>(no_eos), stream),
        "areal_advantage_prep");
  return py::make_tuple(lm, old.view(logp_src.sizes()), kl, tot, opt(gkl), opt(outcome), no_eos, py::none());
}

// Token-level GAE of padded rows that leaves each row's masked sums: (advantages, returns, sums [5, bs]), or
// nothing when the layout is not one for it.
std::optional<std::tuple<Tensor, Tensor, Tensor>> gae_row_stats(const Tensor& rewards, const OptTensor& values,
                                                                const Tensor& loss_mask, const Tensor& no_eos,
                                                                double discount, double lambda,
                                                                const OptTensor& lambda_seq) {
  const Tensor v = f32(or_undefined(values)), lam = or_undefined(lambda_seq);
  require_gpu(rewards, v, loss_mask, no_eos, lam);
  const c10::hip::HIPGuard guard(rewards.device().index());
  const int64_t bs = rewards.size(0), L = rewards.size(1);
  const Tensor r = f32(rewards), m = f32(loss_mask), ne = no_eos.to(at::kBool).contiguous();
  const Tensor adv = at::empty_like(r), ret = at::empty_like(r), sums = empty(r, {5, bs}, at::kDouble);
  const int rc = areal_gae_padded_row_stats(ptr<float>(r), ptr<float>(v), ptr<float>(m), ptr<uint8_t>(ne), ptr<float>(lam),
                                            bs, L, (float)discount, (float)lambda, ptr<float>(adv), ptr<float>(ret),
                                            ptr<double>(sums), stream_of(r));
  if (rc == AREAL_ERR_UNSUPPORTED) return std::nullopt;
  check(rc, "areal_gae_padded_row_stats");
  return std::make_tuple(adv, ret, sums);
}

// x (rows of one length) normalised with the sums gae_row_stats left.
OptTensor norm_from_row_stats(const Tensor& x, const Tensor& mask, const Tensor& sums, const NormTables& norm) {
  require_gpu(x, mask, sums);
  const c10::hip::HIPGuard guard(x.device().index());
  const auto& [off, rows, longest, tail, mean_level, std_level, loo, unbiased, eps] = norm;
  const Tensor out = at::empty_like(x);
  const int rc = areal_group_norm_from_row_stats(ptr<float>(x), ptr<float>(mask), x.size(0), x.size(1), ptr<int64_t>(off),
                                                 ptr<int64_t>(rows), rows.numel(), longest, tail, mean_level, std_level,
                                                 unbiased, eps, ptr<double>(sums), ptr<float>(out), stream_of(x));
  if (rc == AREAL_ERR_UNSUPPORTED) return std::nullopt;
  check(rc, "areal_group_norm_from_row_stats");
  return out;
}

// Normalisation of x [rows, ...] under mask, with its own statistics passes.
Tensor group_norm(const Tensor& x, const OptTensor& mask, const NormTables& norm) {
  const Tensor m = f32(or_undefined(mask));
  require_gpu(x, m);
  const c10::hip::HIPGuard guard(x.device().index());
  const auto& [off, rows, longest, tail, mean_level, std_level, loo, unbiased, eps] = norm;
  const Tensor xf = f32(x), out = at::empty_like(xf);
  const size_t bytes = areal_group_norm_workspace_bytes(rows.numel(), longest);
  const Tensor ws = workspace(xf, bytes);
  check(areal_group_norm(ptr<float>(xf), ptr<float>(m), xf.numel(), ptr<int64_t>(off), ptr<int64_t>(rows), rows.numel(),
                         longest, tail, mean_level, std_level, loo, unbiased, eps, ptr<float>(out), ptr<void>(ws), bytes,
                         stream_of(xf)),
        "areal_group_norm");
  return out;
}

struct HostInt {
  std::shared_ptr<Status> status;  // null: 0
  int wait() const { return status != nullptr ? status->wait() : 0; }
};

// (advantages, returns, malformed-id flags: absent unless they are wanted)
py::tuple turn_gae(const Tensor& rewards, const OptTensor& values, const Tensor& loss_mask, const Tensor& turn_ids,
                   bool roll_ids, const Tensor& no_eos, double discount, double lambda, const OptTensor& lambda_seq,
                   const OptTensor& addend, bool want_flags) {
  const Tensor v = f32(or_undefined(values)), lam = or_undefined(lambda_seq), add = f32(or_undefined(addend));
  require_gpu(rewards, v, loss_mask, turn_ids, lam, add);
  const c10::hip::HIPGuard guard(rewards.device().index());
  const int64_t bs = rewards.size(0), L = rewards.size(1);
  const Tensor r = f32(rewards), m = f32(loss_mask), ne = no_eos.to(r.device(), at::kBool).contiguous();
  // ids beyond int32 cannot be valid (they must be smaller than the sequence length)
  const Tensor ids = (turn_ids.scalar_type() == at::kInt ? turn_ids
                      : turn_ids.scalar_type() == at::kLong ? turn_ids.clamp(-1, INT32_MAX).to(at::kInt)
                                                            : turn_ids.to(at::kInt)).contiguous();
  const Tensor adv = at::empty_like(r), ret = at::empty_like(r);
  std::optional<HostInt> flags;
  if (want_flags) flags.emplace();
  if (bs == 0 || L == 0) return py::make_tuple(adv, ret, flags);
  const Tensor status = at::zeros({1}, r.options().dtype(at::kInt));
  if (want_flags) flags->status = std::make_shared<Status>(status);
  const size_t bytes = areal_turn_gae_workspace_bytes(bs, L);
  const Tensor ws = workspace(r, bytes);
  const areal_stream_t stream = stream_of(r);
  check(areal_turn_gae_ex(ptr<float>(r), ptr<float>(v), ptr<float>(m), ptr<int32_t>(ids), roll_ids, ptr<uint8_t>(ne),
                          ptr<float>(lam), ptr<float>(add), bs, L, (float)discount, (float)lambda, ptr<float>(adv),
                          ptr<float>(ret), ptr<int>(status), ptr<void>(ws), bytes, stream),
        "areal_turn_gae");
  if (!want_flags) return py::make_tuple(adv, ret, flags);
  if (flags->status->target() != nullptr &&
      hipMemcpyAsync(flags->status->target(), status.data_ptr(), sizeof(int), hipMemcpyDeviceToHost,
                     (hipStream_t)stream) != hipSuccess)
    fail("copy of the turn status to the host failed");
  flags->status->mark();  // the normalisation of the advantages is queued before anyone looks
  return py::make_tuple(adv, ret, flags);
}

// Packed GAE and the normalisation of its advantages: (normalised, returns, advantages), or nothing when
// the batch is not one for the fused launches. norm: the groups' first sequences in place of offsets.
std::optional<std::tuple<Tensor, Tensor, Tensor>> gae_packed_normalized(
    const Tensor& rewards, const Tensor& values, const Tensor& loss_mask, const Tensor& cu_seqlens,
    const OptTensor& no_eos_arg, double discount, double lambda, const OptTensor& lambda_seq, const NormTables& norm) {
  const Tensor lam = or_undefined(lambda_seq);
  require_gpu(rewards, values, loss_mask, cu_seqlens, lam);
  const c10::hip::HIPGuard guard(rewards.device().index());
  const Tensor r = f32(rewards), v = f32(values), m = f32(loss_mask), cu = cu_seqlens.to(at::kInt).contiguous();
  const Tensor ne = no_eos_arg.has_value() ? no_eos_arg->to(r.device(), at::kBool).contiguous() : Tensor();
  const auto& [first, rows, longest, tail, mean_level, std_level, loo, unbiased, eps] = norm;
  const int64_t n = r.numel(), n_seqs = cu.numel() - 1;
  const Tensor adv = at::empty_like(r), ret = at::empty_like(r), out = at::empty_like(r);
  const size_t bytes = areal_gae_packed_normalized_workspace_bytes(n, rows.numel());
  const Tensor ws = workspace(r, bytes);
  const int rc = areal_gae_packed_normalized_ex(
      ptr<float>(r), ptr<float>(v), ptr<float>(m), ptr<int32_t>(cu), ptr<uint8_t>(ne), ptr<float>(lam), n, n_seqs,
      (float)discount, (float)lambda, ptr<int64_t>(first), ptr<int64_t>(rows), rows.numel(), longest, tail, mean_level,
      std_level, unbiased, eps, -1, ptr<float>(adv), ptr<float>(ret), ptr<float>(out), ptr<void>(ws), bytes, stream_of(r));
  if (rc == AREAL_ERR_UNSUPPORTED || rc == AREAL_ERR_ALIGNMENT) return std::nullopt;
  check(rc, "areal_gae_packed_normalized");
  return std::make_tuple(out, ret, adv);
}

// ---------------------------------------------------------------------------------------
// Packing: the sizes that the API returns as numbers travel as the losses' results do (HostResult), and the
// allocations and launches of a dict's tensors are one call, and so are the walks over the dict. A batch of 256 x 4096 with six
// tensors packed, padded and one result unpacked (25 us of kernels): 164 us with a tensor call, a ctypes array or a copy for
// each, 65.6 with the dicts walked in Python and the padding prepared when its total had been waited for, now 50.5.
// ---------------------------------------------------------------------------------------
constexpr size_t PACK_MAX_TENSORS = 8;  // of one launch
// Up to this size of its result an unpacking's table is read from pinned host memory by the kernel itself (8 bytes per block
// of 8 to 16 KiB) instead of being copied to the GPU first: 256 x 4096 fp32, kernels 8.0 -> 4.2 us and the host's part 12.1
// -> 9.4; at 1024 x 8192 (32 MiB) the reads cost what the copy did, 11.5 against 9.1 + 2.6.
constexpr int64_t UNPACK_DIRECT_BYTES = 32 << 20;

int64_t token_bytes(const Tensor& t, int64_t lead) {
  int64_t n = t.element_size();
  for (int64_t d = lead; d < t.dim(); ++d) n *= t.size(d);
  return n;
}
// Contiguous [n, ...] array with the trailing dimensions of t from `lead` on.
Tensor tokens_like(const Tensor& t, at::IntArrayRef first, int64_t lead) {
  std::vector<int64_t> shape(first.begin(), first.end());
  for (int64_t d = lead; d < t.dim(); ++d) shape.push_back(t.size(d));
  return at::empty(shape, at::TensorOptions().dtype(t.scalar_type()).device(t.device()));
}

// (cu_seqlens [B + 1], total, longest). Up to ROWS_TO_HOST rows the host adds the rows' lengths itself: it has them a kernel
// before the offsets are ready. The sizes of 64 x 1000 14.6 -> 12.5 us, of 256 x 4096 14.6 -> 13.0 (packing, padding and
// unpacking it 69.0 -> 64.6); of 1024 x 4096 15.4 for 14.7: so many writes to host memory take longer.
constexpr int64_t ROWS_TO_HOST = 512;
std::tuple<Tensor, int64_t, int64_t> seqlens_of_mask(const Tensor& mask) {
  require_gpu(mask);
  const c10::hip::HIPGuard guard(mask.device().index());
  const int64_t bs = mask.size(0), S = mask.size(1);
  const Tensor m = (mask.scalar_type() == at::kBool ? mask : mask.ne(0)).contiguous();
  const Tensor lens = empty(m, {2 * bs + 2}, at::kInt);
  const Tensor cu = lens.narrow(0, bs, bs + 1), longest = lens.narrow(0, 2 * bs + 1, 1);
  if (bs > 0 && bs <= ROWS_TO_HOST) {
    HostResult rows(lens.narrow(0, 0, bs));
    check(areal_seqlens_from_mask_rows(ptr<uint8_t>(m), bs, S, ptr<int32_t>(lens), ptr<int32_t>(cu), ptr<int32_t>(longest),
                                       rows.target(), stream_of(m)),
          "areal_seqlens_from_mask");
    const Tensor counts = rows.value().to(at::kDouble);
    const double* h = (const double*)counts.data_ptr();
    int64_t total = 0, most = 0;
    for (int64_t i = 0; i < bs; ++i) {
      total += (int64_t)h[i];
      most = std::max(most, (int64_t)h[i]);
    }
    return {cu, total, most};
  }
  HostResult host(lens.narrow(0, 2 * bs, 2));
  check(areal_seqlens_from_mask_ex(ptr<uint8_t>(m), bs, S, ptr<int32_t>(lens), ptr<int32_t>(cu), ptr<int32_t>(longest),
                                   host.target(), stream_of(m)),
        "areal_seqlens_from_mask");
  const Tensor sizes = host.value().to(at::kDouble);
  const double* h = (const double*)sizes.data_ptr();
  return {cu, (int64_t)h[0], (int64_t)h[1]};
}

// Last entry of an int32 array for the host: read by a kernel that is launched anyway (pad_rows), or by one of its own when
// it is waited for without.
struct LastValue {
  Tensor last;
  HostResult host;
  bool queued = false;
  static Tensor last_of(const Tensor& x) {
    require_gpu(x);
    if (x.numel() == 0) throw py::index_error("index -1 is out of bounds for dimension 0 with size 0");
    return x.narrow(0, x.numel() - 1, 1);
  }
  explicit LastValue(const Tensor& x) : last(last_of(x)), host(last) {}
  int64_t wait() {
    if (!queued && host.target() != nullptr) {
      const c10::hip::HIPGuard guard(last.device().index());
      check(areal_int_to_host(ptr<int32_t>(last), host.target(), stream_of(last)), "areal_int_to_host");
      queued = true;
    }
    return (int64_t)*(const double*)host.value().to(at::kDouble).data_ptr();
  }
};

// The padded [bs, S, ...] tensors packed to [total, ...].
std::vector<Tensor> pack_rows(const std::vector<Tensor>& padded, const Tensor& cu, int64_t bs, int64_t S, int64_t total) {
  require_gpu(cu);
  const c10::hip::HIPGuard guard(cu.device().index());
  std::vector<Tensor> src, out;
  for (const Tensor& t : padded) {
    require_gpu(t);
    src.push_back(t.contiguous());
    out.push_back(tokens_like(t, {total}, 2));
  }
  for (size_t i = 0; i < src.size(); i += PACK_MAX_TENSORS) {
    const size_t n = std::min(PACK_MAX_TENSORS, src.size() - i);
    const void* from[PACK_MAX_TENSORS];
    void* to[PACK_MAX_TENSORS];
    int64_t sizes[PACK_MAX_TENSORS];
    for (size_t k = 0; k < n; ++k) {
      from[k] = src[i + k].data_ptr();
      to[k] = out[i + k].data_ptr();
      sizes[k] = token_bytes(src[i + k], 2);
    }
    check(areal_pack_padded_multi(from, to, sizes, (int)n, ptr<int32_t>(cu), bs, S, total, stream_of(cu)),
          "areal_pack_padded_multi");
  }
  return out;
}

// The packed [total, ...] tensors with one more sequence behind the others, up to total_new tokens of their fill
// pattern (at most 16 bytes; none: position ids, which count up). Also writes cu_copy and cu_new. last (nullable): of cu.
std::vector<Tensor> pad_rows(const std::vector<Tensor>& packed, const std::vector<std::string>& fills, const Tensor& cu,
                             const Tensor& cu_copy, const Tensor& cu_new, int64_t total, int64_t total_new,
                             LastValue* last) {
  require_gpu(cu);
  const c10::hip::HIPGuard guard(cu.device().index());
  std::vector<Tensor> src, out;
  for (const Tensor& t : packed) {
    require_gpu(t);
    src.push_back(t.contiguous());
    out.push_back(tokens_like(t, {total_new}, 1));
  }
  for (size_t i = 0; i == 0 || i < src.size(); i += PACK_MAX_TENSORS) {
    const size_t n = std::min(PACK_MAX_TENSORS, src.size() - i);
    const void* from[PACK_MAX_TENSORS];
    void* to[PACK_MAX_TENSORS];
    int64_t sizes[PACK_MAX_TENSORS];
    char patterns[16 * PACK_MAX_TENSORS] = {};
    int pattern_bytes[PACK_MAX_TENSORS], ids[PACK_MAX_TENSORS];
    for (size_t k = 0; k < n; ++k) {
      const std::string& fill = fills.at(i + k);
      from[k] = src[i + k].data_ptr();
      to[k] = out[i + k].data_ptr();
      sizes[k] = token_bytes(src[i + k], 1);
      ids[k] = fill.empty();
      pattern_bytes[k] = fill.empty() ? 1 : (int)fill.size();
      fill.copy(patterns + 16 * k, 16);
    }
    double* const host_total = last != nullptr && !last->queued ? last->host.target() : nullptr;
    check(areal_pad_packed_multi_ex(from, to, sizes, patterns, pattern_bytes, ids, (int)n, ptr<int32_t>(cu), cu.numel() - 1,
                                    ptr<int32_t>(cu_copy), ptr<int32_t>(cu_new), total, total_new, host_total, stream_of(cu)),
          "areal_pad_packed_multi");
    if (host_total != nullptr) last->queued = true;
  }
  return out;
}

// The tensors and keys of a batch dict, without a Python call per entry. (A tensor subclass is a tensor here as it is there.)
const Tensor* tensor_of(PyObject* x) { return THPVariable_Check(x) ? &THPVariable_Unpack(x) : nullptr; }
bool is_key(PyObject* k, const char* name) { return PyUnicode_Check(k) && PyUnicode_CompareWithASCIIString(k, name) == 0; }

// A batch dict packed: pack_tensor_dict of areal_amd/packing.py behind its checks.
py::dict pack_dict(const py::dict& data, const Tensor& attention_mask) {
  const int64_t bs = attention_mask.size(0), S = attention_mask.size(1);
  const auto [cu, total, longest] = seqlens_of_mask(attention_mask);
  py::dict out;
  std::vector<PyObject*> keys;
  std::vector<Tensor> moved;
  PyObject *key, *value;
  Py_ssize_t at = 0;
  auto set = [&](PyObject* k, PyObject* v) {
    if (PyDict_SetItem(out.ptr(), k, v) != 0) throw py::error_already_set();
  };
  while (PyDict_Next(data.ptr(), &at, &key, &value)) {
    if (is_key(key, "attention_mask")) {
      out["cu_seqlens"] = cu;
      out["max_seqlen"] = longest;
      continue;
    }
    set(key, value);
    const Tensor* const t = tensor_of(value);
    if (t == nullptr || t->dim() < 2 || t->size(0) != bs || t->size(1) != S) continue;
    keys.push_back(key);
    moved.push_back(*t);
  }
  const std::vector<Tensor> packed = pack_rows(moved, cu, bs, S, total);
  for (size_t i = 0; i < keys.size(); ++i) set(keys[i], py::cast(packed[i]).ptr());
  return out;
}

// A packed batch padded with zeros to `to` tokens, for the total that its tensors' shapes suggest (the elements of the
// one-dimensional ones): (padded dict, pad length, copy of the offsets). The launch reports the total it met. Where that is another
// one, it (the caller pads anew); nothing where this is not the way (no such tensor, or of several lengths, position
// ids, a length that is no plain int, tensors that the kernel does not take: the caller's own way says what is wrong with them).
py::object pad_likely(const py::dict& data, const Tensor& cu, int64_t to) {
  // (a tensor of one entry a sequence is no token tensor; of one that is longer than the batch the padding would be for nothing)
  int64_t total = 0, second = 0, longest = 0;
  PyObject *key, *value;
  Py_ssize_t at = 0;
  while (PyDict_Next(data.ptr(), &at, &key, &value)) {
    if (is_key(key, "position_ids")) return py::none();
    if (is_key(key, "max_seqlen")) {
      int overflow = 0;
      if (!PyLong_CheckExact(value) || (longest = PyLong_AsLongLongAndOverflow(value, &overflow), overflow != 0)) return py::none();
    }
    const Tensor* const t = is_key(key, "cu_seqlens") ? nullptr : tensor_of(value);
    if (t == nullptr || t->dim() != 1 || t->numel() == total) continue;
    second = std::max(second, std::min(total, t->numel()));
    total = std::max(total, t->numel());
  }
  if (total <= 0 || total >= to || second > cu.numel()) return py::none();
  require_gpu(cu);
  const c10::hip::HIPGuard guard(cu.device().index());
  LastValue last(cu);
  const Tensor cu_new = empty(cu, {cu.numel() + 1}, at::kInt), cu_copy = at::empty_like(cu);
  py::dict out;
  std::vector<PyObject*> keys;
  std::vector<Tensor> moved;
  auto set = [&](PyObject* k, PyObject* v) {
    if (PyDict_SetItem(out.ptr(), k, v) != 0) throw py::error_already_set();
  };
  for (at = 0; PyDict_Next(data.ptr(), &at, &key, &value);) {
    if (is_key(key, "cu_seqlens")) {
      set(key, py::cast(cu_new).ptr());
    } else if (is_key(key, "max_seqlen")) {
      set(key, py::cast(std::max(longest, to - total)).ptr());
    } else {
      set(key, value);
      const Tensor* const t = tensor_of(value);
      if (t == nullptr || t->numel() != total) continue;
      if (t->device() != cu.device() || t->layout() != at::kStrided || t->is_nested() || t->element_size() > 16) return py::none();
      keys.push_back(key);
      moved.push_back(*t);
    }
  }
  try {
    std::vector<std::string> fills;
    for (Tensor& t : moved) {
      if (t.dim() != 1) t = t.reshape({total});
      fills.emplace_back(t.element_size(), '\0');
    }
    const std::vector<Tensor> padded = pad_rows(moved, fills, cu, cu_copy, cu_new, total, to, &last);
    for (size_t i = 0; i < keys.size(); ++i) set(keys[i], py::cast(padded[i]).ptr());
  } catch (const c10::OutOfMemoryError&) {  // (nothing is launched yet) of a padding that nobody has asked for it is not the caller's
    const int64_t met = last.wait();
    if (met == total) throw;
    return py::int_(met);
  }
  const int64_t met = last.wait();
  if (met != total) return py::int_(met);
  return py::make_tuple(out, to - total, cu_copy);
}

// Rows of a packed tensor, zero padded, in the given order; nothing where the arguments are not plain lists of
// lengths that add up and a permutation (the caller's general path says what is wrong with them) or where the
// table's copy would be captured.
OptTensor unpack_rows(const Tensor& packed, const py::list& seqlens, const std::optional<py::list>& order) {
  const int64_t n = (int64_t)seqlens.size();
  if (n == 0 || packed.dim() == 0 || !packed.is_cuda() || (order.has_value() && (int64_t)order->size() != n))
    return std::nullopt;
  const c10::hip::HIPGuard guard(packed.device().index());
  if (capturing()) return std::nullopt;
  // list entries that are ints of [0, below)
  auto entry = [](const py::list& list, int64_t i, int64_t below) -> int64_t {
    PyObject* const x = PyList_GET_ITEM(list.ptr(), i);
    if (!PyLong_CheckExact(x)) return -1;
    int overflow = 0;
    const int64_t v = PyLong_AsLongLongAndOverflow(x, &overflow);
    return overflow != 0 || v >= below ? -1 : v;
  };
  const Tensor host = at::empty({n, 2}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
  int32_t* const t = (int32_t*)host.data_ptr();
  std::vector<int32_t> first(n + 1);
  int64_t total = 0, longest = 0;
  for (int64_t i = 0; i < n; ++i) {
    const int64_t len = entry(seqlens, i, (int64_t)INT32_MAX + 1);
    if (len < 0 || (total += len) > INT32_MAX) return std::nullopt;
    first[i + 1] = (int32_t)total;
    longest = std::max(longest, len);
  }
  if (total != packed.size(0)) return std::nullopt;
  std::vector<bool> seen(order.has_value() ? n : 0);
  for (int64_t i = 0; i < n; ++i) {
    int64_t r = i;
    if (order.has_value()) {
      r = entry(*order, i, n);
      if (r < 0 || seen[r]) return std::nullopt;
      seen[r] = true;
    }
    t[2 * i] = first[r];
    t[2 * i + 1] = first[r + 1] - first[r];
  }
  const Tensor src = packed.contiguous(), out = tokens_like(src, {n, longest}, 1);
  // The kernel reads the table where it is, a pair per block; only a long one is worth a copy, see UNPACK_DIRECT_BYTES.
  const bool direct = out.numel() * out.element_size() <= UNPACK_DIRECT_BYTES;
  const Tensor table = direct ? host : host.to(packed.device(), /*non_blocking=*/true);
  const auto stream = c10::hip::getCurrentHIPStream(src.device().index());
  check(areal_unpack_rows(ptr<void>(src), ptr<void>(out), ptr<uint32_t>(table), n, longest, token_bytes(src, 1),
                          (areal_stream_t)stream.stream()),
        "areal_unpack_rows");
  if (direct) hold_or_wait(host, stream);
  return out;
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  m.def("set_error_class", [](py::object cls) { error_class = cls.release().ptr(); });
  py::class_<StatRows>(m, "StatRows").def(py::init([](std::vector<std::tuple<int, py::str, py::str>> rows) {
    return StatRows{std::move(rows)};
  }));
  py::class_<HostResult, HostResultPtr>(m, "HostResult")
      .def("wait", &HostResult::wait)
      .def("counters", &HostResult::counters)
      .def("mark", &HostResult::mark)
      .def("fill", &HostResult::fill);
  m.def("hold_or_wait", [](const Tensor& pinned, int64_t device) {
    hold_or_wait(pinned, c10::hip::getCurrentHIPStream((c10::DeviceIndex)device));
  });
  m.def("actor_loss", &actor_loss);
  m.def("proximal_stats", &proximal_stats);
  m.def("sapo_loss", &sapo_loss);
  m.def("critic_loss", &critic_loss);
  py::class_<LMHeadState, std::shared_ptr<LMHeadState>>(m, "LMHeadState")
      .def_property_readonly("probs", [](const LMHeadState& s) { return s.probs.defined() ? OptTensor(s.probs) : OptTensor(); })
      .def_property_readonly("probs_ref", [](const LMHeadState& s) { return s.probs_ref.defined() ? OptTensor(s.probs_ref) : OptTensor(); })
      .def_property_readonly("probs_status", [](const LMHeadState& s) { return s.probs_status.defined() ? OptTensor(s.probs_status) : OptTensor(); });
  m.def("lm_head", &lm_head);
  m.def("lm_head_backward", &lm_head_backward);
  m.def("default_token_chunk", &default_token_chunk);
  m.def("logits_logprobs", &logits_logprobs);
  py::class_<HostInt>(m, "HostInt").def("wait", &HostInt::wait);
  m.def("advantage_prep", &advantage_prep);
  m.def("gae_row_stats", &gae_row_stats);
  m.def("norm_from_row_stats", &norm_from_row_stats);
  m.def("group_norm", &group_norm);
  m.def("turn_gae", &turn_gae);
  m.def("gae_packed_normalized", &gae_packed_normalized);
  m.def("seqlens_of_mask", &seqlens_of_mask);
  py::class_<LastValue>(m, "LastValue")
      .def(py::init([](const Tensor& x) {
        require_gpu(x);
        const c10::hip::HIPGuard guard(x.device().index());
        return std::make_unique<LastValue>(x);
      }))
      .def("wait", &LastValue::wait);
  m.def("pack_rows", &pack_rows);
  m.def("pack_dict", &pack_dict);
  m.def("pad_likely", &pad_likely);
  m.def("pad_rows", [](const std::vector<Tensor>& packed, const std::vector<py::bytes>& fills, const Tensor& cu,
                       const Tensor& cu_copy, const Tensor& cu_new, int64_t total, int64_t total_new) {
    return pad_rows(packed, std::vector<std::string>(fills.begin(), fills.end()), cu, cu_copy, cu_new, total, total_new, nullptr);
  });
  m.def("unpack_rows", &unpack_rows);
}
