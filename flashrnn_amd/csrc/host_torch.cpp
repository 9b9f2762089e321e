// _host.so: the host side of flashrnn() and flashrnn_step() for the usual call (see flashrnn.py: plain tensors in the kernels'
// layouts, no transform, tracing or dispatch mode active), and the record of failed waits of every fused call.
//
// A short call is bound by the host: LSTM bf16 B5 T19 N3 D256, forward and backward, takes ~60 us on the device.  With an
// autograd function and ctypes calls in Python a pass took 300 us (a copy, an event and a tensor view per call to fetch
// its status word, a dozen ctypes calls, the interpreter on the autograd worker thread); here it takes 87 to 107 alone and 64 to 95
// behind others, by process.  The forward alone 57 -> 17 us of host time, flashrnn_step 9.6 -> 7 us a call.
// The entry points of libflashrnn_hip.so are handed over as addresses (bind), so the library that FLASHRNN_HIP_LIBRARY names is
// the one that runs, and this file needs no HIP symbol of its own.
#include <torch/extension.h>
#include <torch/csrc/autograd/functions/basic_ops.h>

#include <c10/hip/HIPStream.h>

#include <atomic>
#include <cstring>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "../../include/flashrnn_hip.h"

namespace {

using torch::Tensor;

struct Api {
  decltype(&frnn_last_error) last_error;
  decltype(&frnn_fused_supported) fused_supported, alt_supported, recompute_supported;
  decltype(&frnn_fused_max_batch) max_batch;
  decltype(&frnn_fused_cache_bytes_opt) fused_cache_bytes, alt_cache_bytes;
  decltype(&frnn_fused_workspace_bytes_opt) fused_workspace_bytes;
  decltype(&frnn_alt_workspace_bytes) alt_workspace_bytes;
  decltype(&frnn_fused_forward_opt) fused_forward, alt_forward;
  decltype(&frnn_fused_backward_opt) fused_backward, alt_backward;
  decltype(&frnn_fused_backward_recompute) backward_recompute;
  decltype(&frnn_fused_step) fused_step, alt_step;
  decltype(&frnn_stream_capturing) stream_capturing;
  decltype(&frnn_wait_launches) wait_launches;
};
Api api{};

void bind(const std::unordered_map<std::string, uintptr_t>& f) {
  auto get = [&](auto& p, const char* name) { p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(f.at(name)); };
  get(api.last_error, "frnn_last_error");
  get(api.fused_supported, "frnn_fused_supported");
  get(api.alt_supported, "frnn_alt_supported");
  get(api.recompute_supported, "frnn_fused_recompute_supported");
  get(api.max_batch, "frnn_fused_max_batch");
  get(api.fused_cache_bytes, "frnn_fused_cache_bytes_opt");
  get(api.alt_cache_bytes, "frnn_alt_cache_bytes_opt");
  get(api.fused_workspace_bytes, "frnn_fused_workspace_bytes_opt");
  get(api.alt_workspace_bytes, "frnn_alt_workspace_bytes");
  get(api.fused_forward, "frnn_fused_forward_opt");
  get(api.alt_forward, "frnn_alt_forward_opt");
  get(api.fused_backward, "frnn_fused_backward_opt");
  get(api.alt_backward, "frnn_alt_backward_opt");
  get(api.backward_recompute, "frnn_fused_backward_recompute");
  get(api.fused_step, "frnn_fused_step");
  get(api.alt_step, "frnn_alt_step");
  get(api.stream_capturing, "frnn_stream_capturing");
  get(api.wait_launches, "frnn_wait_launches");
}

// (as _raise in flashrnn.py: the reference raises ValueError when no tiling exists)
void check_rc(int rc, bool fused, const char* what) {
  if (rc == 0) return;
  const std::string msg = std::string(fused ? "hip_fused" : "hip") + " " + what + ": " + api.last_error() + " (code " + std::to_string(rc) + ")";
  TORCH_CHECK_VALUE(rc != FRNN_E_UNSUPPORTED, msg);
  TORCH_CHECK(false, msg);
}

// ---- failed waits -------------------------------------------------------------------------------------------------
// A fused kernel whose bounded wait between workgroups ran out fills its outputs with NaN and sets the status word of its
// workspace.  It also sets two words of pinned host memory that the call was given (frnn_options.report / report_any): one that
// belongs to the call, out of kSlots, and one that all calls share.  So nothing is copied or recorded per call: a later call
// reads the shared word, and only where it is set looks for the calls that set theirs, once the launches so far have ended.
// A word belongs to its call until the call's launches are known to have ended: when none is free, a call waits for what
// was launched so far and frees those words, reading them as it does.  The words of calls that were not launched yet
// (another thread, between take and the launch) stay theirs.
constexpr int kSlots = 4096;
const char* const kNames[4] = {"lstm", "slstm", "gru", "elman"};
struct CallInfo { int kind, function, B, T, N, D; };
struct StatusRing {
  enum State : char { kFree, kTaken, kLaunched };
  struct Slot { CallInfo call; State state = kFree; bool reported = false; long id = -1; };
  std::mutex mu;
  Tensor words;              // pinned: [kSlots] and the shared word
  std::atomic<int*> base{nullptr};  // its memory, for threads that look at the shared word without holding mu
  std::vector<Slot> slots;
  std::vector<int> free_slots;
  long taken = 0;
  struct { int slot = -1; long id = -1; int failed = 0; } last[2];  // the most recent call of each kind; failed: once its word is another call's
  std::vector<std::string> found;  // failed calls whose words were freed before anyone asked

  // a call's word, from take to behind its launches
  struct Ticket {
    StatusRing* ring = nullptr;
    int slot = -1;
    Ticket() = default;
    Ticket(Ticket&& o) : ring(o.ring), slot(o.slot) { o.slot = -1; }
    ~Ticket() { if (slot >= 0) ring->launched(slot); }
  };

  volatile int* any() {
    int* const w = base.load(std::memory_order_acquire);
    return w ? w + kSlots : nullptr;
  }
  // the words of a call on `stream`; calls under capture are not recorded: a replay repeats the kernels, not this
  Ticket take(const CallInfo& c, void* stream, frnn_options& o) {
    Ticket t;
    o.report = o.report_any = nullptr;
    if (api.stream_capturing(stream)) return t;
    std::unique_lock<std::mutex> lk(mu);
    if (!words.defined()) {
      words = torch::zeros({kSlots + 1}, torch::TensorOptions().dtype(torch::kInt).pinned_memory(true));
      slots.assign(kSlots, Slot{});
      for (int i = kSlots - 1; i >= 0; --i) free_slots.push_back(i);
      base.store(words.data_ptr<int>(), std::memory_order_release);
    }
    while (free_slots.empty()) {  // (again where other threads took them all meanwhile)
      const auto ended = wait_for_launched(lk);
      if (!words.defined()) return t;  // (drained meanwhile: the process ends)
      for (const auto& [i, id] : ended) {
        if (slots[i].state != kLaunched || slots[i].id != id) continue;  // (another thread freed it meanwhile)
        read(i, found);
        for (auto& l : last)
          if (l.slot == i && l.id == id) { l.failed = word(i) != 0; l.slot = -1; }
        word(i) = 0;
        slots[i].state = kFree;
        free_slots.push_back(i);
      }
      if (!found.empty()) *any() = 1;
    }
    t.ring = this;
    t.slot = free_slots.back();
    free_slots.pop_back();
    Slot& s = slots[t.slot];
    s.call = c; s.state = kTaken; s.reported = false; s.id = taken++;
    auto& l = last[c.kind];
    l.slot = t.slot; l.id = s.id; l.failed = 0;
    o.report = words.data_ptr<int>() + t.slot;
    o.report_any = words.data_ptr<int>() + kSlots;
    return t;
  }
  void launched(int slot) {
    std::lock_guard<std::mutex> lk(mu);
    if (slot < (int)slots.size() && slots[slot].state == kTaken) slots[slot].state = kLaunched;
  }
  // descriptions of the calls whose word is set, once each
  std::vector<std::string> collect() {
    std::unique_lock<std::mutex> lk(mu);
    std::vector<std::string> failed;
    if (!words.defined() || *any() == 0) return failed;
    *any() = 0;  // (in front of the wait: what ends behind it sets the word again)
    const auto ended = wait_for_launched(lk);  // (the other workgroups of a call that reported may still be on their way out)
    if (!words.defined()) return failed;
    failed.swap(found);
    for (const auto& [i, id] : ended)
      if (slots[i].state == kLaunched && slots[i].id == id) read(i, failed);
    for (int i = 0; i < kSlots; ++i)  // (calls launched behind the wait began: asked for again)
      if (slots[i].state != kFree && !slots[i].reported && word(i) != 0) *any() = 1;
    return failed;
  }
  // Waits, without the lock, for the calls that are launched by now; returns them.
  std::vector<std::pair<int, long>> wait_for_launched(std::unique_lock<std::mutex>& lk) {
    std::vector<std::pair<int, long>> ended;
    for (int i = 0; i < kSlots; ++i)
      if (slots[i].state == kLaunched) ended.emplace_back(i, slots[i].id);
    lk.unlock();
    api.wait_launches();
    lk.lock();
    return ended;
  }
  volatile int& word(int i) { return words.data_ptr<int>()[i]; }
  void read(int i, std::vector<std::string>& failed) {  // (the call has ended, mu is held)
    if (slots[i].reported || word(i) == 0) return;
    slots[i].reported = true;
    const CallInfo& c = slots[i].call;
    failed.push_back(std::string(c.kind ? "backward" : "forward") + " of " + kNames[c.function] + " B" + std::to_string(c.B) + " T" +
                     std::to_string(c.T) + " N" + std::to_string(c.N) + " D" + std::to_string(c.D));
  }
  void poll(bool wait, void* stream) {
    const volatile int* a = any();
    if (!a || (!wait && *a == 0) || api.stream_capturing(stream)) return;
    if (wait) api.wait_launches();
    const auto failed = collect();
    if (failed.empty()) return;
    std::string what;
    for (const auto& f : failed) what += (what.empty() ? "" : "; ") + f;
    TORCH_CHECK(false, "flashrnn_amd: a bounded wait between the workgroups of a head ran out in an earlier fused call (", what,
                "): its outputs are NaN.  The workgroups of a head must all be resident; another process's kernels on the same device "
                "can prevent that");
  }
  int last_word(int kind) {
    api.wait_launches();
    std::lock_guard<std::mutex> lk(mu);
    const auto& l = last[kind];
    return l.slot >= 0 ? word(l.slot) != 0 : l.failed;
  }
  std::vector<std::string> drain() {
    api.wait_launches();
    auto failed = collect();
    std::lock_guard<std::mutex> lk(mu);
    base.store(nullptr);
    words.reset();  // (pinned memory goes back while the HIP runtime is up)
    slots.clear(); free_slots.clear();
    for (auto& l : last) l = {};
    return failed;
  }
};
StatusRing& ring() { static StatusRing* r = new StatusRing; return *r; }  // (never destroyed: calls may end after static destruction began)

void* stream_of(const Tensor& x) { return c10::hip::getCurrentHIPStream(x.device().index()).stream(); }

constexpr int kGr[4] = {4, 4, 3, 1}, kGw[4] = {4, 4, 3, 1}, kGt[4] = {4, 4, 4, 1}, kS[4] = {2, 4, 1, 1};
c10::ScalarType kernel_type(int d) { return d == FRNN_BF16 ? torch::kBFloat16 : d == FRNN_F16 ? torch::kHalf : torch::kFloat; }

// what a call was configured with (frnn_options and the rest of FlashRNNConfig that reaches the kernels)
struct Call : torch::CustomClassHolder {
  int function, dtype;
  bool fused, amp, training;
  bool zero_s0 = false;  // s0 is this call's own, and its launches set it to zero
  frnn_options o;
};
using CallPtr = c10::intrusive_ptr<Call>;
CallPtr make_call(int function, int dtype, bool fused, double h_clip, double g_clip, bool cut, bool rc, bool amp) {
  auto c = c10::make_intrusive<Call>();
  c->function = function; c->dtype = dtype; c->fused = fused; c->amp = amp; c->training = false;
  c->o = frnn_options{};
  c->o.struct_size = sizeof(frnn_options);
  c->o.forward_clipval = (float)h_clip; c->o.gradient_recurrent_clipval = (float)g_clip;
  c->o.gradient_recurrent_cut = cut; c->o.recompute = rc && fused;
  return c;
}

// what the reverse pass needs of it, as whole numbers: an autograd node's record has to be hashable (compiled autograd keys its graphs by it)
c10::List<int64_t> pack(const Call& c) {
  int32_t h, g;
  std::memcpy(&h, &c.o.forward_clipval, 4); std::memcpy(&g, &c.o.gradient_recurrent_clipval, 4);
  return c10::List<int64_t>({c.function, c.dtype, c.fused, h, g, c.o.gradient_recurrent_cut, c.o.recompute, c.o.weight_grads});
}
Call unpack(const std::vector<int64_t>& p) {
  Call c;
  c.function = (int)p.at(0); c.dtype = (int)p.at(1); c.fused = p.at(2) != 0; c.amp = c.training = true;
  c.o = frnn_options{};
  c.o.struct_size = sizeof(frnn_options);
  const int32_t h = (int32_t)p.at(3), g = (int32_t)p.at(4);
  std::memcpy(&c.o.forward_clipval, &h, 4); std::memcpy(&c.o.gradient_recurrent_clipval, &g, 4);
  c.o.gradient_recurrent_cut = (int)p.at(5); c.o.recompute = (int)p.at(6); c.o.weight_grads = (int)p.at(7);
  return c;
}

Tensor cast(const Tensor& x, const char* name, const Call& c) {
  const auto k = kernel_type(c.dtype);
  TORCH_CHECK_TYPE(c.amp || x.scalar_type() == k, name, " is ", x.scalar_type(), ", the kernel type is ", k,
                   " and enable_automatic_mixed_precision is off");
  return x.detach().to(k).contiguous();
}

struct Saved { Tensor R, b, s0, states, cache, Wx; };

// one forward call of the library (as _run_forward in flashrnn.py)
Saved run_forward(const Tensor& Wx_, const Tensor& R_, const Tensor& b_, const Tensor& s0_, const Call& c) {
  Saved v;
  const int64_t B = Wx_.size(0), T = Wx_.size(1), N = Wx_.size(3), D = Wx_.size(4), S = kS[c.function];
  v.Wx = cast(Wx_, "Wx", c); v.R = cast(R_, "R", c); v.b = cast(b_, "b", c);
  v.s0 = cast(s0_, "states", c);
  c10::DeviceGuard guard(v.Wx.device());
  check_rc((c.fused ? api.fused_supported : api.alt_supported)(c.function, c.dtype, B, N, D), c.fused, "backend");
  if (c.o.recompute) check_rc(api.recompute_supported(c.function, c.dtype, B, N, D), c.fused, "backend");
  const auto bytes = v.Wx.options().dtype(torch::kByte);
  v.states = torch::empty({S, B, T, N, D}, v.Wx.options());
  const size_t cache = c.training ? (c.fused ? api.fused_cache_bytes : api.alt_cache_bytes)(c.function, c.dtype, B, T, N, D, &c.o) : 0;
  v.cache = torch::empty({(int64_t)std::max<size_t>(cache, 16)}, bytes);
  const size_t wsb = std::max<size_t>(256, c.fused ? api.fused_workspace_bytes(c.function, c.dtype, B, T, N, D, 0, &c.o)
                                                   : api.alt_workspace_bytes(c.function, c.dtype, B, T, N, D, 0));
  const Tensor ws = torch::empty({(int64_t)wsb}, bytes);
  void* st = stream_of(v.Wx);
  frnn_options o = c.o;
  if (c.zero_s0) { o.clear = v.s0.data_ptr(); o.clear_bytes = v.s0.nbytes(); }
  const auto ticket = !c.fused ? StatusRing::Ticket() : ring().take({0, c.function, (int)B, (int)T, (int)N, (int)D}, st, o);
  check_rc((c.fused ? api.fused_forward : api.alt_forward)(
               c.function, c.dtype, c.training, B, T, N, D, v.Wx.data_ptr(), v.R.data_ptr(), v.b.data_ptr(), v.s0.data_ptr(),
               v.states.data_ptr(), c.training ? v.cache.data_ptr() : nullptr, ws.data_ptr(), wsb, st, &o),
           c.fused, "forward");
  return v;
}

struct Function : torch::autograd::Function<Function> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& Wx, const Tensor& R, const Tensor& b, const Tensor& s0, CallPtr c) {
    Saved v = run_forward(Wx, R, b, s0, *c);
    ctx->saved_data["call"] = pack(*c);
    // (recompute mode reads Wx again in the backward pass; it is the caller's tensor unless it was cast)
    ctx->save_for_backward({v.R, v.b, v.s0, v.states, v.cache, c->o.recompute ? v.Wx : v.cache});
    return v.states;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const Call c = unpack(ctx->saved_data["call"].toIntVector());
    const auto v = ctx->get_saved_variables();
    const bool again = torch::GradMode::is_enabled() && grads[0].requires_grad();
    torch::autograd::variable_list out;
    {
      torch::NoGradGuard no_grad;
      out = run(c, v, grads[0]);
    }
    if (again) {  // the reverse scan is not differentiable: an error where a second derivative is asked for, not a silent zero
      auto err = std::make_shared<torch::autograd::DelayedError>(
          "trying to differentiate twice a function that was marked with @once_differentiable", (int64_t)out.size());
      for (auto& g : out) { g = g.detach(); g.set_requires_grad(true); }
      out = (*err)(std::move(out));
    }
    out.emplace_back();  // (the call)
    return out;
  }

  static torch::autograd::variable_list run(const Call& c, const torch::autograd::variable_list& v, const Tensor& dstates) {
    const Tensor &R = v[0], &b = v[1], &s0 = v[2], &states = v[3], &cache = v[4], &Wx = v[5];
    const int64_t S = states.size(0), B = states.size(1), T = states.size(2), N = states.size(3), D = states.size(4);
    const int64_t Gr = kGr[c.function], Gw = kGw[c.function], Gt = kGt[c.function];
    c10::DeviceGuard guard(states.device());
    void* st = stream_of(states);
    ring().poll(false, st);
    const Tensor ds = dstates.to(states.scalar_type()).contiguous();
    const auto k = states.options(), f = k.dtype(torch::kFloat);
    const Tensor dWx = torch::empty({B, T, Gw, N, D}, k), ds0 = torch::empty({S, B, N, D}, k);
    const Tensor dR = torch::empty({Gr, N, D, D}, c.o.weight_grads & 1 ? k : f), db = torch::empty({Gt, N, D}, c.o.weight_grads & 2 ? k : f);
    const size_t wsb = std::max<size_t>(256, c.fused ? api.fused_workspace_bytes(c.function, c.dtype, B, T, N, D, 1, &c.o)
                                                     : api.alt_workspace_bytes(c.function, c.dtype, B, T, N, D, 1));
    const Tensor ws = torch::empty({(int64_t)wsb}, k.dtype(torch::kByte));
    frnn_options o = c.o;
    const auto ticket = !c.fused ? StatusRing::Ticket() : ring().take({1, c.function, (int)B, (int)T, (int)N, (int)D}, st, o);
    int rc;
    if (c.o.recompute)
      rc = api.backward_recompute(c.function, c.dtype, B, T, N, D, Wx.data_ptr(), R.data_ptr(), b.data_ptr(), s0.data_ptr(), states.data_ptr(),
                                  ds.data_ptr(), dWx.data_ptr(), ds0.data_ptr(), static_cast<float*>(dR.data_ptr()), static_cast<float*>(db.data_ptr()), ws.data_ptr(), wsb, st, &o);
    else
      rc = (c.fused ? api.fused_backward : api.alt_backward)(
          c.function, c.dtype, B, T, N, D, R.data_ptr(), b.data_ptr(), s0.data_ptr(), states.data_ptr(), cache.data_ptr(), ds.data_ptr(),
          dWx.data_ptr(), ds0.data_ptr(), static_cast<float*>(dR.data_ptr()), static_cast<float*>(db.data_ptr()), ws.data_ptr(), wsb, st, &o);
    check_rc(rc, c.fused, "backward");
    // dR / db of tensors in the kernel type come rounded from the kernels (autograd would cast each in a launch of its own); the
    // others stay fp32, so that fp32 master weights receive unrounded gradients
    return {dWx, dR, db, ds0.view({S, B, 1, N, D})};
  }
};

std::string shape(const Tensor& x) {  // as Python prints a tuple
  std::string s = "(";
  for (int64_t i = 0; i < x.dim(); ++i) s += (i ? ", " : "") + std::to_string(x.size(i));
  return s + (x.dim() == 1 ? ",)" : ")");
}

// (before anything is launched: a kernel that is handed memory of another device faults)
void check_device(const char* name, const Tensor& x, const Tensor& Wx) {
  TORCH_CHECK(x.device() == Wx.device(), "flashrnn_amd: ", name, " is on ", x.device(), ", Wx on ", Wx.device());
}

// flashrnn() on tensors in the kernels' layouts; None where the call needs the general path (two heads per head of 32 units,
// ranges of the batch).
py::object call(const Tensor& Wx, const Tensor& R, const Tensor& b, const std::optional<Tensor>& states, int function, int dtype, bool fused,
                double h_clip, double g_clip, bool cut, bool rc, bool amp) {
  const int64_t Gr = kGr[function], Gw = kGw[function], Gt = kGt[function], S = kS[function];
  TORCH_CHECK_VALUE(Wx.dim() == 5 && Wx.size(2) == Gw, "Wx must be [B,T,", Gw, ",N,D], got ", shape(Wx));
  const int64_t B = Wx.size(0), T = Wx.size(1), N = Wx.size(3), D = Wx.size(4);
  TORCH_CHECK_VALUE(R.sizes() == torch::IntArrayRef({Gr, N, D, D}), "R must be [", Gr, ",", N, ",", D, ",", D, "], got ", shape(R));
  TORCH_CHECK_VALUE(b.sizes() == torch::IntArrayRef({Gt, N, D}), "b must be [", Gt, ",", N, ",", D, "], got ", shape(b));
  TORCH_CHECK_VALUE(!states || states->sizes() == torch::IntArrayRef({S, B, 1, N, D}), "states must be [", S, ",", B, ",1,", N, ",", D, "], got ",
                    states ? shape(*states) : "");
  if (D == 16 || !Wx.is_cuda() || (rc && !fused) || B > INT_MAX || T > INT_MAX || N > INT_MAX || D > INT_MAX) return py::none();
  check_device("R", R, Wx); check_device("b", b, Wx);
  if (states) check_device("states", *states, Wx);
  auto c = make_call(function, dtype, fused, h_clip, g_clip, cut, rc, amp);
  c->training = torch::GradMode::is_enabled() &&
                (Wx.requires_grad() || R.requires_grad() || b.requires_grad() || (states && states->requires_grad()));
  if (fused) {
    long rows = api.max_batch(function, dtype, T, N, D, 0, c->training, &c->o);
    if (const char* limit = getenv("FRNN_TEST_MAX_BATCH")) rows = std::min(rows, atol(limit));  // (tests: see _apply_in_batch_ranges)
    if (rows < B) return py::none();
  }
  Tensor out, last;
  {
    py::gil_scoped_release nogil;
    ring().poll(false, stream_of(Wx));
    const auto k = kernel_type(dtype);
    Tensor s0;
    if (states) s0 = *states;
    else {
      c10::DeviceGuard guard(Wx.device());
      s0 = torch::empty({S, B, 1, N, D}, Wx.options().dtype(k).requires_grad(false));
      c->zero_s0 = true;
    }
    if (k != torch::kFloat) c->o.weight_grads = (R.scalar_type() == k ? 1 : 0) | (b.scalar_type() == k ? 2 : 0);
    out = c->training ? Function::apply(Wx, R, b, s0, c) : run_forward(Wx, R, b, s0, *c).states;
    last = out.narrow(2, T - 1, 1);
  }
  return py::make_tuple(out, last);
}

Tensor step(const Tensor& Wx, const Tensor& R, const Tensor& b, const Tensor& states, int function, int dtype, bool fused, double h_clip,
            double g_clip, bool cut, bool rc, const std::optional<Tensor>& carry) {
  const int64_t Gr = kGr[function], Gw = kGw[function], Gt = kGt[function], S = kS[function];
  TORCH_CHECK_VALUE(Wx.dim() == 5 && Wx.size(1) == 1 && Wx.size(2) == Gw, "Wx must be [B,1,", Gw, ",N,D], got ", shape(Wx));
  const int64_t B = Wx.size(0), N = Wx.size(3), D = Wx.size(4);
  TORCH_CHECK_VALUE(R.sizes() == torch::IntArrayRef({Gr, N, D, D}) && b.sizes() == torch::IntArrayRef({Gt, N, D}) &&
                        states.sizes() == torch::IntArrayRef({S, B, 1, N, D}),
                    "R, b, states must be [", Gr, ",", N, ",", D, ",", D, "], [", Gt, ",", N, ",", D, "], [", S, ",", B, ",1,", N, ",", D, "]; got ",
                    shape(R), ", ", shape(b), ", ", shape(states));
  const auto k = kernel_type(dtype);
  const std::pair<const char*, const Tensor&> in[] = {{"Wx", Wx}, {"R", R}, {"b", b}, {"states", states}};
  for (const auto& [name, x] : in) {
    TORCH_CHECK(x.is_cuda(), "flashrnn_amd runs on a GPU only (got a CPU tensor); there is no CPU fallback");
    check_device(name, x, Wx);
    TORCH_CHECK_TYPE(x.scalar_type() == k && x.is_contiguous(), name, " must be a contiguous ", k, " tensor (the step path casts and copies nothing)");
  }
  TORCH_CHECK_TYPE(!carry || (carry->scalar_type() == torch::kFloat && carry->sizes() == torch::IntArrayRef({S, B, N, D}) &&
                              carry->is_contiguous() && carry->device() == Wx.device()),
                   "carry must be a contiguous float32 tensor [", S, ",", B, ",", N, ",", D, "] on the device of Wx");
  py::gil_scoped_release nogil;
  c10::DeviceGuard guard(Wx.device());
  const Tensor out = torch::empty({S, B, 1, N, D}, Wx.options().requires_grad(false));
  const auto c = make_call(function, dtype, fused, h_clip, g_clip, cut, rc, true);
  check_rc((fused ? api.fused_step : api.alt_step)(function, dtype, B, N, D, Wx.data_ptr(), R.data_ptr(), b.data_ptr(), states.data_ptr(),
                                                   out.data_ptr(), carry ? carry->data_ptr<float>() : nullptr, stream_of(Wx), &c->o),
           fused, "step");
  return out;
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  m.def("bind", &bind);
  m.def("call", &call);
  m.def("step", &step);
  // (the general path's calls, made from Python: addresses of the two words, 0 under capture, and what status_launched gets behind the launches)
  m.def("status_take", [](int kind, int function, int B, int T, int N, int D, uintptr_t stream) {
    frnn_options o{};
    auto t = ring().take({kind, function, B, T, N, D}, reinterpret_cast<void*>(stream), o);
    return std::make_tuple(reinterpret_cast<uintptr_t>(o.report), reinterpret_cast<uintptr_t>(o.report_any), std::exchange(t.slot, -1));
  }, py::call_guard<py::gil_scoped_release>());  // (it waits for the device where no word is free)
  m.def("status_launched", [](int slot) { if (slot >= 0) ring().launched(slot); }, py::call_guard<py::gil_scoped_release>());
  m.def("status_poll", [](bool wait) { ring().poll(wait, c10::hip::getCurrentHIPStream().stream()); }, py::call_guard<py::gil_scoped_release>());
  m.def("status_last", [](int kind) { return ring().last_word(kind); }, py::call_guard<py::gil_scoped_release>());
  m.def("status_drain", []() { return ring().drain(); }, py::call_guard<py::gil_scoped_release>());
}
