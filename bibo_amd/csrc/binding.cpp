// Host path of the layer modules: argument checks, allocation, workspace and the autograd node in one native call each,
// over the C ABI of include/bibo_moe.h.  A decode-size layer is four launches of 3 to 10 us; the same work done by
// ctypes and torch.autograd.Function in Python took 40 us of host time per forward and 355 us per training step, which is
// what bounded every call below a few thousand tokens.
//
// Nothing here computes: tensors are checked, results allocated, one library function called.
#include <ATen/SavedTensorHooks.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <map>
#include <memory>
#include <mutex>

#include "../../include/bibo_moe.h"

namespace {

using at::Tensor;

void check(int code, const char* what) {
  TORCH_CHECK(code == BIBO_OK, what, " failed: ", bibo_moe_strerror(code), " (code ", code, ")");
}

// ---- workspace: one grow-only byte buffer per (device, stream); calls on one stream are ordered, so they may share it ----
// A library call is several launches, so a thread keeps its stream's buffer (a Scratch) until the last of them is queued: the
// autograd thread runs a backward pass while another thread runs a forward on the same stream.
//
// Order of locks: nobody waits for a buffer with the interpreter lock in hand, and nothing is allocated or dropped with a
// buffer in hand (a tensor that Python has seen takes the interpreter lock when it goes, and so does an allocation with
// memory recording on).  A Python caller (Held) runs Python code with a buffer in hand, in which a finaliser may call the
// library again: the same thread may take its buffer twice.  The inner call's launches then lie whole between two of the
// outer's statements, and the outer holds the tensor it began with.
//
// A call under graph capture gets memory of its own, from the graph's pool, which lasts as long as the graph: the stream's
// buffer goes when a larger call comes, and another graph's replays may run beside this one's.
struct Buffer {
  std::recursive_mutex busy;
  Tensor bytes;
};
struct Pool {
  std::mutex m;                          // held for a look-up only
  std::map<std::pair<int, hipStream_t>, std::shared_ptr<Buffer>> buffers;
};
Pool& pool() {
  static Pool* p = new Pool;             // never destroyed: tensors must not outlive the allocator at exit
  return *p;
}

class Scratch {
 public:
  Scratch(c10::Device dev, hipStream_t stream, size_t bytes) {
    auto fresh = [&] { return at::empty({(int64_t)std::max<size_t>(bytes, 1)}, at::TensorOptions().dtype(at::kByte).device(dev)); };
    if (capturing(stream)) {
      bytes_ = fresh();
      return;
    }
    buffer_ = find(dev, stream);
    lock_ = std::unique_lock<std::recursive_mutex>(buffer_->busy, std::defer_lock);
    take();
    if (small(bytes)) {
      lock_.unlock();
      spare_ = fresh();
      take();
      if (small(bytes)) std::swap(buffer_->bytes, spare_);       // (or another thread has been here: the spare one goes)
    }
    bytes_ = buffer_->bytes;
  }
  const Tensor& tensor() const { return bytes_; }
  void* data_ptr() const { return bytes_.data_ptr(); }
  int64_t numel() const { return bytes_.numel(); }

 private:
  static std::shared_ptr<Buffer> find(c10::Device dev, hipStream_t stream) {
    Pool& p = pool();
    std::lock_guard<std::mutex> lock(p.m);
    std::shared_ptr<Buffer>& b = p.buffers[{dev.index(), stream}];
    if (!b) b = std::make_shared<Buffer>();
    return b;
  }
  static bool capturing(hipStream_t stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) == hipSuccess) return status != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return false;
  }
  bool small(size_t bytes) const { return !buffer_->bytes.defined() || (size_t)buffer_->bytes.numel() < bytes; }
  void take() {
    if (lock_.try_lock()) return;
    if (PyGILState_Check()) {
      py::gil_scoped_release no_gil;
      lock_.lock();
    } else {
      lock_.lock();
    }
  }
  // destroyed from the last to the first: the tensors go after the lock
  std::shared_ptr<Buffer> buffer_;
  Tensor spare_, bytes_;
  std::unique_lock<std::recursive_mutex> lock_;
};

std::unique_ptr<Scratch> scratch_of(int device_index, int64_t bytes) {
  const c10::Device dev(c10::DeviceType::CUDA, (c10::DeviceIndex)device_index);
  c10::DeviceGuard guard(dev);
  return std::make_unique<Scratch>(dev, c10::hip::getCurrentHIPStream(dev.index()).stream(), (size_t)bytes);
}

// the current stream's buffer as a Python context: (address, size), nobody else's until it ends
class Held {
 public:
  Held(int device_index, int64_t bytes) : device_index_(device_index), bytes_(bytes) {}
  std::pair<uintptr_t, int64_t> enter() {
    scratch_ = scratch_of(device_index_, bytes_);
    return {reinterpret_cast<uintptr_t>(scratch_->data_ptr()), scratch_->numel()};
  }
  void exit(py::args) { scratch_.reset(); }

 private:
  int device_index_;
  int64_t bytes_;
  std::unique_ptr<Scratch> scratch_;
};

// the same as a tensor, to look at or to fill: calls that use it take it as above
Tensor workspace(int device_index, int64_t bytes) { return scratch_of(device_index, bytes)->tensor(); }

void workspace_clear() {
  std::map<std::pair<int, hipStream_t>, std::shared_ptr<Buffer>> gone;       // goes after the lock
  Pool& p = pool();
  std::lock_guard<std::mutex> lock(p.m);
  gone.swap(p.buffers);
}

// ---- operands ----------------------------------------------------------------------------------------------------
void check_tensor(const Tensor& t, const char* name, at::ScalarType dtype, at::IntArrayRef shape) {
  TORCH_CHECK(t.is_cuda(), name, " must live on the GPU (got ", t.device(), "); bibo_amd has no CPU path");
  TORCH_CHECK_VALUE(t.is_contiguous(), name, " must be contiguous");
  TORCH_CHECK_TYPE(t.scalar_type() == dtype, name, " must be ", dtype, ", got ", t.scalar_type());
  TORCH_CHECK_VALUE(t.sizes() == shape, name, " must have shape ", shape, ", got ", t.sizes());
}

// What a call needs besides the rows: the layer's operands in kernel dtype and its settings.
struct Layer {
  Tensor w_router, bias, w_gate_up, w_down, theta;
  int k, norm, algo, n_pos, n_neg, act;
};

int dtype_code(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? BIBO_DTYPE_BF16 : BIBO_DTYPE_F32; }

// Checks the operands against the rows x [.., H] (contiguous) and fills in the shape.
bibo_moe_shape shape_of(const Tensor& x, const Layer& l, int flags = 0) {
  TORCH_CHECK(x.is_cuda(), "x must live on the GPU (got ", x.device(), "); bibo_amd has no CPU path");
  const at::ScalarType dt = x.scalar_type();
  TORCH_CHECK_TYPE(dt == at::kBFloat16 || dt == at::kFloat, "hidden states and weights must be bfloat16 or float32, got ", dt);
  const int64_t H = x.size(-1), T = H > 0 ? x.numel() / H : 0;
  TORCH_CHECK_VALUE(l.w_gate_up.dim() == 3, "w_gate_up must have three dimensions");
  const int64_t Eg = l.w_gate_up.size(0), I = l.w_gate_up.size(1) / 2, E = Eg + l.n_pos + l.n_neg;
  check_tensor(l.w_router, "w_router", dt, {E, H});
  check_tensor(l.bias, "bias", at::kFloat, {E});
  check_tensor(l.w_gate_up, "w_gate_up", dt, {Eg, 2 * I, H});
  check_tensor(l.w_down, "w_down", dt, {Eg, H, I});
  check_tensor(l.theta, "theta", at::kFloat, {Eg});
  TORCH_CHECK_VALUE(T <= INT32_MAX, "too many tokens");
  return bibo_moe_shape{(int32_t)T, (int32_t)H, (int32_t)E, l.k, (int32_t)I, dtype_code(x), l.n_pos, l.n_neg, l.act, flags};
}

Tensor counts_for(const Tensor& x, const bibo_moe_shape& sh) {
  return at::empty({sh.E}, x.options().dtype(at::kInt).requires_grad(false));
}

int32_t* int_ptr(const Tensor& t) { return t.defined() ? static_cast<int32_t*>(t.data_ptr()) : nullptr; }
const float* f32(const Tensor& t) { return static_cast<const float*>(t.data_ptr()); }
float* f32_out(Tensor& t) { return static_cast<float*>(t.data_ptr()); }

Tensor in_dtype(const Tensor& t, at::ScalarType dt) { return (t.scalar_type() == dt ? t : t.to(dt)).contiguous(); }

py::object maybe(const Tensor& t) { return t.defined() ? py::cast(t) : py::none(); }

// ---- inference: x [.., H] in compute dtype -> (out like x, counts int32 [E] or None) ----
py::tuple layer_forward(const Tensor& x_, const Tensor& w_router, const Tensor& bias, const Tensor& w_gate_up, const Tensor& w_down,
                        const Tensor& theta, int k, int norm, int algo, int n_pos, int n_neg, int act, bool want_counts,
                        at::ScalarType compute) {
  at::NoGradGuard no_grad;
  const Layer l{w_router, bias, w_gate_up, w_down, theta, k, norm, algo, n_pos, n_neg, act};
  c10::DeviceGuard guard(x_.device());
  const Tensor x = in_dtype(x_, compute);
  const bibo_moe_shape sh = shape_of(x, l);
  Tensor out = at::empty_like(x), counts;
  if (want_counts) counts = counts_for(x, sh);
  hipStream_t s = c10::hip::getCurrentHIPStream(x.device().index()).stream();
  size_t bytes = 0;
  check(bibo_moe_workspace_bytes(&sh, &bytes), "bibo_moe_workspace_bytes");
  {
    const Scratch ws(x.device(), s, bytes);
    check(bibo_moe_forward(x.data_ptr(), w_router.data_ptr(), f32(bias), w_gate_up.data_ptr(), w_down.data_ptr(), f32(theta), &sh, norm,
                           algo, out.data_ptr(), nullptr, nullptr, int_ptr(counts), nullptr, ws.data_ptr(), (size_t)ws.numel(), s),
          "bibo_moe_forward");
  }
  return py::make_tuple(out, maybe(counts));
}

// ---- the caller's seam: h [.., H] -> (residual + moe(rmsnorm(h)) like h, counts or None) ----
// residual: a tensor like h, or undefined: h itself unless flags say none.
py::tuple ffn_forward(const Tensor& h, const Tensor& norm_weight, double eps, const c10::optional<Tensor>& residual,
                      const Tensor& w_router, const Tensor& bias, const Tensor& w_gate_up, const Tensor& w_down,
                      const Tensor& theta, int k, int norm, int algo, int n_pos, int n_neg, int act, int flags, bool want_counts) {
  at::NoGradGuard no_grad;
  const Layer l{w_router, bias, w_gate_up, w_down, theta, k, norm, algo, n_pos, n_neg, act};
  c10::DeviceGuard guard(h.device());
  const Tensor x = h.contiguous();
  Tensor nw = norm_weight.detach();
  if (nw.scalar_type() == at::kBFloat16 && nw.is_contiguous() && reinterpret_cast<uintptr_t>(nw.data_ptr()) % 16 == 0)
    flags |= BIBO_FLAG_NORM_BF16;                        // read in place
  else
    nw = in_dtype(nw, at::kFloat);
  const bibo_moe_shape sh = shape_of(x, l, flags);
  check_tensor(nw, "norm_weight", nw.scalar_type(), {sh.H});
  Tensor res;
  if (residual.has_value()) {
    res = in_dtype(*residual, x.scalar_type());
    TORCH_CHECK_VALUE(res.numel() == x.numel() && res.is_cuda(), "residual must have the shape of the hidden states");
  }
  Tensor out = at::empty_like(x), counts;
  if (want_counts) counts = counts_for(x, sh);
  hipStream_t s = c10::hip::getCurrentHIPStream(x.device().index()).stream();
  size_t bytes = 0;
  check(bibo_moe_ffn_workspace_bytes(&sh, &bytes), "bibo_moe_ffn_workspace_bytes");
  {
    const Scratch ws(x.device(), s, bytes);
    check(bibo_moe_ffn_forward(x.data_ptr(), f32(nw), (float)eps, res.defined() ? res.data_ptr() : nullptr,
                               w_router.data_ptr(), f32(bias), w_gate_up.data_ptr(), w_down.data_ptr(), f32(theta), &sh, norm, algo,
                               out.data_ptr(), nullptr, nullptr, int_ptr(counts), ws.data_ptr(), (size_t)ws.numel(), s),
          "bibo_moe_ffn_forward");
  }
  return py::make_tuple(out, maybe(counts));
}

// ---- training: the whole layer as one autograd node --------------------------------------------------------------
// Gradients are what autograd gives the reference's eager layer with the selection held fixed (moe.py:157-183); the
// balancing bias gets none (router.py:38).  Two ways through the library: with `keep`,
// forward = bibo_moe_forward_train, which leaves routing, permutation and, for most shapes, pre-activations in a state tensor (about 4 I
// bytes per routed slot, 8 I for the fp32 tile kernels), and backward = bibo_moe_backward_saved; otherwise forward = bibo_moe_forward and
// backward = bibo_moe_backward, which computes all of that again from the saved input rows.  The same gradients, bit for bit.
// H = 192, I = 88, 16 experts, k = 3, T = 777 in fp32, forward and backward: 19 launches without, 13 with (one of them less for the
// balancing step, which rides on the forward's combine, and one for the copy of the biases).
struct TrainCall {
  Layer l;               // kernel-dtype copies of the parameters (the parameters themselves where they have that dtype)
  at::ScalarType compute;
  bool keep;
  Tensor counts;         // int32 [E] to fill, or undefined
  const bibo_moe_balance* balance = nullptr;   // the balancing step behind the forward, which a saved one takes along,
  bool balanced = false;                       // and whether it has
};

class LayerFn : public torch::autograd::Function<LayerFn> {
 public:
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& x, const Tensor& w_router, const Tensor& w_gate_up,
                        const Tensor& w_down, const Tensor& theta, TrainCall* c) {
    const Layer& l = c->l;
    const Tensor xb = in_dtype(x, c->compute);
    // a family that was asked for by name runs in training as well
    const bool aligned = ((reinterpret_cast<uintptr_t>(xb.data_ptr()) | reinterpret_cast<uintptr_t>(l.w_gate_up.data_ptr()) |
                           reinterpret_cast<uintptr_t>(l.w_down.data_ptr())) & 15) == 0;
    const int any = aligned ? BIBO_FLAG_KEEP_ANY : 0;
    const bibo_moe_shape sh = shape_of(xb, l, l.algo == BIBO_ALGO_AUTO ? BIBO_FLAG_TRAIN_AUTO | any : 0);
    Tensor out = at::empty_like(xb);
    hipStream_t s = c10::hip::getCurrentHIPStream(xb.device().index()).stream();
    size_t bytes = 0, state_bytes = 0;
    check(bibo_moe_workspace_bytes(&sh, &bytes), "bibo_moe_workspace_bytes");
    const bool saved = c->keep && (l.algo == BIBO_ALGO_AUTO || l.algo == BIBO_ALGO_FUSED) &&
                       bibo_moe_train_state_bytes(&sh, &state_bytes) == BIBO_OK;
    Tensor last;           // the state or, where the backward pass routes again, the selection biases
    if (saved) {
      last = at::empty({(int64_t)std::max<size_t>(state_bytes, 256)}, xb.options().dtype(at::kByte));
      const Scratch ws(xb.device(), s, bytes);
      if (c->balance != nullptr)
        check(bibo_moe_forward_train_balance(xb.data_ptr(), l.w_router.data_ptr(), f32(l.bias), l.w_gate_up.data_ptr(), l.w_down.data_ptr(),
                                             f32(l.theta), &sh, l.norm, out.data_ptr(), nullptr, c->balance, last.data_ptr(),
                                             (size_t)last.numel(), ws.data_ptr(), (size_t)ws.numel(), s),
              "bibo_moe_forward_train_balance");
      else
        check(bibo_moe_forward_train(xb.data_ptr(), l.w_router.data_ptr(), f32(l.bias), l.w_gate_up.data_ptr(), l.w_down.data_ptr(),
                                     f32(l.theta), &sh, l.norm, out.data_ptr(), int_ptr(c->counts), last.data_ptr(),
                                     (size_t)last.numel(), ws.data_ptr(), (size_t)ws.numel(), s),
              "bibo_moe_forward_train");
      c->balanced = c->balance != nullptr;
    } else {
      if (c->balance != nullptr) c->counts = counts_for(xb, sh);       // for a step behind this call
      // A private copy: the layer's balancing step writes gate.bias in place later in the same forward, and the backward
      // pass has to route with the values the forward saw.
      last = l.bias.detach().clone();
      const Scratch ws(xb.device(), s, bytes);
      check(bibo_moe_forward(xb.data_ptr(), l.w_router.data_ptr(), f32(last), l.w_gate_up.data_ptr(), l.w_down.data_ptr(),
                             f32(l.theta), &sh, l.norm, l.algo, out.data_ptr(), nullptr, nullptr, int_ptr(c->counts), nullptr,
                             ws.data_ptr(), (size_t)ws.numel(), s),
            "bibo_moe_forward");
    }
    ctx->save_for_backward({xb, l.w_router, l.w_gate_up, l.w_down, l.theta, last});
    auto& d = ctx->saved_data;
    d["conf"] = std::vector<int64_t>{l.k, l.norm, l.n_pos, l.n_neg, l.act, saved ? 1 : 0, sh.flags & BIBO_FLAG_KEEP_ANY};
    d["dtypes"] = std::vector<int64_t>{(int64_t)x.scalar_type(), (int64_t)w_router.scalar_type(), (int64_t)w_gate_up.scalar_type(),
                                       (int64_t)w_down.scalar_type(), (int64_t)theta.scalar_type()};
    return out;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    at::NoGradGuard no_grad;
    const auto t = ctx->get_saved_variables();           // read once: activation checkpointing unpacks on access
    const auto conf = ctx->saved_data["conf"].toIntVector();
    const auto dtypes = ctx->saved_data["dtypes"].toIntVector();
    const Tensor &x = t[0], &last = t[5];
    const bool saved = conf[5] != 0;
    const Layer l{t[1], saved ? Tensor() : last, t[2], t[3], t[4], (int)conf[0], (int)conf[1], BIBO_ALGO_AUTO, (int)conf[2], (int)conf[3], (int)conf[4]};
    c10::DeviceGuard guard(x.device());
    const Tensor d = in_dtype(grads[0], x.scalar_type());
    const int64_t Eg = l.w_gate_up.size(0);
    // fp32 master weights behind bf16 operands: the kernels' fp32 sums are the gradients
    const bool grad_f32 = x.scalar_type() != at::kFloat && dtypes[1] == (int64_t)at::kFloat && dtypes[2] == (int64_t)at::kFloat &&
                          dtypes[3] == (int64_t)at::kFloat;
    const bibo_moe_shape sh{(int32_t)(x.numel() / x.size(-1)), (int32_t)x.size(-1), (int32_t)(Eg + l.n_pos + l.n_neg), l.k,
                            (int32_t)(l.w_gate_up.size(1) / 2), dtype_code(x), l.n_pos, l.n_neg, l.act,
                            (grad_f32 ? BIBO_FLAG_GRAD_F32 : 0) | (int)conf[6]};
    const at::TensorOptions wopt = l.w_gate_up.options().requires_grad(false).dtype(grad_f32 ? at::kFloat : x.scalar_type());
    Tensor d_x = at::empty_like(x), d_wr = at::empty(l.w_router.sizes(), wopt), d_gu = at::empty(l.w_gate_up.sizes(), wopt),
           d_dn = at::empty(l.w_down.sizes(), wopt), d_th = at::empty_like(l.theta);
    hipStream_t s = c10::hip::getCurrentHIPStream(x.device().index()).stream();
    size_t bytes = 0;
    check(bibo_moe_backward_workspace_bytes(&sh, &bytes), "bibo_moe_backward_workspace_bytes");
    {
      const Scratch ws(x.device(), s, bytes);
      if (saved)
        check(bibo_moe_backward_saved(x.data_ptr(), d.data_ptr(), l.w_router.data_ptr(), l.w_gate_up.data_ptr(), l.w_down.data_ptr(),
                                      f32(l.theta), &sh, l.norm, last.data_ptr(), (size_t)last.numel(), d_x.data_ptr(),
                                      d_wr.data_ptr(), d_gu.data_ptr(), d_dn.data_ptr(), f32_out(d_th), nullptr, ws.data_ptr(),
                                      (size_t)ws.numel(), s),
              "bibo_moe_backward_saved");
      else
        check(bibo_moe_backward(x.data_ptr(), d.data_ptr(), l.w_router.data_ptr(), f32(last), l.w_gate_up.data_ptr(),
                                l.w_down.data_ptr(), f32(l.theta), &sh, l.norm, d_x.data_ptr(), d_wr.data_ptr(), d_gu.data_ptr(),
                                d_dn.data_ptr(), f32_out(d_th), nullptr, ws.data_ptr(), (size_t)ws.numel(), s),
              "bibo_moe_backward");
    }
    torch::autograd::variable_list out{d_x, d_wr, d_gu, d_dn, d_th, Tensor()};
    for (int i = 0; i < 5; ++i)
      if (out[i].scalar_type() != (at::ScalarType)dtypes[i]) out[i] = out[i].to((at::ScalarType)dtypes[i]);
    return out;
  }
};

// x and the parameters as the caller holds them, then their kernel-dtype copies -> (out like x in compute dtype, counts or None, whether the
// balancing step is done).  accumulated, balance_bias, factor, update: the arguments of balance_step, where the caller leaves the step to this
// call; counts only come back if it did not take it.
py::tuple layer_train(const Tensor& x, const Tensor& w_router, const Tensor& w_gate_up, const Tensor& w_down, const Tensor& theta,
                      const Tensor& wr_k, const Tensor& bias_k, const Tensor& gu_k, const Tensor& dn_k, const Tensor& th_k, int k,
                      int norm, int algo, int n_pos, int n_neg, int act, bool want_counts, at::ScalarType compute, bool keep,
                      const c10::optional<Tensor>& accumulated, const c10::optional<Tensor>& balance_bias, double factor, bool update) {
  TORCH_CHECK(x.is_cuda(), "x must live on the GPU (got ", x.device(), "); bibo_amd has no CPU path");
  c10::DeviceGuard guard(x.device());
  TrainCall c{{wr_k, bias_k, gu_k, dn_k, th_k, k, norm, algo, n_pos, n_neg, act}, compute, keep, Tensor()};
  const int64_t E = gu_k.size(0) + n_pos + n_neg;
  bibo_moe_balance balance;
  // A pack hook may end this call behind the forward's launches, as activation checkpointing ends a recomputation with the last tensor it
  // needs: the caller then counts no step, so none may have been taken.
  const bool hooked = !at::SavedTensorDefaultHooks::get_tls_state().stack.empty();
  if (accumulated.has_value() && balance_bias.has_value() && !hooked) {
    check_tensor(*accumulated, "accumulated_tpe", at::kFloat, {E});
    check_tensor(*balance_bias, "bias", at::kFloat, {E});
    balance = {static_cast<float*>(accumulated->data_ptr()), static_cast<float*>(balance_bias->data_ptr()), (float)factor, update ? 1 : 0};
    c.balance = &balance;
  } else if (want_counts) {
    c.counts = at::empty({E}, x.options().dtype(at::kInt).requires_grad(false));
  }
  Tensor out = LayerFn::apply(x, w_router, w_gate_up, w_down, theta, &c);
  if (c.balanced) {                                      // written in place
    accumulated->unsafeGetTensorImpl()->bump_version();
    if (update) balance_bias->unsafeGetTensorImpl()->bump_version();
  }
  return py::make_tuple(out, maybe(c.counts), c.balanced);
}

// accumulated += counts; with `update`, bias += factor * (mean(load) - load) for load = accumulated / max(sum, 1), and
// accumulated = 0 (moe.py:131-155).  All [E], fp32 but for the counts.
void balance_step(const Tensor& counts, Tensor accumulated, Tensor bias, double factor, bool update) {
  at::NoGradGuard no_grad;
  const int64_t E = bias.numel();
  check_tensor(counts, "counts", at::kInt, {E});
  check_tensor(accumulated, "accumulated_tpe", at::kFloat, {E});
  check_tensor(bias, "bias", at::kFloat, {E});
  c10::DeviceGuard guard(bias.device());
  check(bibo_moe_balance_step(int_ptr(counts), f32_out(accumulated), f32_out(bias), (int)E, (float)factor, update ? 1 : 0,
                              c10::hip::getCurrentHIPStream(bias.device().index()).stream()),
        "bibo_moe_balance_step");
  accumulated.unsafeGetTensorImpl()->bump_version();     // written in place
  if (update) bias.unsafeGetTensorImpl()->bump_version();
}

// ---- the 10-layer forward's own launches (bibo_amd/exp_model.py); bf16, no autograd -------------------------------
void check_rows(const Tensor& t, const char* name, int64_t cols) {
  TORCH_CHECK(t.is_cuda(), name, " must live on the GPU (got ", t.device(), "); bibo_amd has no CPU path");
  TORCH_CHECK_VALUE(t.is_contiguous() && t.dim() >= 1 && t.size(-1) == cols, name, " must be contiguous rows of ", cols);
  TORCH_CHECK_TYPE(t.scalar_type() == at::kBFloat16, name, " must be bfloat16");
}
// Small parameter vectors of one launch in the type the kernels read them in: bf16 in place where every one is bf16 and
// 16-byte aligned, else fp32 (copies of those that are not).
struct Vecs {
  std::vector<Tensor> t;
  int dtype;
  const void* operator[](size_t i) const { return t[i].defined() ? t[i].data_ptr() : nullptr; }
};
Vecs vecs(std::initializer_list<c10::optional<Tensor>> in, int64_t n, const char* what) {
  Vecs v{{}, BIBO_DTYPE_BF16};
  for (const auto& o : in) {
    const Tensor t = o.has_value() ? o->detach().reshape({-1}).contiguous() : Tensor();
    if (t.defined()) {
      TORCH_CHECK(t.is_cuda(), what, " must live on the GPU (got ", t.device(), "); bibo_amd has no CPU path");
      TORCH_CHECK_VALUE(t.numel() == n, what, " must have ", n, " elements, got ", t.numel());
      if (t.scalar_type() != at::kBFloat16 || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0) v.dtype = BIBO_DTYPE_F32;
    }
    v.t.push_back(t);
  }
  if (v.dtype == BIBO_DTYPE_F32)
    for (Tensor& t : v.t)
      if (t.defined()) t = t.to(at::kFloat);
  return v;
}
hipStream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// candidates [T, H] -> (their depth mix with score weight score_a * score_b, its RMSNorm or None)
py::tuple exp_attn_res_norm(const std::vector<Tensor>& candidates, const Tensor& score_a, const c10::optional<Tensor>& score_b,
                            double eps, const c10::optional<Tensor>& norm_weight, double norm_eps) {
  at::NoGradGuard no_grad;
  TORCH_CHECK_VALUE(!candidates.empty() && candidates.size() <= 8, "1 to 8 candidates");
  const Tensor& c0 = candidates[0];
  const int64_t H = c0.size(-1), T = c0.numel() / H;
  const void* ptrs[8];
  for (size_t i = 0; i < candidates.size(); ++i) {
    check_rows(candidates[i], "candidate", H);
    TORCH_CHECK_VALUE(candidates[i].numel() == c0.numel(), "candidates must have one size");
    ptrs[i] = candidates[i].data_ptr();
  }
  c10::DeviceGuard guard(c0.device());
  const Vecs v = vecs({score_a, score_b, norm_weight}, H, "score and norm weights");
  const void* nw = v[2];
  Tensor out = at::empty_like(c0), normed;
  if (nw != nullptr) normed = at::empty_like(c0);
  check(bibo_moe_exp_attn_res_norm_fwd(ptrs, (int)candidates.size(), v[0], v[1], (float)eps, nw, (float)norm_eps, v.dtype, (int)T, (int)H,
                                       BIBO_DTYPE_BF16, out.data_ptr(), nw != nullptr ? normed.data_ptr() : nullptr, stream_of(c0)),
        "bibo_moe_exp_attn_res_norm_fwd");
  return py::make_tuple(out, maybe(normed));
}

// Weights [n_i, K] of one dtype as a single matrix: in place where they lie one behind the other in one storage (where the
// modules put them), else a copy of the call's own (2.4 MB of q|k|v at H = 768: 6.5 us and a launch).
Tensor joined(std::initializer_list<Tensor> ws) {
  const Tensor& first = *ws.begin();
  int64_t rows = 0;
  bool adjacent = true;
  for (const Tensor& w : ws) {
    adjacent = adjacent && w.dim() == 2 && w.is_contiguous() && w.size(1) == first.size(1) && w.scalar_type() == first.scalar_type() &&
               w.storage().is_alias_of(first.storage()) && w.storage_offset() == first.storage_offset() + rows * first.size(1);
    rows += w.size(0);
  }
  return adjacent ? first.as_strided({rows, first.size(1)}, {first.size(1), 1}) : at::cat(at::ITensorListRef(ws.begin(), ws.size()));
}

// inv_freq [d / 2] -> cos, sin bf16 [S, d]
py::tuple exp_rope_tables(const Tensor& inv_freq, int64_t S) {
  at::NoGradGuard no_grad;
  c10::DeviceGuard guard(inv_freq.device());
  const int64_t half = inv_freq.numel();
  const Vecs f = vecs({inv_freq}, half, "inv_freq");
  const at::TensorOptions opt = inv_freq.options().requires_grad(false).dtype(at::kBFloat16);
  Tensor cos = at::empty({S, 2 * half}, opt), sin = at::empty({S, 2 * half}, opt);
  check(bibo_moe_exp_rope_tables(f[0], f.dtype, (int)S, (int)half, cos.data_ptr(), sin.data_ptr(), stream_of(cos)), "bibo_moe_exp_rope_tables");
  return py::make_tuple(cos, sin);
}

// x [B, S, H] -> attention output [B, S, H]: one projection to q|k|v rows, attention of their norms and rotations with XSA, output
// projection (the two products are library GEMMs)
Tensor exp_attention(const Tensor& x, const Tensor& w_q, const Tensor& w_k, const Tensor& w_v, const Tensor& w_o, const c10::optional<Tensor>& q_weight,
                     const c10::optional<Tensor>& k_weight, double eps, const c10::optional<Tensor>& cos,
                     const c10::optional<Tensor>& sin, const c10::optional<Tensor>& xsa_alpha, int n_heads, int n_kv_heads,
                     int head_dim, int window, double scale) {
  at::NoGradGuard no_grad;
  const int64_t B = x.size(0), S = x.size(1);
  check_rows(x, "x", x.size(2));
  c10::DeviceGuard guard(x.device());
  const Vecs norm = vecs({q_weight, k_weight}, head_dim, "q and k norm weights"), rope = vecs({cos, sin}, S * head_dim, "cos and sin"),
             alpha = vecs({xsa_alpha}, n_heads, "xsa_alpha");
  const Tensor qkv = at::linear(x, joined({w_q, w_k, w_v}));
  check_rows(qkv, "q|k|v rows", (int64_t)(n_heads + 2 * n_kv_heads) * head_dim);
  const int ld = (int)qkv.size(-1);
  hipStream_t s = stream_of(x);
  const Tensor y = at::empty({B, S, (int64_t)n_heads * head_dim}, x.options());
  check(bibo_moe_exp_norm_attention_fwd(qkv.data_ptr(), ld, (int)B, (int)S, n_heads, n_kv_heads, head_dim, norm[0], norm[1], norm.dtype,
                                        (float)eps, rope[0], rope[1], rope.dtype, head_dim, window, (float)scale, alpha[0], alpha.dtype,
                                        y.data_ptr(), s),
        "bibo_moe_exp_norm_attention_fwd");
  return at::linear(y, w_o);
}

// (attn_read + theta a, prefix + a or a itself)
py::tuple exp_carry(const Tensor& attn_read, const Tensor& a, const c10::optional<Tensor>& theta, const c10::optional<Tensor>& prefix) {
  at::NoGradGuard no_grad;
  const int64_t H = a.size(-1);
  check_rows(attn_read, "attn_read", H);
  check_rows(a, "a", H);
  TORCH_CHECK_VALUE(attn_read.numel() == a.numel(), "attn_read must have the size of a");
  c10::DeviceGuard guard(a.device());
  const Vecs th = vecs({theta}, H, "theta");
  Tensor out = at::empty_like(a), prefix_out;
  if (prefix.has_value()) {
    check_rows(*prefix, "prefix", H);
    TORCH_CHECK_VALUE(prefix->numel() == a.numel(), "prefix must have the size of a");
    prefix_out = at::empty_like(a);
  }
  check(bibo_moe_exp_carry_fwd(attn_read.data_ptr(), a.data_ptr(), th[0], th.dtype, prefix.has_value() ? prefix->data_ptr() : nullptr,
                               (int)(a.numel() / H), (int)H, out.data_ptr(), prefix.has_value() ? prefix_out.data_ptr() : nullptr,
                               stream_of(a)),
        "bibo_moe_exp_carry_fwd");
  return py::make_tuple(out, prefix.has_value() ? prefix_out : a);
}

// base + SwiGLU(x): gate and up in one library product, SiLU(gate) * up in one launch, base added by the down product
Tensor exp_mlp(const Tensor& x, const Tensor& w_gate, const Tensor& w_up, const Tensor& w_down, const Tensor& base) {
  at::NoGradGuard no_grad;
  const int64_t H = x.size(-1), T = x.numel() / H, I = w_gate.size(0);
  check_rows(x, "x", H);
  c10::DeviceGuard guard(x.device());
  const Tensor gu = at::linear(x.view({T, H}), joined({w_gate, w_up}));
  check_rows(gu, "gate|up rows", 2 * I);
  Tensor h = at::empty({T, I}, x.options());
  check(bibo_moe_exp_silu_mul_fwd(gu.data_ptr(), (int)T, (int)I, h.data_ptr(), stream_of(x)), "bibo_moe_exp_silu_mul_fwd");
  return at::addmm(base.reshape({T, w_down.size(0)}), h, w_down.t()).view_as(base);
}

}  // namespace

PYBIND11_MODULE(_native, m) {
  m.def("abi_version", [] { return bibo_moe_abi_version(); });
  py::class_<Held>(m, "Held").def(py::init<int, int64_t>()).def("__enter__", &Held::enter).def("__exit__", &Held::exit);
  m.def("workspace", &workspace);
  m.def("workspace_clear", &workspace_clear);
  m.def("layer_forward", &layer_forward);
  m.def("ffn_forward", &ffn_forward);
  m.def("layer_train", &layer_train);
  m.def("balance_step", &balance_step);
  m.def("exp_attn_res_norm", &exp_attn_res_norm);
  m.def("exp_rope_tables", &exp_rope_tables);
  m.def("exp_attention", &exp_attention);
  m.def("exp_carry", &exp_carry);
  m.def("exp_mlp", &exp_mlp);
}
