// Host path of the layer modules: argument checks, allocation, workspace and the autograd node in one native call each,
// over the C ABI of include/bibo_moe.h.  A decode-size layer is four launches of 3 to 10 us; the same work done by
// ctypes and torch.autograd.Function in Python took 40 us of host time per forward and 355 us per training step, which is
// what bounded every call below a few thousand tokens.
//
// Nothing here computes: tensors are checked, results allocated, one library function called.
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <map>
#include <mutex>

#include "../../include/bibo_moe.h"

namespace {

using at::Tensor;

void check(int code, const char* what) {
  TORCH_CHECK(code == BIBO_OK, what, " failed: ", bibo_moe_strerror(code), " (code ", code, ")");
}

// ---- workspace: one grow-only byte buffer per (device, stream); calls on one stream are ordered, so they may share it ----
struct Pool {
  std::mutex m;
  std::map<std::pair<int, hipStream_t>, Tensor> buffers;
};
Pool& pool() {
  static Pool* p = new Pool;             // never destroyed: tensors must not outlive the allocator at exit
  return *p;
}

Tensor workspace_on(c10::Device dev, hipStream_t stream, size_t bytes) {
  Pool& p = pool();
  std::lock_guard<std::mutex> lock(p.m);
  Tensor& t = p.buffers[{dev.index(), stream}];
  if (!t.defined() || (size_t)t.numel() < bytes)
    t = at::empty({(int64_t)std::max<size_t>(bytes, 1)}, at::TensorOptions().dtype(at::kByte).device(dev));
  return t;
}

Tensor workspace(int device_index, int64_t bytes) {
  const c10::Device dev(c10::DeviceType::CUDA, (c10::DeviceIndex)device_index);
  c10::DeviceGuard guard(dev);
  return workspace_on(dev, c10::hip::getCurrentHIPStream(dev.index()).stream(), (size_t)bytes);
}

void workspace_clear() {
  Pool& p = pool();
  std::lock_guard<std::mutex> lock(p.m);
  p.buffers.clear();
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
  const Tensor ws = workspace_on(x.device(), s, bytes);
  check(bibo_moe_forward(x.data_ptr(), w_router.data_ptr(), f32(bias), w_gate_up.data_ptr(), w_down.data_ptr(), f32(theta), &sh, norm,
                         algo, out.data_ptr(), nullptr, nullptr, int_ptr(counts), nullptr, ws.data_ptr(), (size_t)ws.numel(), s),
        "bibo_moe_forward");
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
  const bibo_moe_shape sh = shape_of(x, l, flags);
  check_tensor(norm_weight, "norm_weight", at::kFloat, {sh.H});
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
  const Tensor ws = workspace_on(x.device(), s, bytes);
  check(bibo_moe_ffn_forward(x.data_ptr(), f32(norm_weight), (float)eps, res.defined() ? res.data_ptr() : nullptr,
                             w_router.data_ptr(), f32(bias), w_gate_up.data_ptr(), w_down.data_ptr(), f32(theta), &sh, norm, algo,
                             out.data_ptr(), nullptr, nullptr, int_ptr(counts), ws.data_ptr(), (size_t)ws.numel(), s),
        "bibo_moe_ffn_forward");
  return py::make_tuple(out, maybe(counts));
}

// ---- training: the whole layer as one autograd node --------------------------------------------------------------
// Gradients are what autograd gives the reference's eager layer with the selection held fixed (moe.py:157-183); the
// balancing bias gets none (router.py:38).  Two ways through the library: with `keep` and a shape that has the pair,
// forward = bibo_moe_forward_train, which leaves routing, permutation and pre-activations in a state tensor (about 4 I
// bytes per routed slot), and backward = bibo_moe_backward_saved; otherwise forward = bibo_moe_forward and backward =
// bibo_moe_backward, which computes all of that again from the saved input rows.  The same gradients, bit for bit.
struct TrainCall {
  Layer l;               // kernel-dtype copies of the parameters (the parameters themselves where they have that dtype)
  at::ScalarType compute;
  bool keep;
  Tensor counts;         // int32 [E] to fill, or undefined
};

class LayerFn : public torch::autograd::Function<LayerFn> {
 public:
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& x, const Tensor& w_router, const Tensor& w_gate_up,
                        const Tensor& w_down, const Tensor& theta, TrainCall* c) {
    const Layer& l = c->l;
    const Tensor xb = in_dtype(x, c->compute);
    const bibo_moe_shape sh = shape_of(xb, l);
    Tensor out = at::empty_like(xb);
    hipStream_t s = c10::hip::getCurrentHIPStream(xb.device().index()).stream();
    size_t bytes = 0, state_bytes = 0;
    check(bibo_moe_workspace_bytes(&sh, &bytes), "bibo_moe_workspace_bytes");
    const Tensor ws = workspace_on(xb.device(), s, bytes);
    const bool saved = c->keep && (l.algo == BIBO_ALGO_AUTO || l.algo == BIBO_ALGO_FUSED) &&
                       bibo_moe_train_state_bytes(&sh, &state_bytes) == BIBO_OK;
    Tensor last;           // the state or, where the backward pass routes again, the selection biases
    if (saved) {
      last = at::empty({(int64_t)std::max<size_t>(state_bytes, 256)}, xb.options().dtype(at::kByte));
      check(bibo_moe_forward_train(xb.data_ptr(), l.w_router.data_ptr(), f32(l.bias), l.w_gate_up.data_ptr(), l.w_down.data_ptr(),
                                   f32(l.theta), &sh, l.norm, out.data_ptr(), int_ptr(c->counts), last.data_ptr(),
                                   (size_t)last.numel(), ws.data_ptr(), (size_t)ws.numel(), s),
            "bibo_moe_forward_train");
    } else {
      // A private copy: the layer's balancing step writes gate.bias in place later in the same forward, and the backward
      // pass has to route with the values the forward saw.
      last = l.bias.detach().clone();
      check(bibo_moe_forward(xb.data_ptr(), l.w_router.data_ptr(), f32(last), l.w_gate_up.data_ptr(), l.w_down.data_ptr(),
                             f32(l.theta), &sh, l.norm, l.algo, out.data_ptr(), nullptr, nullptr, int_ptr(c->counts), nullptr,
                             ws.data_ptr(), (size_t)ws.numel(), s),
            "bibo_moe_forward");
    }
    ctx->save_for_backward({xb, l.w_router, l.w_gate_up, l.w_down, l.theta, last});
    auto& d = ctx->saved_data;
    d["conf"] = std::vector<int64_t>{l.k, l.norm, l.n_pos, l.n_neg, l.act, saved ? 1 : 0};
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
    const bibo_moe_shape sh{(int32_t)(x.numel() / x.size(-1)), (int32_t)x.size(-1), (int32_t)(Eg + l.n_pos + l.n_neg), l.k,
                            (int32_t)(l.w_gate_up.size(1) / 2), dtype_code(x), l.n_pos, l.n_neg, l.act, 0};
    Tensor d_x = at::empty_like(x), d_wr = at::empty_like(l.w_router), d_gu = at::empty_like(l.w_gate_up),
           d_dn = at::empty_like(l.w_down), d_th = at::empty_like(l.theta);
    hipStream_t s = c10::hip::getCurrentHIPStream(x.device().index()).stream();
    size_t bytes = 0;
    check(bibo_moe_backward_workspace_bytes(&sh, &bytes), "bibo_moe_backward_workspace_bytes");
    const Tensor ws = workspace_on(x.device(), s, bytes);
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
    torch::autograd::variable_list out{d_x, d_wr, d_gu, d_dn, d_th, Tensor()};
    for (int i = 0; i < 5; ++i)
      if (out[i].scalar_type() != (at::ScalarType)dtypes[i]) out[i] = out[i].to((at::ScalarType)dtypes[i]);
    return out;
  }
};

// x and the parameters as the caller holds them, then their kernel-dtype copies -> (out like x in compute dtype, counts or None)
py::tuple layer_train(const Tensor& x, const Tensor& w_router, const Tensor& w_gate_up, const Tensor& w_down, const Tensor& theta,
                      const Tensor& wr_k, const Tensor& bias_k, const Tensor& gu_k, const Tensor& dn_k, const Tensor& th_k, int k,
                      int norm, int algo, int n_pos, int n_neg, int act, bool want_counts, at::ScalarType compute, bool keep) {
  TORCH_CHECK(x.is_cuda(), "x must live on the GPU (got ", x.device(), "); bibo_amd has no CPU path");
  c10::DeviceGuard guard(x.device());
  TrainCall c{{wr_k, bias_k, gu_k, dn_k, th_k, k, norm, algo, n_pos, n_neg, act}, compute, keep, Tensor()};
  if (want_counts) c.counts = at::empty({gu_k.size(0) + n_pos + n_neg}, x.options().dtype(at::kInt).requires_grad(false));
  Tensor out = LayerFn::apply(x, w_router, w_gate_up, w_down, theta, &c);
  return py::make_tuple(out, maybe(c.counts));
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

}  // namespace

PYBIND11_MODULE(_native, m) {
  m.def("abi_version", [] { return bibo_moe_abi_version(); });
  m.def("workspace", &workspace);
  m.def("workspace_clear", &workspace_clear);
  m.def("layer_forward", &layer_forward);
  m.def("ffn_forward", &ffn_forward);
  m.def("layer_train", &layer_train);
  m.def("balance_step", &balance_step);
}
