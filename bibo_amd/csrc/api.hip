// extern "C" entry points: host-side argument checks, workspace carving and kernel dispatch.
// Nothing here allocates or synchronises; see include/bibo_moe.h for the contract.
#include <mutex>

#include "common.h"

// Workspace of bibo_moe_forward_static: one copy per GPU, alive until the process ends.  In host code the
// name is only a handle for hipGetSymbolAddress; kernels get the per-device address looked up below.
static __device__ __align__(256) unsigned char scratch[BIBO_MOE_STATIC_SCRATCH_BYTES];

namespace {

using namespace bibo;

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// Address of `scratch` on the current device, looked up once per device.
int static_scratch(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return BIBO_ERR_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (p == nullptr) return (int)hipErrorInvalidSymbol;
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return BIBO_OK;
}

constexpr size_t kAlign = 256;
inline size_t align_up(size_t v) { return (v + kAlign - 1) & ~(kAlign - 1); }
inline size_t elt_size(int dtype) { return dtype == BIBO_DTYPE_BF16 ? 2 : 4; }
inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
inline bool aligned_ws(const void* p) { return (reinterpret_cast<uintptr_t>(p) & (kAlign - 1)) == 0; }

inline Vec vec(const void* p, int dtype) { return Vec{p, dtype == BIBO_DTYPE_BF16}; }
inline bool vec_ok(const void* p, int dtype) { return dtype != BIBO_DTYPE_BF16 || aligned16(p); }
inline bool act_ok(int act) { return act >= BIBO_ACT_RADIAL_SIGMOID && act <= BIBO_ACT_SILU; }

int check_dims(int T, int H, int E, int k, int I, int dtype, int n_pos = 0, int n_neg = 0) {
  if (n_pos < 0 || n_neg < 0 || n_pos + n_neg >= E) return BIBO_ERR_BAD_SHAPE;     // at least one GLU expert
  if (dtype != BIBO_DTYPE_BF16 && dtype != BIBO_DTYPE_F32) return BIBO_ERR_BAD_DTYPE;
  if (T < 0 || H < 1 || I < 1 || E < 1 || E > kMaxE || k < 1 || k > kMaxK || k > E) return BIBO_ERR_BAD_SHAPE;
  if ((long long)T * k > 0x3fffffffLL) return BIBO_ERR_BAD_SHAPE;
  return BIBO_OK;
}

// Rows per expert up to which `auto` resolves to the weight-streaming family by name.
inline long long stream_rows_per_expert(int H, int I, int dtype) {
  if (H <= 512 && I <= 512) return 24;
  return fused_supported(H, I, dtype) ? 10 : 17;
}

// `distinct`: the k experts of a token are known to differ (indices that come straight from the router kernel), so
// one expert gets at most T rows.  A caller's indices may name an expert several times per token, up to all T*k
// slots on one expert, and the row list of a streaming workgroup holds kStreamMaxRows entries.
// the fused kernel addresses hidden-state rows with 32-bit byte offsets
inline bool fused_fits(int T, int H) { return (long long)T * H < (1LL << 31); }

// what the streaming kernels can run: the slots fit a workgroup's scan and an expert's rows its row list
inline bool stream_possible(int T, int H, int E, int k, int I, int dtype, bool distinct) {
  return stream_supported(H, I, dtype) && (long long)T * k <= kStreamMaxSlots &&
         (distinct ? T : (long long)T * k) <= kStreamMaxRows;
}

// what `auto` gives them: few enough rows per expert that streaming beats the tile kernels
inline bool stream_eligible(int T, int H, int E, int k, int I, int dtype, bool distinct) {
  return stream_possible(T, H, E, k, I, dtype, distinct) && (long long)T * k <= stream_rows_per_expert(H, I, dtype) * E;
}

// Routed slots up to which a call that `auto` resolved to streaming does stream; beyond them the tile kernels take it under that name.  With H
// and I up to 512 a wave's 16 weight rows stay in registers for all of the expert's rows, and a further 16-row pass only costs its
// staging.  Wider rows are streamed again, from L2, for every pass of 16 that some expert needs.  Sum of the layer's kernels, streaming ->
// tiles: H = 512, I = 256, E = 64: 31 -> 31 us at 9 rows per expert with weights in the Infinity Cache, 34 -> 35 at 12 and 39 -> 36 at 18
// from HBM; E = 32: 27 -> 31 at 12, 32 -> 30 at 20; E = 16: 28 -> 30 at 20, 36 -> 29 at 36; E = 9: 24 -> 25 at 14, 30 -> 29 at 28.
// H = 1024, I = 512, E = 64: 63 -> 63 at 10, 69 -> 63 at 12, 80 -> 63 at 16; E = 9: 30 -> 34 at 11, 38 -> 34 at 14.
// Those tiles hand fp32 rows to the combine, as streaming does (f32_rows); the others' are bf16.
inline long long stream_slots(int E, int H, int I, int dtype) {
  if (H <= 512 && I <= 512) return 24 * E < 704 ? 24 * E : 704;
  return (fused_wide_supported(H, I, dtype) ? 11LL : 17LL) * E;
}

// What `auto` runs in a composite call under the name of a family: the fused kernel on shorter tiles where it resolves to the
// MFMA family at I = 512 (H = 1024, T = 3001, k = 8: 199 -> 167 us), and the fused kernel's two halves with a tile's columns cut over
// several workgroups where there are few tiles (split_columns).  An explicit request for a family runs the kernels its stage
// calls run, whose results they repeat bit for bit.
constexpr int kAlgoFusedWide = 100, kAlgoSplit = 101;
inline int composite_algo(bool automatic, int resolved, int T, int H, int E, int k, int I, int dtype) {
  if (!automatic) return resolved;
  const bool fits = fused_fits(T, H);
  if (resolved == BIBO_ALGO_STREAM && (long long)T * k > stream_slots(E, H, I, dtype) && fits) {
    if (fused_supported(H, I, dtype)) resolved = BIBO_ALGO_FUSED;
    else if (fused_wide_supported(H, I, dtype)) resolved = BIBO_ALGO_MFMA;
  }
  const bool wide = resolved == BIBO_ALGO_MFMA && fused_wide_supported(H, I, dtype) && fits;
  if ((wide || resolved == BIBO_ALGO_FUSED) && split_columns(T * k, E, H, I)) return kAlgoSplit;
  return wide ? kAlgoFusedWide : resolved;
}

// `composite`: the caller is bibo_moe_experts_fwd / bibo_moe_forward, the only entry points that can run
// the streaming kernels (they hand bf16 pre-activations, not `hidden`, from one kernel to the next) and
// the fused kernel (its activations never reach memory).
int resolve_algo(int algo, int T, int H, int E, int k, int I, int dtype, bool composite, bool distinct, int* out) {
  switch (algo) {
    case BIBO_ALGO_AUTO:
      if (composite && stream_eligible(T, H, E, k, I, dtype, distinct)) *out = BIBO_ALGO_STREAM;
      else if (composite && fused_supported(H, I, dtype) && fused_fits(T, H)) *out = BIBO_ALGO_FUSED;
      else *out = mfma_supported(H, I, dtype) ? BIBO_ALGO_MFMA : BIBO_ALGO_GENERIC;
      break;
    case BIBO_ALGO_GENERIC: *out = BIBO_ALGO_GENERIC; break;
    case BIBO_ALGO_MFMA:
      if (!mfma_supported(H, I, dtype)) return BIBO_ERR_UNSUPPORTED;
      *out = BIBO_ALGO_MFMA;
      break;
    case BIBO_ALGO_STREAM:
      // more rows per expert than the limit: refused here, before anything is launched
      if (!composite || !stream_possible(T, H, E, k, I, dtype, distinct)) return BIBO_ERR_UNSUPPORTED;
      *out = BIBO_ALGO_STREAM;
      break;
    case BIBO_ALGO_FUSED:
      if (!composite || !fused_supported(H, I, dtype) || !fused_fits(T, H)) return BIBO_ERR_UNSUPPORTED;
      *out = BIBO_ALGO_FUSED;
      break;
    default: return BIBO_ERR_UNSUPPORTED;
  }
  // the generic kernels keep one activation row (H + 2I floats) in LDS
  if (*out == BIBO_ALGO_GENERIC && (size_t)(H + 2 * I) * sizeof(float) > 64 * 1024) return BIBO_ERR_UNSUPPORTED;
  return BIBO_OK;
}

// Whether the generic family's fp32 tile kernels take a shape, given 16-byte aligned operands.  Their pre-activations
// [S, 2I] lie where the slot rows [S, H] go later (the last segment of the workspace).
inline bool generic_tiles(int H, int I, int dtype) {
  return tile_f32_supported(H, I) && (dtype == BIBO_DTYPE_F32 || !mfma_supported(H, I, dtype));
}

// Whether a composite call that resolved to `algo` runs the few-token kernels (experts_few.hip).  A bf16 shape of the MFMA
// families that a caller asks the generic one for does not.
inline bool few_taken(int algo, int T, int H, int k, int I, int dtype, const void* x, const void* wgu, const void* wd) {
  return few_supported(T, H, k, I) && (algo == BIBO_ALGO_STREAM || (algo == BIBO_ALGO_GENERIC && generic_tiles(H, I, dtype))) &&
         aligned16(x) && aligned16(wgu) && aligned16(wd);
}

struct Workspace {
  size_t hist, idx, w, counts, offsets, perm_slot, perm_token, hidden, gu, yw, pre;
  size_t least;        // with room for the slot rows only: what every kernel family can do with
  size_t total;
};

Workspace carve(int T, int H, int E, int k, int I, int dtype) {
  const size_t S = (size_t)T * k;
  Workspace ws;
  size_t o = 0;
  ws.hist = o;       o += align_up(permute_workspace_bytes(T) > router_hist_bytes(T) ? permute_workspace_bytes(T)
                                                                                    : router_hist_bytes(T));
  ws.idx = o;        o += align_up(S * sizeof(int32_t));
  ws.w = o;          o += align_up(S * sizeof(float));
  ws.counts = o;     o += align_up(kMaxE * sizeof(int32_t));
  ws.offsets = o;    o += align_up((kMaxE + 1) * sizeof(int32_t));
  ws.perm_slot = o;  o += align_up(S * sizeof(int32_t));
  ws.perm_token = o; o += align_up(S * sizeof(int32_t));
  ws.hidden = o;     o += align_up(S * (size_t)I * elt_size(dtype));
  // gate/up pre-activations of the few-token kernels (fp32) and of the streaming kernels (bf16), where they are eligible
  ws.gu = o;         o += align_up(few_supported(T, H, k, I) ? S * (size_t)2 * I * sizeof(float)
                                   : stream_possible(T, H, E, k, I, dtype, true) ? S * (size_t)2 * I * sizeof(bf16_t) : 0);
  ws.yw = o;
  ws.least = o + align_up(S * (size_t)H * sizeof(float));
  ws.total = o + align_up(S * (size_t)(generic_tiles(H, I, dtype) && 2 * I > H ? 2 * I : H) * sizeof(float));
  // fp32 pre-activations of a call whose tiles are cut by columns: behind its slot rows, fp32 where `auto` streamed before, else bf16
  ws.pre = o + align_up(S * (size_t)H * (stream_eligible(T, H, E, k, I, dtype, true) ? sizeof(float) : sizeof(bf16_t)));
  if (dtype == BIBO_DTYPE_BF16 && mfma_supported(H, I, dtype) && split_columns(T * k, E, H, I)) {
    const size_t end = ws.pre + align_up(S * (size_t)2 * I * sizeof(float));
    if (end > ws.total) ws.total = end;
  }
  return ws;
}

inline int hip_rc(hipError_t e) { return e == hipSuccess ? BIBO_OK : (int)e; }

int gateup_dispatch(const void* x, const void* wgu, const float* theta, const int32_t* offsets,
                    const int32_t* perm_token, int T, int H, int E, int k, int I, int dtype, int algo, int act,
                    void* hidden, hipStream_t s) {
  if (algo == BIBO_ALGO_MFMA) {
    if (!aligned16(x) || !aligned16(wgu) || !aligned16(hidden)) return BIBO_ERR_MISALIGNED;
    return hip_rc(launch_gateup_mfma(x, wgu, theta, offsets, perm_token, T, H, E, k, I, act, hidden, s));
  }
  return hip_rc(launch_gateup_generic(x, wgu, theta, offsets, perm_token, T, H, E, k, I, dtype, act, hidden, s));
}

// E here and in gateup_dispatch counts the GLU experts (those that have weights)
int down_dispatch(const void* hidden, const void* wd, const float* w, const int32_t* offsets, const int32_t* perm_slot,
                  const CombineArgs& ca, int T, int H, int E, int k, int I, int dtype, int algo, void* out, float* yw,
                  hipStream_t s) {
  hipError_t e;
  if (algo == BIBO_ALGO_MFMA) {
    if (!aligned16(hidden) || !aligned16(wd)) return BIBO_ERR_MISALIGNED;
    // weighted expert outputs travel to the combine in bf16 (the reference's bf16 eager path rounds each
    // expert output to bf16 as well, moe.py:92)
    e = launch_down_mfma(hidden, wd, w, offsets, perm_slot, T, H, E, k, I, yw, s);
    if (e != hipSuccess) return (int)e;
    return hip_rc(launch_combine(yw, 1, ca, T, H, k, dtype, out, s));
  }
  e = launch_down_generic(hidden, wd, w, offsets, perm_slot, T, H, E, k, I, dtype, yw, s);
  if (e != hipSuccess) return (int)e;
  return hip_rc(launch_combine(yw, 0, ca, T, H, k, dtype, out, s));
}

// kernels 3 and 4 (+ combine) after the permutation, for the composite entry points
// Eg = GLU experts (with weights), np / nn = +/-Identity specials behind them (moe.py:39-44).
int experts_dispatch(const void* x, const void* wgu, const void* wd, const float* theta, const int32_t* idx,
                     const float* w, const int32_t* offsets, const int32_t* perm_slot, const int32_t* perm_token,
                     const void* residual, bool idx_trusted, int T, int H, int Eg, int np, int nn, int k, int I, int dtype,
                     int algo, int act, int flags, void* out, char* base, const Workspace& ws, size_t ws_bytes,
                     hipStream_t s, bool f32_rows = false, void* preact = nullptr, const ScanArgs& scan = ScanArgs(),
                     bool gate_up_done = false, float* keep_gu = nullptr, const BalanceArgs& balance = BalanceArgs()) {
  float* yw = reinterpret_cast<float*>(base + ws.yw);
  CombineArgs ca;
  ca.balance = balance;
  ca.residual = residual;
  ca.round_block = (residual != nullptr && (flags & BIBO_FLAG_ROUND_BLOCK_OUT)) ? 1 : 0;   // layers.py:62-63
  // indices that come straight from the router kernel are in range; a caller's may hold padding values, whose
  // slots the combine has to skip; specials are the combine's work either way (moe.py:95-99)
  if (!idx_trusted || np + nn > 0) { ca.idx = idx; ca.w = w; ca.x = x; ca.E_glu = Eg; ca.n_pos = np; ca.n_neg = nn; }
  if (few_taken(algo, T, H, k, I, dtype, x, wgu, wd)) {
    ca.x = x; ca.n_pos = np; ca.n_neg = nn;
    const hipError_t e = launch_experts_few(x, wgu, wd, theta, idx, w, ca, T, H, Eg, k, I, dtype, act, reinterpret_cast<float*>(base + ws.gu),
                                            out, gate_up_done, s);
    return hip_rc(e == hipSuccess && balance.counts != nullptr ? launch_balance_step(balance, s) : e);
  }
  if (algo == BIBO_ALGO_STREAM) {
    if (!aligned16(x) || !aligned16(wgu) || !aligned16(wd)) return BIBO_ERR_MISALIGNED;
    if (!stream_possible(T, H, Eg + np + nn, k, I, dtype, idx_trusted)) return BIBO_ERR_UNSUPPORTED;   // no pre-activation segment carved, or more rows than a row list holds
    void* gu = base + ws.gu;
    hipError_t e = launch_gateup_stream(x, wgu, idx, T, H, Eg, k, I, gu, s);
    if (e != hipSuccess) return (int)e;
    e = launch_down_stream(gu, wd, theta, w, idx, T, H, Eg, k, I, act, base + ws.hidden, yw, s);
    if (e != hipSuccess) return (int)e;
    return hip_rc(launch_combine(yw, 0, ca, T, H, k, dtype, out, s));
  }
  if (algo == kAlgoSplit) {
    if (!aligned16(x) || !aligned16(wgu) || !aligned16(wd)) return BIBO_ERR_MISALIGNED;
    void* pre = base + ws.pre;
    hipError_t e = launch_gateup_raw(x, wgu, offsets, perm_token, T, H, Eg, k, I, pre, true, true, s, scan);
    if (e != hipSuccess) return (int)e;
    if ((e = launch_down_act(pre, wd, theta, w, offsets, perm_slot, T * k, H, Eg, I, act, yw, f32_rows, preact, s)) != hipSuccess)
      return (int)e;
    return hip_rc(launch_combine(yw, f32_rows ? 0 : 1, ca, T, H, k, dtype, out, s));
  }
  if (algo == BIBO_ALGO_FUSED || algo == kAlgoFusedWide) {
    if (!aligned16(x) || !aligned16(wgu) || !aligned16(wd)) return BIBO_ERR_MISALIGNED;
    hipError_t e = launch_experts_fused(x, wgu, wd, theta, w, offsets, perm_slot, perm_token, T, H, Eg, k, I, act, yw, f32_rows, preact, s,
                                        scan);
    if (e != hipSuccess) return (int)e;
    return hip_rc(launch_combine(yw, f32_rows ? 0 : 1, ca, T, H, k, dtype, out, s));
  }
  // (a bf16 shape of the MFMA families that a caller asks the generic one for runs the row kernels, like the stage calls)
  if (algo == BIBO_ALGO_GENERIC && generic_tiles(H, I, dtype) && aligned16(x) && aligned16(wgu) && aligned16(wd) &&
      ws_bytes >= ws.total) {
    hipError_t e = launch_experts_tiled(x, wgu, wd, theta, w, offsets, perm_slot, perm_token, T, H, Eg, k, I, dtype, act,
                                        keep_gu != nullptr ? keep_gu : yw, base + ws.hidden, yw, s);
    if (e != hipSuccess) return (int)e;
    return hip_rc(launch_combine(yw, 0, ca, T, H, k, dtype, out, s));
  }
  const int rc = gateup_dispatch(x, wgu, theta, offsets, perm_token, T, H, Eg, k, I, dtype, algo, act, base + ws.hidden, s);
  if (rc != BIBO_OK) return rc;
  return down_dispatch(base + ws.hidden, wd, w, offsets, perm_slot, ca, T, H, Eg, k, I, dtype, algo, out, yw, s);
}

// What a training forward leaves for its backward pass in a caller-owned buffer: the routing (selection, combine
// weights, fp32 logits), the permutation and, of every routed row, the gate/up pre-activations: in bf16 where the fused forward kernel
// and the MFMA backward both take the shape; where a caller asks for every shape, in fp32 if the tile kernels of the generic family run,
// whose forward has them in memory anyway, and else none.
enum class Keeps { kNothing, kBf16, kF32, kRouting };

Keeps kept_state(const bibo_moe_shape* sh) {
  const bool fast = backward_supported(sh->H, sh->I, sh->k, sh->dtype);      // the MFMA backward family
  if (fast && fused_supported(sh->H, sh->I, sh->dtype) && fused_fits(sh->T, sh->H)) return Keeps::kBf16;
  if ((sh->flags & BIBO_FLAG_KEEP_ANY) == 0) return Keeps::kNothing;
  int algo;
  const bool tiled = resolve_algo(BIBO_ALGO_AUTO, sh->T, sh->H, sh->E, sh->k, sh->I, sh->dtype, true, true, &algo) == BIBO_OK &&
                     algo == BIBO_ALGO_GENERIC && generic_tiles(sh->H, sh->I, sh->dtype) && !few_supported(sh->T, sh->H, sh->k, sh->I);
  return !fast && tiled ? Keeps::kF32 : Keeps::kRouting;
}

struct TrainState {
  size_t idx, w, logits, offsets, perm_slot, perm_token, gu, total;
};

TrainState carve_state(int T, int E, int k, int I, Keeps keeps) {
  const size_t S = (size_t)T * k;
  TrainState st;
  size_t o = 0;
  st.idx = o;        o += align_up(S * sizeof(int32_t));
  st.w = o;          o += align_up(S * sizeof(float));
  st.logits = o;     o += align_up((size_t)T * E * sizeof(float));
  st.offsets = o;    o += align_up((kMaxE + 1) * sizeof(int32_t));
  st.perm_slot = o;  o += align_up(S * sizeof(int32_t));
  st.perm_token = o; o += align_up(S * sizeof(int32_t));
  st.gu = o;         o += align_up(S * 2 * (size_t)I * (keeps == Keeps::kBf16 ? sizeof(bf16_t) : keeps == Keeps::kF32 ? sizeof(float) : 0));
  st.total = o;
  return st;
}

// The whole layer on `x`; `residual` (or NULL) is added in the combine.  With `norm_src` given, `x` is a buffer the
// router kernel first fills with RMSNorm(norm_src) (weight `norm_weight`, `eps`): the caller's seam in one read of
// the raw rows.
int forward_impl(const void* x, const void* w_router, const float* bias, const void* w_gate_up, const void* w_down,
                 const float* theta, const bibo_moe_shape* sh, int norm_mode, int algo, const void* residual, void* out,
                 int32_t* idx_out, float* w_out, int32_t* counts_out, float* logits_out, void* workspace,
                 size_t workspace_bytes, void* stream, const void* norm_src = nullptr, Vec norm_weight = Vec{nullptr, 0},
                 float eps = 0.f, char* state = nullptr, const bibo_moe_balance* moves = nullptr) {
  if (sh == nullptr) return BIBO_ERR_NULL_POINTER;
  const int T = sh->T, H = sh->H, E = sh->E, k = sh->k, I = sh->I, dtype = sh->dtype;
  int rc = check_dims(T, H, E, k, I, dtype, sh->n_pos, sh->n_neg);
  if (rc != BIBO_OK) return rc;
  const int Eg = E - sh->n_pos - sh->n_neg;
  if (norm_mode < BIBO_NORM_NONE || norm_mode > BIBO_NORM_SOFTMAX || !act_ok(sh->act)) return BIBO_ERR_UNSUPPORTED;
  int a;
  if ((rc = resolve_algo(algo, T, H, E, k, I, dtype, true, true, &a)) != BIBO_OK) return rc;
  const int resolved = a;
  a = composite_algo(algo == BIBO_ALGO_AUTO || (state != nullptr && (sh->flags & BIBO_FLAG_TRAIN_AUTO) != 0), a, T, H, E, k, I, dtype);
  const bool f32_rows = resolved == BIBO_ALGO_STREAM && a != BIBO_ALGO_STREAM;
  if (a == kAlgoSplit && workspace_bytes < carve(T, H, E, k, I, dtype).total) a = BIBO_ALGO_FUSED;
  if (!workspace) return BIBO_ERR_NULL_POINTER;
  if (!aligned_ws(workspace)) return BIBO_ERR_MISALIGNED;
  if (T > 0 && (!x || !w_router || !bias || !w_gate_up || !w_down || !out)) return BIBO_ERR_NULL_POINTER;
  if (T > 0 && !theta && sh->act != BIBO_ACT_SILU) return BIBO_ERR_NULL_POINTER;
  const Workspace ws = carve(T, H, E, k, I, dtype);
  if (workspace_bytes < ws.least) return BIBO_ERR_WORKSPACE_TOO_SMALL;
  char* base = static_cast<char*>(workspace);
  hipStream_t s = static_cast<hipStream_t>(stream);
  int32_t* idx = idx_out ? idx_out : reinterpret_cast<int32_t*>(base + ws.idx);
  float* w = w_out ? w_out : reinterpret_cast<float*>(base + ws.w);
  int32_t* counts = counts_out ? counts_out : reinterpret_cast<int32_t*>(base + ws.counts);
  int32_t* offsets = reinterpret_cast<int32_t*>(base + ws.offsets);
  int32_t* perm_slot = reinterpret_cast<int32_t*>(base + ws.perm_slot);
  int32_t* perm_token = reinterpret_cast<int32_t*>(base + ws.perm_token);
  void* preact = nullptr;
  float* keep_gu = nullptr;
  if (state != nullptr) {                // a training forward: what the backward pass needs lands in the caller's state buffer
    const Keeps keeps = kept_state(sh);
    const TrainState st = carve_state(T, E, k, I, keeps);
    idx = reinterpret_cast<int32_t*>(state + st.idx);
    w = reinterpret_cast<float*>(state + st.w);
    logits_out = reinterpret_cast<float*>(state + st.logits);
    offsets = reinterpret_cast<int32_t*>(state + st.offsets);
    perm_slot = reinterpret_cast<int32_t*>(state + st.perm_slot);
    perm_token = reinterpret_cast<int32_t*>(state + st.perm_token);
    if (keeps == Keeps::kBf16) preact = state + st.gu;
    if (keeps == Keeps::kF32) keep_gu = reinterpret_cast<float*>(state + st.gu);
  }
  // the streaming and few-token kernels find their rows themselves; the permutation then only serves the counts
  const bool few = few_taken(a, T, H, k, I, dtype, x, w_gate_up, w_down);
  const bool need_permute = (a != BIBO_ALGO_STREAM && !few) || counts_out != nullptr || state != nullptr || T == 0;
  // the router kernel can leave per-workgroup histograms of its selections, which save the permutation its
  // histogram launch and its counting pass
  int32_t* hist = reinterpret_cast<int32_t*>(base + ws.hist);
  int hist_tokens = 0;
  bool gate_up_done = false;
  // with few slots, the fused kernel and its first half find their rows themselves; of a permutation they leave what a backward pass reads
  const bool may_scan = (a == BIBO_ALGO_FUSED || a == kAlgoFusedWide || a == kAlgoSplit) && T > 0 &&
                        (long long)T * k <= (a == BIBO_ALGO_FUSED ? kScanSlots : kScanSlots / 2) &&
                        (state != nullptr ? Eg == E && (preact != nullptr || a == kAlgoSplit) : counts_out == nullptr) && aligned16(x) && aligned16(w_gate_up) && aligned16(w_down);
  const bool want_hist = may_scan || (need_permute && T > 0 && permute_takes_router_hist(T, k));
  const void* rows = norm_src != nullptr ? norm_src : x;
  void* xn = norm_src != nullptr ? const_cast<void*>(x) : nullptr;
  if (few && !want_hist && router_gateup_supported(T, H, k, I, dtype, rows, w_router)) {
    rc = hip_rc(launch_router_gateup(rows, w_router, bias, T, H, E, k, norm_mode, logits_out, idx, w, w_gate_up, Eg, I,
                                     reinterpret_cast<float*>(base + ws.gu), norm_weight, eps, xn, s));
    if (rc != BIBO_OK) return rc;
    gate_up_done = true;
  } else if (T > 0 && norm_src != nullptr) {
    rc = hip_rc(launch_router_norm(norm_src, norm_weight, eps, w_router, bias, T, H, E, k, norm_mode, xn, logits_out, idx, w,
                                   want_hist ? hist : nullptr, &hist_tokens, s));
    if (rc != BIBO_OK) return rc;
  } else if (T > 0 && (rc = hip_rc(launch_router(x, w_router, bias, T, H, E, k, dtype, norm_mode, logits_out, idx, w, nullptr,
                                                 want_hist ? hist : nullptr, &hist_tokens, s))) != BIBO_OK)
    return rc;
  ScanArgs scan;
  if (may_scan && hist_tokens == 16) {
    scan.idx = idx;
    scan.hist = hist;
    scan.nhist = (T + 15) / 16;
    scan.S = T * k;
    scan.k = k;
    scan.perm_slot = perm_slot;
    scan.offsets = offsets;
    if (state != nullptr) {
      scan.perm_token = perm_token;
      scan.counts = counts;
    }
  } else if (need_permute) {
    const hipError_t e = (want_hist && hist_tokens > 0 && permute_takes_router_hist(T, k))
                             ? launch_permute_from_hist(idx, T, E, k, hist, hist_tokens, counts, offsets, perm_slot,
                                                        perm_token, s)
                             : launch_permute(idx, T, E, k, counts, offsets, perm_slot, perm_token, hist, s);
    if (e != hipSuccess) return (int)e;
  }
  BalanceArgs balance;
  if (moves != nullptr) balance = BalanceArgs{counts, moves->accumulated, moves->bias, E, moves->factor, moves->update};
  if (T == 0) return moves != nullptr ? hip_rc(launch_balance_step(balance, s)) : BIBO_OK;
  return experts_dispatch(x, w_gate_up, w_down, theta, idx, w, offsets, perm_slot, perm_token, residual, true, T, H, Eg,
                          sh->n_pos, sh->n_neg, k, I, dtype, a, sh->act, sh->flags, out, base, ws, workspace_bytes, s, f32_rows, preact, scan,
                          gate_up_done, keep_gu, balance);
}


struct BackwardWorkspace {
  size_t hist, idx, w, logits, counts, offsets, perm_slot, perm_token, dw_slot, dl, dtheta_row, dwr_part, zrow, gu, dhp, dgu,
      hidden, dxs, wgrad_part, wgrad_plan, total;
};

BackwardWorkspace carve_backward(int T, int H, int E, int k, int I) {
  const size_t S = (size_t)T * k, b = sizeof(bf16_t);
  BackwardWorkspace ws;
  size_t o = 0;
  ws.hist = o;       o += align_up(permute_workspace_bytes(T) > router_hist_bytes(T) ? permute_workspace_bytes(T)
                                                                                    : router_hist_bytes(T));
  ws.idx = o;        o += align_up(S * sizeof(int32_t));
  ws.w = o;          o += align_up(S * sizeof(float));
  ws.logits = o;     o += align_up((size_t)T * E * sizeof(float));
  ws.counts = o;     o += align_up(kMaxE * sizeof(int32_t));
  ws.offsets = o;    o += align_up((kMaxE + 1) * sizeof(int32_t));
  ws.perm_slot = o;  o += align_up(S * sizeof(int32_t));
  ws.perm_token = o; o += align_up(S * sizeof(int32_t));
  ws.dw_slot = o;    o += align_up(S * sizeof(float));
  ws.dl = o;         o += align_up(S * sizeof(float));
  ws.dtheta_row = o; o += align_up(S * sizeof(float));
  ws.dwr_part = o;   o += align_up((size_t)backward_chunk_slots((int)S, E) * backward_dwr_split() * H * sizeof(float));
  ws.zrow = o;       o += align_up(backward_zero_row_bytes(H, I));
  ws.gu = o;         o += align_up(S * 2 * I * b);
  ws.dhp = o;        o += align_up(S * I * b);
  ws.dgu = o;        o += align_up(S * 2 * I * b);
  ws.hidden = o;     o += align_up(S * I * b);
  ws.dxs = o;        o += align_up(S * H * b);
  ws.wgrad_part = o; o += align_up(backward_wgrad_part_bytes((int)S, H, E, I));
  ws.wgrad_plan = o; o += align_up(backward_plan_bytes((int)S, E));
  ws.total = o;
  return ws;
}

// the generic family keeps its intermediates in fp32: [dg, du], w h and the per-slot dx rows
struct GenericBackwardWorkspace {
  size_t hist, idx, w, logits, counts, offsets, perm_slot, perm_token, dw_slot, dl, dtheta_row, dgu, hw, dxs, total;
};

GenericBackwardWorkspace carve_backward_generic(int T, int H, int E, int k, int I) {
  const size_t S = (size_t)T * k;
  GenericBackwardWorkspace ws;
  size_t o = 0;
  ws.hist = o;       o += align_up(permute_workspace_bytes(T) > router_hist_bytes(T) ? permute_workspace_bytes(T)
                                                                                    : router_hist_bytes(T));
  ws.idx = o;        o += align_up(S * sizeof(int32_t));
  ws.w = o;          o += align_up(S * sizeof(float));
  ws.logits = o;     o += align_up((size_t)T * E * sizeof(float));
  ws.counts = o;     o += align_up(kMaxE * sizeof(int32_t));
  ws.offsets = o;    o += align_up((kMaxE + 1) * sizeof(int32_t));
  ws.perm_slot = o;  o += align_up(S * sizeof(int32_t));
  ws.perm_token = o; o += align_up(S * sizeof(int32_t));
  ws.dw_slot = o;    o += align_up(S * sizeof(float));
  ws.dl = o;         o += align_up(S * sizeof(float));
  ws.dtheta_row = o; o += align_up(S * sizeof(float));
  ws.dgu = o;        o += align_up(S * 2 * I * sizeof(float));
  ws.hw = o;         o += align_up(S * I * sizeof(float));
  ws.dxs = o;        o += align_up(S * H * sizeof(float));
  ws.total = o;
  return ws;
}

// which backward family a shape runs: the MFMA kernels (bf16, H and I multiples of 128, I <= 512) or the generic ones
inline bool backward_fast(const bibo_moe_shape* sh) { return backward_supported(sh->H, sh->I, sh->k, sh->dtype); }

int backward_check(const bibo_moe_shape* sh, int norm_mode) {
  if (sh == nullptr) return BIBO_ERR_NULL_POINTER;
  const int rc = check_dims(sh->T, sh->H, sh->E, sh->k, sh->I, sh->dtype, sh->n_pos, sh->n_neg);
  if (rc != BIBO_OK) return rc;
  if (norm_mode < BIBO_NORM_NONE || norm_mode > BIBO_NORM_SOFTMAX || !act_ok(sh->act)) return BIBO_ERR_UNSUPPORTED;
  // the MFMA family (bf16, dimensions its tiles divide) or the generic one (a row of 2H + 5I floats within 64 KB)
  if (!backward_fast(sh) && !backward_generic_supported(sh->H, sh->I, sh->k)) return BIBO_ERR_UNSUPPORTED;
  return BIBO_OK;
}


// The MFMA backward family behind bibo_moe_backward and bibo_moe_backward_saved.  `state` (or NULL): what a training
// forward kept (routing, permutation, pre-activations); without it the routing and the permutation are computed again
// from x - same kernels, same inputs, hence the same selection and weights - and so are the pre-activations.
int backward_mfma(const void* x, const void* d_out, const void* w_router, const float* bias, const void* w_gate_up,
                  const void* w_down, const float* theta, const bibo_moe_shape* sh, int norm_mode, const char* state, void* d_x,
                  void* d_w_router, void* d_w_gate_up, void* d_w_down, float* d_theta, float* d_w_out, void* workspace,
                  size_t workspace_bytes, void* stream) {
  const int T = sh->T, H = sh->H, E = sh->E, k = sh->k, I = sh->I;
  int rc;
  if (!aligned16(x) || !aligned16(d_out) || !aligned16(w_router) || !aligned16(w_gate_up) || !aligned16(w_down) ||
      !aligned16(d_x) || !aligned16(d_w_gate_up) || !aligned16(d_w_down))
    return BIBO_ERR_MISALIGNED;
  const BackwardWorkspace ws = carve_backward(T, H, E, k, I);
  if (workspace_bytes < ws.total) return BIBO_ERR_WORKSPACE_TOO_SMALL;
  char* base = static_cast<char*>(workspace);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int32_t* idx; const float* w; const float* logits; const int32_t* offsets; const int32_t* perm_slot;
  const int32_t* perm_token; const void* gu_saved = nullptr;
  if (state != nullptr) {
    const Keeps keeps = kept_state(sh);
    const TrainState st = carve_state(T, E, k, I, keeps);
    idx = reinterpret_cast<const int32_t*>(state + st.idx);
    w = reinterpret_cast<const float*>(state + st.w);
    logits = reinterpret_cast<const float*>(state + st.logits);
    offsets = reinterpret_cast<const int32_t*>(state + st.offsets);
    perm_slot = reinterpret_cast<const int32_t*>(state + st.perm_slot);
    perm_token = reinterpret_cast<const int32_t*>(state + st.perm_token);
    if (keeps == Keeps::kBf16) gu_saved = state + st.gu;
  } else {
    int32_t* idx_w = reinterpret_cast<int32_t*>(base + ws.idx);
    float* w_w = reinterpret_cast<float*>(base + ws.w);
    float* logits_w = reinterpret_cast<float*>(base + ws.logits);
    int32_t* counts = reinterpret_cast<int32_t*>(base + ws.counts);
    int32_t* offsets_w = reinterpret_cast<int32_t*>(base + ws.offsets);
    int32_t* slot_w = reinterpret_cast<int32_t*>(base + ws.perm_slot);
    int32_t* token_w = reinterpret_cast<int32_t*>(base + ws.perm_token);
    // (the router kernel leaves per-workgroup histograms of its selections for the permutation, as in the forward pass)
    int32_t* hist = reinterpret_cast<int32_t*>(base + ws.hist);
    int hist_tokens = 0;
    const bool want_hist = T > 0 && permute_takes_router_hist(T, k);
    if (T > 0 && (rc = hip_rc(launch_router(x, w_router, bias, T, H, E, k, sh->dtype, norm_mode, logits_w, idx_w, w_w, nullptr,
                                            want_hist ? hist : nullptr, &hist_tokens, s))) != BIBO_OK)
      return rc;
    rc = hip_rc((want_hist && hist_tokens > 0)
                    ? launch_permute_from_hist(idx_w, T, E, k, hist, hist_tokens, counts, offsets_w, slot_w, token_w, s)
                    : launch_permute(idx_w, T, E, k, counts, offsets_w, slot_w, token_w, hist, s));
    if (rc != BIBO_OK) return rc;
    idx = idx_w; w = w_w; logits = logits_w; offsets = offsets_w; perm_slot = slot_w; perm_token = token_w;
  }
  BackwardBuffers b;
  b.gu = base + ws.gu; b.dhp = base + ws.dhp; b.dgu = base + ws.dgu;
  b.hidden = base + ws.hidden; b.dxs = base + ws.dxs; b.zrow = base + ws.zrow;
  b.dw_slot = d_w_out ? d_w_out : reinterpret_cast<float*>(base + ws.dw_slot);
  b.dl = reinterpret_cast<float*>(base + ws.dl);
  b.dtheta_row = reinterpret_cast<float*>(base + ws.dtheta_row);
  b.dwr_part = reinterpret_cast<float*>(base + ws.dwr_part);
  b.wgrad_part = reinterpret_cast<float*>(base + ws.wgrad_part);
  b.wgrad_plan = reinterpret_cast<int*>(base + ws.wgrad_plan);
  return hip_rc(launch_backward(x, d_out, w_router, w_gate_up, w_down, theta, logits, idx, w, offsets, perm_slot, perm_token,
                                T, H, E - sh->n_pos - sh->n_neg, sh->n_pos, sh->n_neg, k, I, norm_mode, sh->act, b, d_x,
                                d_w_router, d_w_gate_up, d_w_down, d_theta, (sh->flags & BIBO_FLAG_GRAD_F32) != 0, s, gu_saved));
}

// The generic family, likewise.
int backward_generic(const void* x, const void* d_out, const void* w_router, const float* bias, const void* w_gate_up, const void* w_down,
                     const float* theta, const bibo_moe_shape* sh, int norm_mode, const char* state, void* d_x, void* d_w_router,
                     void* d_w_gate_up, void* d_w_down, float* d_theta, float* d_w_out, void* workspace, size_t workspace_bytes,
                     void* stream) {
  const int T = sh->T, H = sh->H, E = sh->E, k = sh->k, I = sh->I;
  const GenericBackwardWorkspace ws = carve_backward_generic(T, H, E, k, I);
  if (workspace_bytes < ws.total) return BIBO_ERR_WORKSPACE_TOO_SMALL;
  char* base = static_cast<char*>(workspace);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int32_t* idx; const float* w; const float* logits; const int32_t* offsets; const int32_t* perm_slot; const int32_t* perm_token;
  GenericBackwardBuffers b;
  if (state != nullptr) {
    const Keeps keeps = kept_state(sh);
    const TrainState st = carve_state(T, E, k, I, keeps);
    idx = reinterpret_cast<const int32_t*>(state + st.idx);
    w = reinterpret_cast<const float*>(state + st.w);
    logits = reinterpret_cast<const float*>(state + st.logits);
    offsets = reinterpret_cast<const int32_t*>(state + st.offsets);
    perm_slot = reinterpret_cast<const int32_t*>(state + st.perm_slot);
    perm_token = reinterpret_cast<const int32_t*>(state + st.perm_token);
    if (keeps == Keeps::kF32) b.gu_saved = reinterpret_cast<const float*>(state + st.gu);
  } else {
    int32_t* idx_w = reinterpret_cast<int32_t*>(base + ws.idx);
    float* w_w = reinterpret_cast<float*>(base + ws.w);
    float* logits_w = reinterpret_cast<float*>(base + ws.logits);
    int32_t* offsets_w = reinterpret_cast<int32_t*>(base + ws.offsets);
    int32_t* slot_w = reinterpret_cast<int32_t*>(base + ws.perm_slot);
    int32_t* token_w = reinterpret_cast<int32_t*>(base + ws.perm_token);
    int32_t* counts = reinterpret_cast<int32_t*>(base + ws.counts);
    int32_t* hist = reinterpret_cast<int32_t*>(base + ws.hist);
    int hist_tokens = 0, rc;
    const bool want_hist = T > 0 && permute_takes_router_hist(T, k);
    if (T > 0 && (rc = hip_rc(launch_router(x, w_router, bias, T, H, E, k, sh->dtype, norm_mode, logits_w, idx_w, w_w, nullptr,
                                            want_hist ? hist : nullptr, &hist_tokens, s))) != BIBO_OK)
      return rc;
    if ((rc = hip_rc((want_hist && hist_tokens > 0)
                         ? launch_permute_from_hist(idx_w, T, E, k, hist, hist_tokens, counts, offsets_w, slot_w, token_w, s)
                         : launch_permute(idx_w, T, E, k, counts, offsets_w, slot_w, token_w, hist, s))) != BIBO_OK)
      return rc;
    idx = idx_w; w = w_w; logits = logits_w; offsets = offsets_w; perm_slot = slot_w; perm_token = token_w;
  }
  b.dgu = reinterpret_cast<float*>(base + ws.dgu); b.hw = reinterpret_cast<float*>(base + ws.hw);
  b.dxs = reinterpret_cast<float*>(base + ws.dxs);
  b.dw_slot = d_w_out ? d_w_out : reinterpret_cast<float*>(base + ws.dw_slot);
  b.dl = reinterpret_cast<float*>(base + ws.dl); b.dtheta_row = reinterpret_cast<float*>(base + ws.dtheta_row);
  return hip_rc(launch_backward_generic(x, d_out, w_router, w_gate_up, w_down, theta, logits, idx, w, offsets, perm_slot, perm_token, T, H,
                                        E - sh->n_pos - sh->n_neg, sh->n_pos, sh->n_neg, k, I, sh->dtype, norm_mode, sh->act, b, d_x,
                                        d_w_router, d_w_gate_up, d_w_down, d_theta, (sh->flags & BIBO_FLAG_GRAD_F32) != 0, s));
}

}  // namespace

extern "C" {

int bibo_moe_abi_version(void) { return BIBO_MOE_ABI_VERSION; }

const char* bibo_moe_strerror(int code) {
  switch (code) {
    case BIBO_OK: return "success";
    case BIBO_ERR_NULL_POINTER: return "a required pointer is NULL";
    case BIBO_ERR_BAD_SHAPE:
      return "bad shape: need T >= 0, H, I >= 1, 1 <= E <= 64, 1 <= k <= min(E, 8), n_pos, n_neg >= 0, n_pos + n_neg < E";
    case BIBO_ERR_BAD_DTYPE: return "dtype must be BIBO_DTYPE_BF16 or BIBO_DTYPE_F32";
    case BIBO_ERR_WORKSPACE_TOO_SMALL: return "workspace smaller than bibo_moe_workspace_bytes() for this shape";
    case BIBO_ERR_MISALIGNED: return "tensor base pointers must be 16-byte aligned and the workspace 256-byte aligned";
    case BIBO_ERR_UNSUPPORTED: return "requested kernel family does not support this shape or dtype";
    case BIBO_ERR_STATIC_SCRATCH:
      return "shape needs more workspace than the static scratch array holds (BIBO_MOE_STATIC_SCRATCH_BYTES = 16 MiB); "
             "use bibo_moe_forward with a caller-owned workspace";
    default: break;
  }
  if (code > 0) return hipGetErrorString((hipError_t)code);
  return "unknown error code";
}

int bibo_moe_workspace_bytes(const bibo_moe_shape* sh, size_t* bytes) {
  if (sh == nullptr || bytes == nullptr) return BIBO_ERR_NULL_POINTER;
  const int rc = check_dims(sh->T, sh->H, sh->E, sh->k, sh->I, sh->dtype, sh->n_pos, sh->n_neg);
  if (rc != BIBO_OK) return rc;
  *bytes = carve(sh->T, sh->H, sh->E, sh->k, sh->I, sh->dtype).total;
  return BIBO_OK;
}

int bibo_moe_select_algo(const bibo_moe_shape* sh, int algo, int* selected) {
  if (sh == nullptr || selected == nullptr) return BIBO_ERR_NULL_POINTER;
  const int rc = check_dims(sh->T, sh->H, sh->E, sh->k, sh->I, sh->dtype, sh->n_pos, sh->n_neg);
  if (rc != BIBO_OK) return rc;
  return resolve_algo(algo, sh->T, sh->H, sh->E, sh->k, sh->I, sh->dtype, true, true, selected);
}

int bibo_moe_router_fwd(const void* x, const void* w_router, const float* bias, int T, int H, int E, int k, int dtype,
                        int norm_mode, float* logits, int32_t* idx, float* w, float* gap, void* stream) {
  const int rc = check_dims(T, H, E, k, 1, dtype);
  if (rc != BIBO_OK) return rc;
  if (norm_mode < BIBO_NORM_NONE || norm_mode > BIBO_NORM_SOFTMAX) return BIBO_ERR_UNSUPPORTED;
  if (T == 0) return BIBO_OK;
  if (!x || !w_router || !bias || !idx || !w) return BIBO_ERR_NULL_POINTER;
  return hip_rc(launch_router(x, w_router, bias, T, H, E, k, dtype, norm_mode, logits, idx, w, gap, nullptr, nullptr,
                              static_cast<hipStream_t>(stream)));
}

int bibo_moe_permute(const int32_t* idx, int T, int E, int k, int32_t* counts, int32_t* offsets, int32_t* perm_slot,
                     int32_t* perm_token, void* workspace, size_t workspace_bytes, void* stream) {
  const int rc = check_dims(T, 1, E, k, 1, BIBO_DTYPE_BF16);
  if (rc != BIBO_OK) return rc;
  if (!counts || !offsets || !workspace) return BIBO_ERR_NULL_POINTER;
  if (T > 0 && (!idx || !perm_slot || !perm_token)) return BIBO_ERR_NULL_POINTER;
  if (workspace_bytes < permute_workspace_bytes(T)) return BIBO_ERR_WORKSPACE_TOO_SMALL;
  return hip_rc(launch_permute(idx, T, E, k, counts, offsets, perm_slot, perm_token, workspace,
                               static_cast<hipStream_t>(stream)));
}

int bibo_moe_gateup_fwd(const void* x, const void* w_gate_up, const float* theta, const int32_t* offsets,
                        const int32_t* perm_token, int T, int H, int E, int k, int I, int dtype, int algo, int act,
                        void* hidden, void* stream) {
  int rc = check_dims(T, H, E, k, I, dtype);
  if (rc != BIBO_OK) return rc;
  if (!act_ok(act)) return BIBO_ERR_UNSUPPORTED;
  int a;
  if ((rc = resolve_algo(algo, T, H, E, k, I, dtype, false, false, &a)) != BIBO_OK) return rc;
  if (T == 0) return BIBO_OK;
  if (!x || !w_gate_up || (!theta && act != BIBO_ACT_SILU) || !offsets || !perm_token || !hidden) return BIBO_ERR_NULL_POINTER;
  return gateup_dispatch(x, w_gate_up, theta, offsets, perm_token, T, H, E, k, I, dtype, a, act, hidden,
                         static_cast<hipStream_t>(stream));
}

int bibo_moe_down_combine_fwd(const void* hidden, const void* w_down, const float* w, const int32_t* offsets,
                              const int32_t* perm_slot, int T, int H, int E, int k, int I, int dtype, int algo,
                              void* out, void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_dims(T, H, E, k, I, dtype);
  if (rc != BIBO_OK) return rc;
  int a;
  if ((rc = resolve_algo(algo, T, H, E, k, I, dtype, false, false, &a)) != BIBO_OK) return rc;
  if (T == 0) return BIBO_OK;
  if (!hidden || !w_down || !w || !offsets || !perm_slot || !out || !workspace) return BIBO_ERR_NULL_POINTER;
  if (!aligned_ws(workspace)) return BIBO_ERR_MISALIGNED;       // the slot rows live there, 16 bytes at a time
  if (workspace_bytes < (size_t)T * k * H * sizeof(float)) return BIBO_ERR_WORKSPACE_TOO_SMALL;
  return down_dispatch(hidden, w_down, w, offsets, perm_slot, CombineArgs{}, T, H, E, k, I, dtype, a, out,
                       static_cast<float*>(workspace), static_cast<hipStream_t>(stream));
}

int bibo_moe_gateup_down_fwd(const void* x, const void* w_gate_up, const void* w_down, const float* theta,
                             const float* w, const int32_t* offsets, const int32_t* perm_slot,
                             const int32_t* perm_token, int T, int H, int E, int k, int I, int dtype, int act,
                             void* yw, void* stream) {
  const int rc = check_dims(T, H, E, k, I, dtype);
  if (rc != BIBO_OK) return rc;
  if (!fused_supported(H, I, dtype) || !fused_fits(T, H) || !act_ok(act)) return BIBO_ERR_UNSUPPORTED;
  if (T == 0) return BIBO_OK;
  if (!x || !w_gate_up || !w_down || (!theta && act != BIBO_ACT_SILU) || !w || !offsets || !perm_slot || !perm_token || !yw)
    return BIBO_ERR_NULL_POINTER;
  if (!aligned16(x) || !aligned16(w_gate_up) || !aligned16(w_down) || !aligned16(yw)) return BIBO_ERR_MISALIGNED;
  return hip_rc(launch_experts_fused(x, w_gate_up, w_down, theta, w, offsets, perm_slot, perm_token, T, H, E, k, I, act,
                                     yw, false, nullptr, static_cast<hipStream_t>(stream)));
}

int bibo_moe_combine_fwd(const void* yw, int yw_is_bf16, int T, int H, int k, int dtype, void* out, void* stream) {
  const int rc = check_dims(T, H, k, k, 1, dtype);   // no expert dimension here: E := k, I := 1 pass the range checks
  if (rc != BIBO_OK) return rc;
  if (yw_is_bf16 && dtype != BIBO_DTYPE_BF16) return BIBO_ERR_BAD_DTYPE;
  if (T == 0) return BIBO_OK;
  if (!yw || !out) return BIBO_ERR_NULL_POINTER;
  return hip_rc(launch_combine(yw, yw_is_bf16 ? 1 : 0, CombineArgs{}, T, H, k, dtype, out, static_cast<hipStream_t>(stream)));
}

int bibo_moe_combine_ex_fwd(const void* yw, int yw_is_bf16, const int32_t* idx, const float* w, const void* x, int E_glu,
                            int n_pos, int n_neg, const void* residual, int T, int H, int k, int dtype, void* out,
                            void* stream) {
  const int rc = check_dims(T, H, k, k, 1, dtype);   // no expert dimension here: E := k, I := 1 pass the range checks
  if (rc != BIBO_OK) return rc;
  if (yw_is_bf16 && dtype != BIBO_DTYPE_BF16) return BIBO_ERR_BAD_DTYPE;
  if (E_glu < 0 || n_pos < 0 || n_neg < 0 || E_glu + n_pos + n_neg > kMaxE) return BIBO_ERR_BAD_SHAPE;
  if (T == 0) return BIBO_OK;
  if (!yw || !out) return BIBO_ERR_NULL_POINTER;
  if (n_pos + n_neg > 0 && (!idx || !w || !x)) return BIBO_ERR_NULL_POINTER;
  CombineArgs ca;
  ca.idx = idx; ca.w = w; ca.x = x; ca.E_glu = E_glu; ca.n_pos = n_pos; ca.n_neg = n_neg; ca.residual = residual;
  return hip_rc(launch_combine(yw, yw_is_bf16 ? 1 : 0, ca, T, H, k, dtype, out, static_cast<hipStream_t>(stream)));
}

int bibo_moe_experts_fwd(const void* x, const int32_t* idx, const float* w, const void* w_gate_up, const void* w_down,
                         const float* theta, const bibo_moe_shape* sh, int algo, void* out, int32_t* counts_out,
                         void* workspace, size_t workspace_bytes, void* stream) {
  if (sh == nullptr) return BIBO_ERR_NULL_POINTER;
  const int T = sh->T, H = sh->H, E = sh->E, k = sh->k, I = sh->I, dtype = sh->dtype;
  int rc = check_dims(T, H, E, k, I, dtype, sh->n_pos, sh->n_neg);
  if (rc != BIBO_OK) return rc;
  const int Eg = E - sh->n_pos - sh->n_neg;
  if (!act_ok(sh->act)) return BIBO_ERR_UNSUPPORTED;
  int a;
  // a caller's indices may repeat an expert inside a token (moe.py:46-71 accepts that)
  if ((rc = resolve_algo(algo, T, H, E, k, I, dtype, true, false, &a)) != BIBO_OK) return rc;
  const int resolved = a;
  a = composite_algo(algo == BIBO_ALGO_AUTO, a, T, H, E, k, I, dtype);
  const bool f32_rows = resolved == BIBO_ALGO_STREAM && a != BIBO_ALGO_STREAM;
  if (a == kAlgoSplit && workspace_bytes < carve(T, H, E, k, I, dtype).total) a = BIBO_ALGO_FUSED;
  if (!workspace) return BIBO_ERR_NULL_POINTER;
  if (!aligned_ws(workspace)) return BIBO_ERR_MISALIGNED;
  if (T > 0 && (!x || !idx || !w || !w_gate_up || !w_down || !out)) return BIBO_ERR_NULL_POINTER;
  if (T > 0 && !theta && sh->act != BIBO_ACT_SILU) return BIBO_ERR_NULL_POINTER;
  const Workspace ws = carve(T, H, E, k, I, dtype);
  if (workspace_bytes < ws.least) return BIBO_ERR_WORKSPACE_TOO_SMALL;
  char* base = static_cast<char*>(workspace);
  hipStream_t s = static_cast<hipStream_t>(stream);
  int32_t* counts = counts_out ? counts_out : reinterpret_cast<int32_t*>(base + ws.counts);
  int32_t* offsets = reinterpret_cast<int32_t*>(base + ws.offsets);
  int32_t* perm_slot = reinterpret_cast<int32_t*>(base + ws.perm_slot);
  int32_t* perm_token = reinterpret_cast<int32_t*>(base + ws.perm_token);
  // the streaming and few-token kernels find their rows themselves; the permutation then only serves the counts
  const bool need_permute = (a != BIBO_ALGO_STREAM && !few_taken(a, T, H, k, I, dtype, x, w_gate_up, w_down)) ||
                            counts_out != nullptr || T == 0;
  if (need_permute &&
      (rc = hip_rc(launch_permute(idx, T, E, k, counts, offsets, perm_slot, perm_token, base + ws.hist, s))) != BIBO_OK)
    return rc;
  if (T == 0) return BIBO_OK;
  return experts_dispatch(x, w_gate_up, w_down, theta, idx, w, offsets, perm_slot, perm_token, nullptr, false, T, H, Eg,
                          sh->n_pos, sh->n_neg, k, I, dtype, a, sh->act, 0, out, base, ws, workspace_bytes, s, f32_rows);
}

int bibo_moe_forward(const void* x, const void* w_router, const float* bias, const void* w_gate_up, const void* w_down,
                     const float* theta, const bibo_moe_shape* sh, int norm_mode, int algo, void* out, int32_t* idx_out,
                     float* w_out, int32_t* counts_out, float* logits_out, void* workspace, size_t workspace_bytes,
                     void* stream) {
  return forward_impl(x, w_router, bias, w_gate_up, w_down, theta, sh, norm_mode, algo, nullptr, out, idx_out, w_out,
                      counts_out, logits_out, workspace, workspace_bytes, stream);
}

int bibo_moe_forward_static(const void* x, const void* w_router, const float* bias, const void* w_gate_up,
                            const void* w_down, const float* theta, const bibo_moe_shape* sh, int norm_mode, int algo,
                            void* out, int32_t* idx_out, float* w_out, int32_t* counts_out, float* logits_out,
                            void* stream) {
  if (sh == nullptr) return BIBO_ERR_NULL_POINTER;
  int rc = check_dims(sh->T, sh->H, sh->E, sh->k, sh->I, sh->dtype, sh->n_pos, sh->n_neg);
  if (rc != BIBO_OK) return rc;
  if (carve(sh->T, sh->H, sh->E, sh->k, sh->I, sh->dtype).least > (size_t)BIBO_MOE_STATIC_SCRATCH_BYTES)
    return BIBO_ERR_STATIC_SCRATCH;
  void* ws = nullptr;
  if ((rc = static_scratch(&ws)) != BIBO_OK) return rc;
  return forward_impl(x, w_router, bias, w_gate_up, w_down, theta, sh, norm_mode, algo, nullptr, out, idx_out, w_out,
                      counts_out, logits_out, ws, (size_t)BIBO_MOE_STATIC_SCRATCH_BYTES, stream);
}

int bibo_moe_rmsnorm_fwd(const void* x, const float* norm_weight, float eps, int T, int H, int dtype, void* out,
                         void* stream) {
  const int rc = check_dims(T, H, 1, 1, 1, dtype);
  if (rc != BIBO_OK) return rc;
  if (T == 0) return BIBO_OK;
  if (!x || !norm_weight || !out) return BIBO_ERR_NULL_POINTER;
  return hip_rc(launch_rmsnorm(x, vec(norm_weight, BIBO_DTYPE_F32), eps, T, H, dtype, out, static_cast<hipStream_t>(stream)));
}

int bibo_moe_ffn_workspace_bytes(const bibo_moe_shape* sh, size_t* out) {
  if (sh == nullptr || out == nullptr) return BIBO_ERR_NULL_POINTER;
  const int rc = check_dims(sh->T, sh->H, sh->E, sh->k, sh->I, sh->dtype, sh->n_pos, sh->n_neg);
  if (rc != BIBO_OK) return rc;
  *out = carve(sh->T, sh->H, sh->E, sh->k, sh->I, sh->dtype).total + align_up((size_t)sh->T * sh->H * elt_size(sh->dtype));
  return BIBO_OK;
}

int bibo_moe_ffn_forward(const void* h, const float* norm_weight, float eps, const void* residual, const void* w_router,
                         const float* bias, const void* w_gate_up, const void* w_down, const float* theta, const bibo_moe_shape* sh,
                         int norm_mode, int algo, void* out, int32_t* idx_out, float* w_out, int32_t* counts_out,
                         void* workspace, size_t workspace_bytes, void* stream) {
  if (sh == nullptr) return BIBO_ERR_NULL_POINTER;
  const int rc = check_dims(sh->T, sh->H, sh->E, sh->k, sh->I, sh->dtype, sh->n_pos, sh->n_neg);
  if (rc != BIBO_OK) return rc;
  if (!workspace) return BIBO_ERR_NULL_POINTER;
  if (!aligned_ws(workspace)) return BIBO_ERR_MISALIGNED;
  if (sh->T > 0 && (!h || !norm_weight || !out)) return BIBO_ERR_NULL_POINTER;
  const Vec nw = vec(norm_weight, (sh->flags & BIBO_FLAG_NORM_BF16) ? BIBO_DTYPE_BF16 : BIBO_DTYPE_F32);
  if (nw.bf16 && !aligned16(norm_weight)) return BIBO_ERR_MISALIGNED;
  const size_t inner = carve(sh->T, sh->H, sh->E, sh->k, sh->I, sh->dtype).total;
  const size_t xn_bytes = align_up((size_t)sh->T * sh->H * elt_size(sh->dtype));
  if (workspace_bytes < inner + xn_bytes) return BIBO_ERR_WORKSPACE_TOO_SMALL;
  void* xn = static_cast<char*>(workspace) + inner;              // post_attention_layernorm(h), layers.py:60
  // what the block's output is added to: h itself (layers.py:62-64), another tensor, or nothing
  const void* res = (sh->flags & BIBO_FLAG_NO_RESIDUAL) ? nullptr : (residual != nullptr ? residual : h);
  if (sh->T > 0 && w_router != nullptr && router_norm_supported(sh->H, sh->dtype, h, w_router, xn))
    // the router kernel normalises the rows it reads and leaves them in xn: no norm launch, one read of h
    return forward_impl(xn, w_router, bias, w_gate_up, w_down, theta, sh, norm_mode, algo, res, out, idx_out, w_out,
                        counts_out, nullptr, workspace, inner, stream, h, nw, eps);
  const hipError_t e = launch_rmsnorm(h, nw, eps, sh->T, sh->H, sh->dtype, xn, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return (int)e;
  return forward_impl(xn, w_router, bias, w_gate_up, w_down, theta, sh, norm_mode, algo, res, out, idx_out, w_out,
                      counts_out, nullptr, workspace, inner, stream);
}

int bibo_moe_backward_workspace_bytes(const bibo_moe_shape* sh, size_t* bytes) {
  if (bytes == nullptr) return BIBO_ERR_NULL_POINTER;
  const int rc = backward_check(sh, BIBO_NORM_SUM);
  if (rc != BIBO_OK) return rc;
  *bytes = backward_fast(sh) ? carve_backward(sh->T, sh->H, sh->E, sh->k, sh->I).total
                             : carve_backward_generic(sh->T, sh->H, sh->E, sh->k, sh->I).total;
  return BIBO_OK;
}

int bibo_moe_backward(const void* x, const void* d_out, const void* w_router, const float* bias, const void* w_gate_up,
                      const void* w_down, const float* theta, const bibo_moe_shape* sh, int norm_mode, void* d_x,
                      void* d_w_router, void* d_w_gate_up, void* d_w_down, float* d_theta, float* d_w_out,
                      void* workspace, size_t workspace_bytes, void* stream) {
  const int rc = backward_check(sh, norm_mode);
  if (rc != BIBO_OK) return rc;
  const int T = sh->T;
  if (!workspace) return BIBO_ERR_NULL_POINTER;
  if (!aligned_ws(workspace)) return BIBO_ERR_MISALIGNED;
  if (!d_w_router || !d_w_gate_up || !d_w_down || !d_theta) return BIBO_ERR_NULL_POINTER;
  if (T > 0 && (!x || !d_out || !w_router || !bias || !w_gate_up || !w_down || !d_x)) return BIBO_ERR_NULL_POINTER;
  if (T > 0 && !theta && sh->act != BIBO_ACT_SILU) return BIBO_ERR_NULL_POINTER;
  if (!backward_fast(sh)) {
    return backward_generic(x, d_out, w_router, bias, w_gate_up, w_down, theta, sh, norm_mode, nullptr, d_x, d_w_router, d_w_gate_up,
                            d_w_down, d_theta, d_w_out, workspace, workspace_bytes, stream);
  }
  return backward_mfma(x, d_out, w_router, bias, w_gate_up, w_down, theta, sh, norm_mode, nullptr, d_x, d_w_router,
                       d_w_gate_up, d_w_down, d_theta, d_w_out, workspace, workspace_bytes, stream);
}

int bibo_moe_train_state_bytes(const bibo_moe_shape* sh, size_t* bytes) {
  if (bytes == nullptr) return BIBO_ERR_NULL_POINTER;
  const int rc = backward_check(sh, BIBO_NORM_SUM);
  if (rc != BIBO_OK) return rc;
  const Keeps keeps = kept_state(sh);
  if (keeps == Keeps::kNothing) return BIBO_ERR_UNSUPPORTED;
  *bytes = carve_state(sh->T, sh->E, sh->k, sh->I, keeps).total;
  return BIBO_OK;
}

static int forward_train(const void* x, const void* w_router, const float* bias, const void* w_gate_up, const void* w_down, const float* theta,
                         const bibo_moe_shape* sh, int norm_mode, void* out, int32_t* counts_out, const bibo_moe_balance* balance,
                         void* state, size_t state_bytes, void* workspace, size_t workspace_bytes, void* stream) {
  const int rc = backward_check(sh, norm_mode);
  if (rc != BIBO_OK) return rc;
  const Keeps keeps = kept_state(sh);
  if (keeps == Keeps::kNothing) return BIBO_ERR_UNSUPPORTED;
  if (state == nullptr) return BIBO_ERR_NULL_POINTER;
  if (!aligned_ws(state)) return BIBO_ERR_MISALIGNED;
  if (state_bytes < carve_state(sh->T, sh->E, sh->k, sh->I, keeps).total) return BIBO_ERR_WORKSPACE_TOO_SMALL;
  if (keeps != Keeps::kBf16) {             // (the tile kernels, whose pre-activations are kept, need both)
    if (!aligned16(x) || !aligned16(w_gate_up) || !aligned16(w_down)) return BIBO_ERR_MISALIGNED;
    if (workspace_bytes < carve(sh->T, sh->H, sh->E, sh->k, sh->I, sh->dtype).total) return BIBO_ERR_WORKSPACE_TOO_SMALL;
  }
  return forward_impl(x, w_router, bias, w_gate_up, w_down, theta, sh, norm_mode, keeps == Keeps::kBf16 ? BIBO_ALGO_FUSED : BIBO_ALGO_AUTO,
                      nullptr, out, nullptr, nullptr, counts_out, nullptr, workspace, workspace_bytes, stream, nullptr, Vec{nullptr, 0}, 0.f,
                      static_cast<char*>(state), balance);
}

int bibo_moe_forward_train(const void* x, const void* w_router, const float* bias, const void* w_gate_up, const void* w_down,
                           const float* theta, const bibo_moe_shape* sh, int norm_mode, void* out, int32_t* counts_out,
                           void* state, size_t state_bytes, void* workspace, size_t workspace_bytes, void* stream) {
  return forward_train(x, w_router, bias, w_gate_up, w_down, theta, sh, norm_mode, out, counts_out, nullptr, state, state_bytes, workspace,
                       workspace_bytes, stream);
}

int bibo_moe_forward_train_balance(const void* x, const void* w_router, const float* bias, const void* w_gate_up, const void* w_down,
                                   const float* theta, const bibo_moe_shape* sh, int norm_mode, void* out, int32_t* counts_out,
                                   const bibo_moe_balance* balance, void* state, size_t state_bytes, void* workspace,
                                   size_t workspace_bytes, void* stream) {
  if (balance == nullptr || balance->accumulated == nullptr || balance->bias == nullptr) return BIBO_ERR_NULL_POINTER;
  return forward_train(x, w_router, bias, w_gate_up, w_down, theta, sh, norm_mode, out, counts_out, balance, state, state_bytes, workspace,
                       workspace_bytes, stream);
}

int bibo_moe_backward_saved(const void* x, const void* d_out, const void* w_router, const void* w_gate_up, const void* w_down,
                            const float* theta, const bibo_moe_shape* sh, int norm_mode, const void* state,
                            size_t state_bytes, void* d_x, void* d_w_router, void* d_w_gate_up, void* d_w_down,
                            float* d_theta, float* d_w_out, void* workspace, size_t workspace_bytes, void* stream) {
  const int rc = backward_check(sh, norm_mode);
  if (rc != BIBO_OK) return rc;
  const Keeps keeps = kept_state(sh);
  if (keeps == Keeps::kNothing) return BIBO_ERR_UNSUPPORTED;
  const int T = sh->T;
  if (!workspace || !state) return BIBO_ERR_NULL_POINTER;
  if (!aligned_ws(workspace) || !aligned_ws(state)) return BIBO_ERR_MISALIGNED;
  if (state_bytes < carve_state(T, sh->E, sh->k, sh->I, keeps).total) return BIBO_ERR_WORKSPACE_TOO_SMALL;
  if (!d_w_router || !d_w_gate_up || !d_w_down || !d_theta) return BIBO_ERR_NULL_POINTER;
  if (T > 0 && (!x || !d_out || !w_router || !w_gate_up || !w_down || !d_x)) return BIBO_ERR_NULL_POINTER;
  if (T > 0 && !theta && sh->act != BIBO_ACT_SILU) return BIBO_ERR_NULL_POINTER;
  return (backward_fast(sh) ? backward_mfma : backward_generic)(x, d_out, w_router, nullptr, w_gate_up, w_down, theta, sh, norm_mode,
                                                                static_cast<const char*>(state), d_x, d_w_router, d_w_gate_up, d_w_down,
                                                                d_theta, d_w_out, workspace, workspace_bytes, stream);
}

int bibo_moe_experts_backward(const void* x, const void* d_out, const int32_t* idx, const float* w, const void* w_gate_up,
                              const void* w_down, const float* theta, const bibo_moe_shape* sh, void* d_x, float* d_w,
                              void* d_w_gate_up, void* d_w_down, float* d_theta, void* workspace, size_t workspace_bytes,
                              void* stream) {
  int rc = backward_check(sh, BIBO_NORM_SUM);
  if (rc != BIBO_OK) return rc;
  const int T = sh->T, H = sh->H, E = sh->E, k = sh->k, I = sh->I;
  if (!workspace) return BIBO_ERR_NULL_POINTER;
  if (!aligned_ws(workspace)) return BIBO_ERR_MISALIGNED;
  if (!d_w_gate_up || !d_w_down || !d_theta) return BIBO_ERR_NULL_POINTER;
  if (T > 0 && (!x || !d_out || !idx || !w || !w_gate_up || !w_down || !d_x || !d_w)) return BIBO_ERR_NULL_POINTER;
  if (T > 0 && !theta && sh->act != BIBO_ACT_SILU) return BIBO_ERR_NULL_POINTER;
  if (!backward_fast(sh)) {
    const GenericBackwardWorkspace gw = carve_backward_generic(T, H, E, k, I);
    if (workspace_bytes < gw.total) return BIBO_ERR_WORKSPACE_TOO_SMALL;
    char* gb = static_cast<char*>(workspace);
    hipStream_t gs = static_cast<hipStream_t>(stream);
    int32_t* g_offsets = reinterpret_cast<int32_t*>(gb + gw.offsets);
    int32_t* g_slot = reinterpret_cast<int32_t*>(gb + gw.perm_slot);
    int32_t* g_token = reinterpret_cast<int32_t*>(gb + gw.perm_token);
    if ((rc = hip_rc(launch_permute(idx, T, E, k, reinterpret_cast<int32_t*>(gb + gw.counts), g_offsets, g_slot, g_token,
                                    gb + gw.hist, gs))) != BIBO_OK)
      return rc;
    GenericBackwardBuffers g;
    g.dgu = reinterpret_cast<float*>(gb + gw.dgu); g.hw = reinterpret_cast<float*>(gb + gw.hw);
    g.dxs = reinterpret_cast<float*>(gb + gw.dxs);
    g.dw_slot = d_w;
    g.dl = reinterpret_cast<float*>(gb + gw.dl); g.dtheta_row = reinterpret_cast<float*>(gb + gw.dtheta_row);
    return hip_rc(launch_backward_generic(x, d_out, nullptr, w_gate_up, w_down, theta, nullptr, idx, w, g_offsets, g_slot, g_token,
                                          T, H, E - sh->n_pos - sh->n_neg, sh->n_pos, sh->n_neg, k, I, sh->dtype, BIBO_NORM_SUM,
                                          sh->act, g, d_x, nullptr, d_w_gate_up, d_w_down, d_theta, (sh->flags & BIBO_FLAG_GRAD_F32) != 0, gs));
  }
  if (!aligned16(x) || !aligned16(d_out) || !aligned16(w_gate_up) || !aligned16(w_down) || !aligned16(d_x) ||
      !aligned16(d_w_gate_up) || !aligned16(d_w_down))
    return BIBO_ERR_MISALIGNED;
  const BackwardWorkspace ws = carve_backward(T, H, E, k, I);
  if (workspace_bytes < ws.total) return BIBO_ERR_WORKSPACE_TOO_SMALL;
  char* base = static_cast<char*>(workspace);
  hipStream_t s = static_cast<hipStream_t>(stream);
  int32_t* counts = reinterpret_cast<int32_t*>(base + ws.counts);
  int32_t* offsets = reinterpret_cast<int32_t*>(base + ws.offsets);
  int32_t* perm_slot = reinterpret_cast<int32_t*>(base + ws.perm_slot);
  int32_t* perm_token = reinterpret_cast<int32_t*>(base + ws.perm_token);
  if ((rc = hip_rc(launch_permute(idx, T, E, k, counts, offsets, perm_slot, perm_token, base + ws.hist, s))) != BIBO_OK)
    return rc;
  BackwardBuffers b;
  b.gu = base + ws.gu; b.dhp = base + ws.dhp; b.dgu = base + ws.dgu;
  b.hidden = base + ws.hidden; b.dxs = base + ws.dxs; b.zrow = base + ws.zrow;
  b.dw_slot = d_w;
  b.dl = reinterpret_cast<float*>(base + ws.dl);
  b.dtheta_row = reinterpret_cast<float*>(base + ws.dtheta_row);
  b.dwr_part = reinterpret_cast<float*>(base + ws.dwr_part);
  b.wgrad_part = reinterpret_cast<float*>(base + ws.wgrad_part);
  b.wgrad_plan = reinterpret_cast<int*>(base + ws.wgrad_plan);
  return hip_rc(launch_backward(x, d_out, nullptr, w_gate_up, w_down, theta, nullptr, idx, w, offsets, perm_slot, perm_token,
                                T, H, E - sh->n_pos - sh->n_neg, sh->n_pos, sh->n_neg, k, I, BIBO_NORM_SUM, sh->act, b, d_x,
                                nullptr, d_w_gate_up, d_w_down, d_theta, (sh->flags & BIBO_FLAG_GRAD_F32) != 0, s));
}

int bibo_moe_balance_step(const int32_t* counts, float* accumulated, float* bias, int E, float factor, int update, void* stream) {
  if (E < 1 || E > kMaxE) return BIBO_ERR_BAD_SHAPE;
  if (!counts || !accumulated || !bias) return BIBO_ERR_NULL_POINTER;
  return hip_rc(launch_balance_step(BalanceArgs{counts, accumulated, bias, E, factor, update}, static_cast<hipStream_t>(stream)));
}

int bibo_moe_exp_attn_res_norm_fwd(const void* const* candidates, int n_candidates, const void* score_a, const void* score_b,
                                   float eps, const void* norm_weight, float norm_eps, int weight_dtype, int T, int H, int dtype,
                                   void* out, void* normed, void* stream) {
  const int rc = check_dims(T, H, 1, 1, 1, dtype);
  if (rc != BIBO_OK) return rc;
  if (!attn_res_supported(H, n_candidates, dtype)) return BIBO_ERR_UNSUPPORTED;
  if (!candidates || !score_a || (normed && !norm_weight)) return BIBO_ERR_NULL_POINTER;
  if (!vec_ok(score_a, weight_dtype) || !vec_ok(score_b, weight_dtype) || !vec_ok(norm_weight, weight_dtype)) return BIBO_ERR_MISALIGNED;
  if (T == 0) return BIBO_OK;
  if (!out) return BIBO_ERR_NULL_POINTER;
  for (int i = 0; i < n_candidates; ++i) {
    if (!candidates[i]) return BIBO_ERR_NULL_POINTER;
    if (!aligned16(candidates[i])) return BIBO_ERR_MISALIGNED;
  }
  if (!aligned16(out) || !aligned16(normed)) return BIBO_ERR_MISALIGNED;
  return hip_rc(launch_attn_res(candidates, n_candidates, vec(score_a, weight_dtype), vec(score_b, weight_dtype), eps, T, H, out,
                                vec(norm_weight, weight_dtype), norm_eps, normed, static_cast<hipStream_t>(stream)));
}

int bibo_moe_exp_attn_res_fwd(const void* const* candidates, int n_candidates, const float* score_weight, float eps, int T, int H,
                              int dtype, void* out, void* stream) {
  return bibo_moe_exp_attn_res_norm_fwd(candidates, n_candidates, score_weight, nullptr, eps, nullptr, 0.f, BIBO_DTYPE_F32, T, H, dtype,
                                        out, nullptr, stream);
}

int bibo_moe_exp_carry_fwd(const void* attn_read, const void* a, const void* theta, int theta_dtype, const void* prefix, int T, int H,
                           void* hs, void* prefix_out, void* stream) {
  const int rc = check_dims(T, H, 1, 1, 1, BIBO_DTYPE_BF16);
  if (rc != BIBO_OK) return rc;
  if (H % 8 != 0) return BIBO_ERR_UNSUPPORTED;
  if (T == 0) return BIBO_OK;
  if (!attn_read || !a || !hs || (prefix && !prefix_out)) return BIBO_ERR_NULL_POINTER;
  if (!aligned16(attn_read) || !aligned16(a) || !aligned16(hs) || !aligned16(prefix) || !aligned16(prefix_out) ||
      !vec_ok(theta, theta_dtype))
    return BIBO_ERR_MISALIGNED;
  return hip_rc(launch_carry(attn_read, a, vec(theta, theta_dtype), prefix, T, H, hs, prefix_out, static_cast<hipStream_t>(stream)));
}

int bibo_moe_exp_silu_mul_fwd(const void* gate_up, int T, int I, void* out, void* stream) {
  const int rc = check_dims(T, 1, 1, 1, I, BIBO_DTYPE_BF16);
  if (rc != BIBO_OK) return rc;
  if (I % 8 != 0) return BIBO_ERR_UNSUPPORTED;
  if (T == 0) return BIBO_OK;
  if (!gate_up || !out) return BIBO_ERR_NULL_POINTER;
  if (!aligned16(gate_up) || !aligned16(out)) return BIBO_ERR_MISALIGNED;
  return hip_rc(launch_silu_mul(gate_up, T, I, out, static_cast<hipStream_t>(stream)));
}

static int qk_norm_rope(void* qkv, int ld, int B, int S, int n_heads, int n_kv_heads, int head_dim, const void* q_weight, const void* k_weight,
                        int weight_dtype, float eps, const void* cos, const void* sin, int rope_dtype, int ld_rope, bool keys_only, void* stream) {
  if (B < 0 || S < 0 || (long long)B * S > 0x3fffffffLL) return BIBO_ERR_BAD_SHAPE;
  if (!exp_attention_supported(n_heads, n_kv_heads, head_dim) || ld < (n_heads + 2 * n_kv_heads) * head_dim || ld % 8 != 0 ||
      (cos == nullptr) != (sin == nullptr) || (cos != nullptr && (ld_rope < head_dim / 2 || ld_rope % 8 != 0)))
    return BIBO_ERR_UNSUPPORTED;
  if (B == 0 || S == 0) return BIBO_OK;
  if (!qkv) return BIBO_ERR_NULL_POINTER;
  if (!aligned16(qkv) || !vec_ok(q_weight, weight_dtype) || !vec_ok(k_weight, weight_dtype) || !vec_ok(cos, rope_dtype) ||
      !vec_ok(sin, rope_dtype))
    return BIBO_ERR_MISALIGNED;
  if (keys_only && k_weight == nullptr && cos == nullptr) return BIBO_OK;
  return hip_rc(launch_qk_norm_rope(qkv, ld, B * S, S, n_heads, n_kv_heads, head_dim, vec(q_weight, weight_dtype),
                                    vec(k_weight, weight_dtype), eps, vec(cos, rope_dtype), vec(sin, rope_dtype), ld_rope, keys_only,
                                    static_cast<hipStream_t>(stream)));
}

int bibo_moe_exp_qk_norm_rope(void* qkv, int ld, int B, int S, int n_heads, int n_kv_heads, int head_dim, const void* q_weight,
                              const void* k_weight, int weight_dtype, float eps, const void* cos, const void* sin, int rope_dtype,
                              int ld_rope, void* stream) {
  return qk_norm_rope(qkv, ld, B, S, n_heads, n_kv_heads, head_dim, q_weight, k_weight, weight_dtype, eps, cos, sin, rope_dtype, ld_rope, false,
                      stream);
}

int bibo_moe_exp_rope_tables(const void* inv_freq, int inv_freq_dtype, int S, int half, void* cos, void* sin, void* stream) {
  if (S < 0 || half < 1) return BIBO_ERR_BAD_SHAPE;
  if (S == 0) return BIBO_OK;
  if (!inv_freq || !cos || !sin) return BIBO_ERR_NULL_POINTER;
  return hip_rc(launch_rope_tables(vec(inv_freq, inv_freq_dtype), S, half, cos, sin, static_cast<hipStream_t>(stream)));
}

static int attention(const void* qkv, int ld, int B, int S, int n_heads, int n_kv_heads, int head_dim, int window, float scale,
                     const void* xsa_alpha, int alpha_dtype, Vec q_weight, float eps, Vec cos, Vec sin, int ld_rope, void* out, void* stream) {
  if (B < 0 || S < 0 || window < 0 || (long long)B * S * n_heads > 0x3fffffffLL) return BIBO_ERR_BAD_SHAPE;
  if (!exp_attention_supported(n_heads, n_kv_heads, head_dim) || ld < (n_heads + 2 * n_kv_heads) * head_dim || ld % 8 != 0)
    return BIBO_ERR_UNSUPPORTED;
  if (B == 0 || S == 0) return BIBO_OK;
  if (!qkv || !out) return BIBO_ERR_NULL_POINTER;
  if (!aligned16(qkv) || !aligned16(out)) return BIBO_ERR_MISALIGNED;
  return hip_rc(launch_exp_attention(qkv, ld, B, S, n_heads, n_kv_heads, head_dim, window, scale, vec(xsa_alpha, alpha_dtype), q_weight, eps, cos,
                                     sin, ld_rope, out, static_cast<hipStream_t>(stream)));
}

int bibo_moe_exp_attention_fwd(const void* qkv, int ld, int B, int S, int n_heads, int n_kv_heads, int head_dim, int window,
                               float scale, const void* xsa_alpha, int alpha_dtype, void* out, void* stream) {
  const Vec none{nullptr, 0};
  return attention(qkv, ld, B, S, n_heads, n_kv_heads, head_dim, window, scale, xsa_alpha, alpha_dtype, none, 0.f, none, none, 0, out, stream);
}

int bibo_moe_exp_norm_attention_fwd(void* qkv, int ld, int B, int S, int n_heads, int n_kv_heads, int head_dim, const void* q_weight,
                                    const void* k_weight, int weight_dtype, float eps, const void* cos, const void* sin, int rope_dtype,
                                    int ld_rope, int window, float scale, const void* xsa_alpha, int alpha_dtype, void* out, void* stream) {
  // what the second half refuses, before the first has written anything
  if (B < 0 || S < 0 || window < 0 || (long long)B * S * n_heads > 0x3fffffffLL) return BIBO_ERR_BAD_SHAPE;
  if (B > 0 && S > 0 && !out) return BIBO_ERR_NULL_POINTER;
  if (!aligned16(out)) return BIBO_ERR_MISALIGNED;
  const bool here = (long long)B * S * n_heads * head_dim >= kQueryElems;
  if (q_weight != nullptr || k_weight != nullptr || cos != nullptr) {
    const int rc = qk_norm_rope(qkv, ld, B, S, n_heads, n_kv_heads, head_dim, q_weight, k_weight, weight_dtype, eps, cos, sin, rope_dtype, ld_rope,
                                here, stream);
    if (rc != BIBO_OK) return rc;
  }
  const Vec none{nullptr, 0};
  return attention(qkv, ld, B, S, n_heads, n_kv_heads, head_dim, window, scale, xsa_alpha, alpha_dtype, here ? vec(q_weight, weight_dtype) : none, eps,
                   here ? vec(cos, rope_dtype) : none, here ? vec(sin, rope_dtype) : none, ld_rope, out, stream);
}

}  // extern "C"
