// Generic backward pass of the sparse-MoE block: any hidden and expert size, bf16 or fp32 operands, fp32 arithmetic.
// It serves what the MFMA backward (backward.hip) does not take: fp32 modules (the reference's own tests take their
// gradients in fp32 at tiny sizes, tests/test_moe.py:53-63, ablate/common/test_eager_radial.py:63-69) and sizes that
// are no multiples of 128.  The gradients are those torch.autograd derives for the eager layer
// (src/modeling/ffn/moe.py:46-101,157-183, src/modeling/ffn/router.py:25-47) with the selection held fixed; the
// formulas are the ones spelled out at the top of backward.hip.  Sizes that are multiples of four run on the fp32 MFMA
// GEMMs of tile_f32.h with a row-wise activation kernel between them; the rest takes one workgroup per routed row for the
// row-wise part and one workgroup per weight row for the weight gradients, which loop over an expert's rows in permuted
// order.  Every sum has a fixed order, so the results are the same bits on every call.
#include "tile_f32.h"

namespace bibo {
namespace {

__device__ __forceinline__ float block_sum(float v, float* red) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  v = wave_sum(v);
  __syncthreads();                                   // red may still be read from the sum before
  if (lane == 0) red[wave] = v;
  __syncthreads();
  return ((red[0] + red[1]) + red[2]) + red[3];
}

// Per routed row of a GLU expert (permuted row `row`, token t, slot s, expert e, combine weight w):
//   gu = W_gate_up[e] x_t;  dh' = W_down[e]^T d_t;  dw[s] = <dh', h>;  (dg, du, dtheta share) from dh = w dh';
//   dgu[row] = [dg, du];  hw[row] = w h;  dxs[s] = W_gate_up[e]^T [dg, du].
// Dynamic LDS: 2H + 5I floats.
template <typename TIn>
__global__ __launch_bounds__(256) void row_bwd_generic_kernel(const TIn* __restrict__ x, const TIn* __restrict__ d_out,
                                                              const TIn* __restrict__ wgu, const TIn* __restrict__ wd,
                                                              const float* __restrict__ theta, const float* __restrict__ w,
                                                              const int32_t* __restrict__ offsets,
                                                              const int32_t* __restrict__ perm_slot,
                                                              const int32_t* __restrict__ perm_token, int H, int E, int I,
                                                              int act, float* __restrict__ dgu, float* __restrict__ hw,
                                                              float* __restrict__ dxs, float* __restrict__ dw_slot,
                                                              float* __restrict__ dtheta_row) {
  extern __shared__ float smem[];
  float* xs = smem;                 // [H]
  float* ds = xs + H;               // [H]
  float* gu = ds + H;               // [2I]
  float* dhp = gu + 2 * I;          // [I]
  float* dg = dhp + I;              // [2I]  dg, then du
  __shared__ int sh_e;
  __shared__ float red[4];
  const int row = blockIdx.x;
  if (row >= offsets[E]) return;                     // E = GLU experts: rows behind theirs have no activation
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  if (tid < E && offsets[tid] <= row && row < offsets[tid + 1]) sh_e = tid;
  const int slot = perm_slot[row];
  const size_t t = (size_t)perm_token[row];
  for (int h = tid; h < H; h += 256) {
    xs[h] = to_float(x[t * H + h]);
    ds[h] = to_float(d_out[t * H + h]);
  }
  __syncthreads();
  const int e = sh_e;
  const float ws = w[slot];
  const TIn* wg = wgu + (size_t)e * 2 * I * H;
  const TIn* wdn = wd + (size_t)e * H * I;
  for (int c = wave; c < 2 * I; c += 4) {            // pre-activations (moe.py:84): one wave per weight row
    const TIn* wrow = wg + (size_t)c * H;
    float acc = 0.f;
    for (int h = lane; h < H; h += kWave) acc = fmaf(xs[h], to_float(wrow[h]), acc);
    acc = wave_sum(acc);
    if (lane == 0) gu[c] = acc;
  }
  for (int i = tid; i < I; i += 256) {               // dh' = W_down^T d: a thread per column, coalesced over i
    float acc = 0.f;
    for (int h = 0; h < H; ++h) acc = fmaf(ds[h], to_float(wdn[(size_t)h * I + i]), acc);
    dhp[i] = acc;
  }
  __syncthreads();
  float ss = 0.f;
  for (int i = tid; i < I; i += 256) ss = fmaf(gu[i], gu[i], ss);
  ss = block_sum(ss, red);
  const bool radial = act != BIBO_ACT_SILU;
  float p = 0.f, r = 1.f, gain = 1.f;
  if (radial) {
    p = radial_exponent(theta, e, act);
    r = sqrtf(ss / (float)I + kNormSiluEps);         // moe.py:88
    gain = powf(r, p);
  }
  const float rinv = 1.f / r;
  // h = r^p a u, a = z s, s = sigmoid(z), z = g / r, a' = s (1 + z (1 - s)); q = w dh' u
  float dot_h = 0.f, sum_qa = 0.f, inner = 0.f;
  for (int i = tid; i < I; i += 256) {
    const float z = gu[i] * rinv, s = 1.f / (1.f + expf(-z));
    const float a = z * s, ad = s * (1.f + z * (1.f - s));
    const float u = gu[I + i];
    dot_h = fmaf(dhp[i], gain * a * u, dot_h);
    const float q = ws * dhp[i] * u;
    sum_qa = fmaf(q, a, sum_qa);
    inner = fmaf(q, gain * rinv * (p * a - ad * z), inner);
  }
  dot_h = block_sum(dot_h, red);
  sum_qa = block_sum(sum_qa, red);
  inner = block_sum(inner, red);
  for (int i = tid; i < I; i += 256) {
    const float z = gu[i] * rinv, s = 1.f / (1.f + expf(-z));
    const float a = z * s, ad = s * (1.f + z * (1.f - s));
    const float u = gu[I + i], dh = ws * dhp[i];
    float g_ = dh * u * gain * rinv * ad;
    if (radial) g_ = fmaf(gu[i] * rinv / (float)I, inner, g_);
    const float u_ = dh * gain * a;
    dg[i] = g_;
    dg[I + i] = u_;
    dgu[(size_t)row * 2 * I + i] = g_;
    dgu[(size_t)row * 2 * I + I + i] = u_;
    hw[(size_t)row * I + i] = ws * gain * a * u;
  }
  if (tid == 0) {
    dw_slot[slot] = dot_h;
    const float dp = act == BIBO_ACT_RADIAL_TANH ? 1.f - p * p : p * (1.f - p);
    dtheta_row[row] = radial ? dp * logf(r) * gain * sum_qa : 0.f;
  }
  __syncthreads();
  for (int h = tid; h < H; h += 256) {               // dx of the slot: a thread per column, coalesced over h
    float acc = 0.f;
    for (int c = 0; c < 2 * I; ++c) acc = fmaf(dg[c], to_float(wg[(size_t)c * H + h]), acc);
    dxs[(size_t)slot * H + h] = acc;
  }
}

// Radial NormSiLU backward of one permuted row per wave (formulas at the top of row_bwd_generic_kernel and backward.hip): gu [S, 2I] holds
// [g, u], dgu receives [dg, du] (it may be gu), dhp [S, I] holds dh' and receives w h.  The row is read three times,
// from L1 after the first.
__global__ __launch_bounds__(256) void act_bwd_f32_kernel(const float* gu, float* dgu, float* __restrict__ dhp,
                                                          const float* __restrict__ w, const float* __restrict__ theta,
                                                          const int32_t* __restrict__ offsets,
                                                          const int32_t* __restrict__ perm_slot, int S, int E, int I, int act,
                                                          float* __restrict__ dw_slot, float* __restrict__ dtheta_row) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= S) return;
  const int e = expert_of_row(offsets, E, row);
  if (e < 0) return;
  const int slot = perm_slot[row];
  const float ws = w[slot];
  const float* gr = gu + (size_t)row * 2 * I;
  float* go = dgu + (size_t)row * 2 * I;
  float* dr = dhp + (size_t)row * I;
  float ss = 0.f;
  for (int c = lane * 4; c < I; c += 4 * kWave) {
    const floatx4 g = load4<float>(gr + c);
#pragma unroll
    for (int q = 0; q < 4; ++q) ss = fmaf(g[q], g[q], ss);
  }
  ss = wave_sum(ss);
  const bool radial = act != BIBO_ACT_SILU;
  float p = 0.f, r = 1.f, gain = 1.f;
  if (radial) {
    p = radial_exponent(theta, e, act);
    r = sqrtf(ss / (float)I + kNormSiluEps);         // moe.py:88
    gain = powf(r, p);
  }
  const float rinv = 1.f / r;
  float dot_h = 0.f, sum_qa = 0.f, inner = 0.f;
  for (int c = lane * 4; c < I; c += 4 * kWave) {
    const floatx4 g = load4<float>(gr + c), u = load4<float>(gr + I + c), d = load4<float>(dr + c);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float z = g[q] * rinv, s = 1.f / (1.f + expf(-z));
      const float a = z * s, ad = s * (1.f + z * (1.f - s));
      dot_h = fmaf(d[q], gain * a * u[q], dot_h);
      const float qq = ws * d[q] * u[q];
      sum_qa = fmaf(qq, a, sum_qa);
      inner = fmaf(qq, gain * rinv * (p * a - ad * z), inner);
    }
  }
  dot_h = wave_sum(dot_h);
  sum_qa = wave_sum(sum_qa);
  inner = wave_sum(inner);
  for (int c = lane * 4; c < I; c += 4 * kWave) {
    const floatx4 g = load4<float>(gr + c), u = load4<float>(gr + I + c), d = load4<float>(dr + c);
    floatx4 og, ou, oh;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float z = g[q] * rinv, s = 1.f / (1.f + expf(-z));
      const float a = z * s, ad = s * (1.f + z * (1.f - s));
      const float dh = ws * d[q];
      float dg = dh * u[q] * gain * rinv * ad;
      if (radial) dg = fmaf(g[q] * rinv / (float)I, inner, dg);
      og[q] = dg;
      ou[q] = dh * gain * a;
      oh[q] = (float)((double)ws * gain * a * u[q]);
    }
    store4(go + c, og);
    store4(go + I + c, ou);
    store4(dr + c, oh);
  }
  if (lane == 0) {
    dw_slot[slot] = dot_h;
    const float dp = act == BIBO_ACT_RADIAL_TANH ? 1.f - p * p : p * (1.f - p);
    dtheta_row[row] = radial ? dp * logf(r) * gain * sum_qa : 0.f;
  }
}

// Everything per token behind the experts, one wave per token: the combine-weight gradients of +/-Identity slots
// (sign <d_out[t], x[t]>, moe.py:95-99), dlogit of the k selected experts (router.py:31,41-47; w_router == NULL: none), and
//   dx[t, h] = sum_j dx of slot j + sum_j dl[t, j] W_router[idx[t, j], h]
// where the dx of a slot is its dxs row or, for an Identity slot, sign w d_out[t].  A slot whose expert id lies outside
// [0, E + n_pos + n_neg) is left out and its dw_slot entry is set to zero.
template <typename TIn>
__global__ __launch_bounds__(256) void token_bwd_generic_kernel(const TIn* __restrict__ x, const TIn* __restrict__ d_out,
                                                                const float* __restrict__ dxs, const float* __restrict__ logits,
                                                                const int32_t* __restrict__ idx, const float* __restrict__ w,
                                                                const TIn* __restrict__ w_router, int T, int H, int E, int n_pos,
                                                                int n_neg, int k, int norm_mode, float* __restrict__ dw_slot,
                                                                float* __restrict__ dl, TIn* __restrict__ dx) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  const int Et = E + n_pos + n_neg;
  // lane j < k holds slot j
  int e_ = -1;
  float w_ = 0.f, dw_ = 0.f, s_ = 0.f;
  if (lane < k) {
    e_ = idx[t * k + lane];
    w_ = w[t * k + lane];
    if (e_ < 0 || e_ >= Et) e_ = -1;
    if (e_ >= 0 && e_ < E) dw_ = dw_slot[t * k + lane];
    if (w_router != nullptr) s_ = 1.f / (1.f + expf(-logits[(size_t)t * Et + e_]));
  }
  if (__ballot(e_ >= E) != 0ull) {
    float dot = 0.f;
    for (int h = lane; h < H; h += kWave) dot = fmaf(to_float(d_out[(size_t)t * H + h]), to_float(x[(size_t)t * H + h]), dot);
    dot = wave_sum(dot);
    if (e_ >= E) dw_ = e_ < E + n_pos ? dot : -dot;
  }
  if (lane < k && (e_ < 0 || e_ >= E)) dw_slot[t * k + lane] = dw_;
  float dl_ = 0.f;
  if (w_router != nullptr) {
    float sum = 0.f, dot = 0.f;
    for (int j = 0; j < k; ++j) {
      sum += __shfl(s_, j, kWave);
      dot = fmaf(__shfl(dw_, j, kWave), __shfl(w_, j, kWave), dot);
    }
    float ds = dw_;
    if (k > 1 && norm_mode == BIBO_NORM_SUM) ds = (ds - dot) / (sum + 1e-20f);
    else if (k > 1 && norm_mode == BIBO_NORM_SOFTMAX) ds = w_ * (ds - dot);
    dl_ = ds * s_ * (1.f - s_);
    if (lane < k) dl[t * k + lane] = dl_;
  }
  int ej[kMaxK];                                     // the k slots, the same in every lane
  float wj[kMaxK], dlj[kMaxK];
#pragma unroll
  for (int j = 0; j < kMaxK; ++j) {
    ej[j] = j < k ? __builtin_amdgcn_readlane(e_, j) : -1;
    wj[j] = __shfl(w_, j, kWave);
    dlj[j] = __shfl(dl_, j, kWave);
  }
  for (int h = lane; h < H; h += kWave) {
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < kMaxK; ++j) {
      const int e = ej[j];
      if (e < 0) continue;
      if (e < E) acc += dxs[((size_t)t * k + j) * H + h];
      else acc = fmaf(e < E + n_pos ? wj[j] : -wj[j], to_float(d_out[(size_t)t * H + h]), acc);
      if (w_router != nullptr) acc = fmaf(dlj[j], to_float(w_router[(size_t)e * H + h]), acc);
    }
    dx[(size_t)t * H + h] = from_float<TIn>(acc);
  }
}

// grid (Et, ceil(H / 64) + 1).  Blocks y < ceil(H / 64): dW_router[e, h] = sum over the rows r of expert e of dl[slot(r)]
// x[token(r), h] for 64 columns: 16 row groups of 16 threads x 4 columns, the groups' sums added in order (dwr == NULL: none).
// The last y: dtheta[e] = the sum of its rows' shares (e < E).
template <typename TIn, typename TG>
__global__ __launch_bounds__(256) void expert_sums_generic_kernel(const TIn* __restrict__ x, const float* __restrict__ dl,
                                                                  const int32_t* __restrict__ offsets,
                                                                  const int32_t* __restrict__ perm_slot,
                                                                  const int32_t* __restrict__ perm_token, int H, int E,
                                                                  const float* __restrict__ dtheta_row,
                                                                  float* __restrict__ dtheta, TG* __restrict__ dwr) {
  __shared__ float red[16][65];
  const int e = blockIdx.x, tid = threadIdx.x;
  const int lo = offsets[e], hi = offsets[e + 1];
  if (blockIdx.y + 1 == gridDim.y) {
    if (e >= E) return;
    float acc = 0.f;
    for (int r = lo + tid; r < hi; r += 256) acc += dtheta_row[r];
    acc = block_sum(acc, red[0]);
    if (tid == 0) dtheta[e] = acc;
    return;
  }
  if (dwr == nullptr) return;
  const int rl = tid >> 4, c4 = (tid & 15) * 4, h0 = blockIdx.y * 64;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  constexpr int kU = 4;                                        // rows of a thread whose loads are in flight together
  for (int r = lo + rl; r < hi; r += 16 * kU) {
    float d[kU], v[kU][4];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int rr = r + 16 * u;
      d[u] = rr < hi ? dl[perm_slot[rr]] : 0.f;
      const size_t t = rr < hi ? perm_token[rr] : 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) v[u][q] = rr < hi && h0 + c4 + q < H ? to_float(x[t * H + h0 + c4 + q]) : 0.f;
    }
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = fmaf(d[u], v[u][q], acc[q]);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) red[rl][c4 + q] = acc[q];
  __syncthreads();
  if (tid < 64 && h0 + tid < H) {
    float sum = 0.f;
#pragma unroll
    for (int g = 0; g < 16; ++g) sum += red[g][tid];
    dwr[(size_t)e * H + h0 + tid] = from_float<TG>(sum);
  }
}

// dW[e][n][m] = sum over the rows r of expert e, in row order, of P[srcP(r)][n] Q[srcQ(r)][m]; grid = (N, E), threads
// over m.  srcP(r) = index[r] (GATHER_P) or r, likewise Q.  P and Q may be fp32 workspace rows or operands.
template <typename TP, typename TQ, typename TOut, bool GATHER_P, bool GATHER_Q>
__global__ __launch_bounds__(256) void wgrad_generic_kernel(const TP* __restrict__ P, const TQ* __restrict__ Q,
                                                            const int32_t* __restrict__ index,
                                                            const int32_t* __restrict__ offsets, int N, int M,
                                                            TOut* __restrict__ dW) {
  const int n = blockIdx.x, e = blockIdx.y;
  const int lo = offsets[e], hi = offsets[e + 1];
  for (int m0 = 0; m0 < M; m0 += 256) {
    const int m = m0 + threadIdx.x;
    float acc = 0.f;
    for (int r = lo; r < hi; ++r) {
      const int ix = (GATHER_P || GATHER_Q) ? index[r] : 0;
      const float pv = to_float(P[(size_t)(GATHER_P ? ix : r) * N + n]);
      if (m < M) acc = fmaf(pv, to_float(Q[(size_t)(GATHER_Q ? ix : r) * M + m]), acc);
    }
    if (m < M) dW[((size_t)e * N + n) * M + m] = from_float<TOut>(acc);
  }
}

template <typename TIn>
__global__ void zero_generic_kernel(TIn* __restrict__ p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    p[i] = from_float<TIn>(0.f);
}

template <typename TIn>
void zero_elems(TIn* p, size_t n, hipStream_t s) {
  if (n == 0) return;
  const unsigned grid = (unsigned)((n + 255) / 256 < 2048 ? (n + 255) / 256 : 2048);
  hipLaunchKernelGGL(zero_generic_kernel<TIn>, dim3(grid), dim3(256), 0, s, p, n);
}

// TG: type of the weight gradients
template <typename TIn, typename TG>
hipError_t launch_t(const void* x_, const void* d_out_, const void* w_router_, const void* wgu_, const void* wd_,
                    const float* theta, const float* logits, const int32_t* idx, const float* w, const int32_t* offsets,
                    const int32_t* perm_slot, const int32_t* perm_token, int T, int H, int E, int n_pos, int n_neg, int k, int I,
                    int norm_mode, int act, const GenericBackwardBuffers& b, void* dx_, void* d_w_router_, void* d_wgu_,
                    void* d_wd_, float* d_theta, hipStream_t s) {
  const TIn* x = static_cast<const TIn*>(x_);
  const TIn* d_out = static_cast<const TIn*>(d_out_);
  const TIn* w_router = static_cast<const TIn*>(w_router_);
  const TIn* wgu = static_cast<const TIn*>(wgu_);
  const TIn* wd = static_cast<const TIn*>(wd_);
  const int Et = E + n_pos + n_neg, S = T * k;
  if (S == 0) {
    zero_elems(d_theta, (size_t)E, s);
    if (d_w_router_ != nullptr) zero_elems(static_cast<TG*>(d_w_router_), (size_t)Et * H, s);
    zero_elems(static_cast<TG*>(d_wgu_), (size_t)E * 2 * I * H, s);
    zero_elems(static_cast<TG*>(d_wd_), (size_t)E * H * I, s);
    return hipGetLastError();
  }
  const bool tiles = tile_f32_supported(H, I) && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(d_out) |
                                                    reinterpret_cast<uintptr_t>(wgu) | reinterpret_cast<uintptr_t>(wd)) & 15) == 0;
  hipError_t err = hipSuccess;
  if (tiles) {
    // gu = x W_gate_up^T, where the forward has not kept it; dh' = d W_down; [dg, du] and w h in their places; dx of every slot = [dg, du] W_gate_up
    const float* gu = b.gu_saved;
    if (gu == nullptr) {
      gu = b.dgu;
      if ((err = launch_ggemm_f32<TIn, TIn, false, true, false>(x, perm_token, wgu, offsets, nullptr, nullptr, S, H, 2 * I, E, b.dgu, s)) != hipSuccess) return err;
    }
    if ((err = launch_ggemm_f32<TIn, TIn, true, true, false>(d_out, perm_token, wd, offsets, nullptr, nullptr, S, H, I, E, b.hw, s)) != hipSuccess) return err;
    hipLaunchKernelGGL(act_bwd_f32_kernel, dim3((S + 3) / 4), dim3(256), 0, s, gu, b.dgu, b.hw, w, theta, offsets, perm_slot, S, E, I,
                       act, b.dw_slot, b.dtheta_row);
    if ((err = launch_ggemm_f32<float, TIn, true, false, true>(b.dgu, nullptr, wgu, offsets, perm_slot, nullptr, S, 2 * I, H, E, b.dxs, s)) != hipSuccess) return err;
  } else {
    const size_t shm = (size_t)(2 * H + 5 * I) * sizeof(float);
    hipLaunchKernelGGL(row_bwd_generic_kernel<TIn>, dim3(S), dim3(256), shm, s, x, d_out, wgu, wd, theta, w, offsets, perm_slot,
                       perm_token, H, E, I, act, b.dgu, b.hw, b.dxs, b.dw_slot, b.dtheta_row);
  }
  const bool with_router = w_router != nullptr;      // else: the experts alone, the caller owns the routing
  hipLaunchKernelGGL(token_bwd_generic_kernel<TIn>, dim3((T + 3) / 4), dim3(256), 0, s, x, d_out, b.dxs, logits, idx, w, w_router, T,
                     H, E, n_pos, n_neg, k, norm_mode, b.dw_slot, b.dl, static_cast<TIn*>(dx_));
  hipLaunchKernelGGL((expert_sums_generic_kernel<TIn, TG>), dim3(Et, (H + 63) / 64 + 1), dim3(256), 0, s, x, b.dl, offsets, perm_slot,
                     perm_token, H, E, b.dtheta_row, d_theta, with_router ? static_cast<TG*>(d_w_router_) : nullptr);
  // dW_down[e] = d^T (w h), d gathered by token; dW_gate_up[e] = [dg, du]^T x, x gathered by token
  if (tiles) {
    if ((err = launch_wgrad_f32<TIn, float, TG, true, false>(d_out, b.hw, perm_token, offsets, H, I, E, static_cast<TG*>(d_wd_), s)) != hipSuccess) return err;
    return launch_wgrad_f32<float, TIn, TG, false, true>(b.dgu, x, perm_token, offsets, 2 * I, H, E, static_cast<TG*>(d_wgu_), s);
  }
  hipLaunchKernelGGL((wgrad_generic_kernel<TIn, float, TG, true, false>), dim3(H, E), dim3(256), 0, s, d_out, b.hw, perm_token,
                     offsets, H, I, static_cast<TG*>(d_wd_));
  hipLaunchKernelGGL((wgrad_generic_kernel<float, TIn, TG, false, true>), dim3(2 * I, E), dim3(256), 0, s, b.dgu, x, perm_token,
                     offsets, 2 * I, H, static_cast<TG*>(d_wgu_));
  return hipGetLastError();
}

}  // namespace

// the row kernel keeps 2H + 5I floats of a row in dynamic LDS next to a few words of its own; 64 KB per workgroup
// need no raised limit
bool backward_generic_supported(int H, int I, int k) {
  return (size_t)(2 * H + 5 * I) * sizeof(float) + 64 <= 64 * 1024 && k <= kMaxK;
}

// Buffers (fp32): dgu [S,2I], hw [S,I], dxs [S,H], dw_slot [S], dl [S], dtheta_row [S].
hipError_t launch_backward_generic(const void* x, const void* d_out, const void* w_router, const void* wgu, const void* wd,
                                   const float* theta, const float* logits, const int32_t* idx, const float* w,
                                   const int32_t* offsets, const int32_t* perm_slot, const int32_t* perm_token, int T, int H,
                                   int E, int n_pos, int n_neg, int k, int I, int dtype, int norm_mode, int act,
                                   const GenericBackwardBuffers& b, void* dx, void* d_w_router, void* d_wgu, void* d_wd,
                                   float* d_theta, int grad_f32, hipStream_t s) {
  if (dtype == BIBO_DTYPE_BF16 && !grad_f32)
    return launch_t<bf16_t, bf16_t>(x, d_out, w_router, wgu, wd, theta, logits, idx, w, offsets, perm_slot, perm_token, T, H, E, n_pos,
                            n_neg, k, I, norm_mode, act, b, dx, d_w_router, d_wgu, d_wd, d_theta, s);
  if (dtype == BIBO_DTYPE_BF16)
    return launch_t<bf16_t, float>(x, d_out, w_router, wgu, wd, theta, logits, idx, w, offsets, perm_slot, perm_token, T, H, E, n_pos,
                            n_neg, k, I, norm_mode, act, b, dx, d_w_router, d_wgu, d_wd, d_theta, s);
  return launch_t<float, float>(x, d_out, w_router, wgu, wd, theta, logits, idx, w, offsets, perm_slot, perm_token, T, H, E, n_pos,
                         n_neg, k, I, norm_mode, act, b, dx, d_w_router, d_wgu, d_wd, d_theta, s);
}

}  // namespace bibo
