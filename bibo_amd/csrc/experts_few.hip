// The layer for a handful of tokens (single-stream decoding), bf16 or fp32: two launches behind the router, no permutation.
//
// With a few routed slots the weight-streaming kernels are all latency: one workgroup per 64 weight rows leaves most CUs
// idle (72 workgroups for one token's six experts), each pulls 98 KB through one CU, and the slot rows cross memory to a
// combine launch.  Here a workgroup takes 32 rows of ONE slot's expert (or 8 output columns of one token) with all of its
// loads in flight at once, so a launch is one round trip of an index and one of the weights.  Slots that share an expert read its
// weights again (from L2), which is why the range ends at kFewSlots.
//   gateup_few_kernel: gu[slot] = W_gate_up[e] x_t, fp32                              (src/modeling/ffn/moe.py:84)
//   down_few_kernel:   out[t] = round(residual + sum_j w_j W_down[e_j] h_j), h = r^p SiLU(g/r) u recomputed by every workgroup,
//                      one wave per slot of the token; +/-Identity slots add +/- w x   (moe.py:87-101)
// Plain FMAs: a matrix instruction would use one of its sixteen columns.  Sixteen lanes share a weight row, 16 bytes (fp32:
// 32) each at a time, i.e. whole 256-byte pieces of a row per request.
#include "few.h"

namespace bibo {
namespace {

// grid (ceil(2I / 32), S)
template <typename T, int NG>
__global__ __launch_bounds__(256) void gateup_few_kernel(const T* __restrict__ x, const T* __restrict__ wgu,
                                                         const int32_t* __restrict__ idx, int k, int H, int I2, int E,
                                                         float* __restrict__ gu) {
  const int slot = blockIdx.y, c = threadIdx.x & 15, rg = threadIdx.x >> 4;
  const int e = idx[slot];
  Raw8<T> xv[NG];
  const T* xr = x + (size_t)(slot / k) * H;
#pragma unroll
  for (int u = 0; u < NG; ++u) {
    const int g = (u * 16 + c) * 8;
    if (g < H) xv[u].load(xr + g); else xv[u].zero();
  }
  if ((unsigned)e >= (unsigned)E) return;                      // no GLU expert
  gateup_rows<T, NG>(xv, wgu + (size_t)e * I2 * H, blockIdx.x * kGateRows + rg, c, H, I2, gu + (size_t)slot * I2);
}

// grid (H / CH, T), 64 k threads: wave j = slot j of the token.  NG = ceil(I / 128).
template <typename T, int NG, int CH>
__global__ __launch_bounds__(64 * kMaxK) void down_few_kernel(const float* __restrict__ gu, const T* __restrict__ wd,
                                                              const float* __restrict__ theta, const float* __restrict__ w,
                                                              const int32_t* __restrict__ idx, CombineArgs a, int k, int H, int E,
                                                              int I, int act, T* __restrict__ out) {
  __shared__ float part[kMaxK][CH];
  const int t = blockIdx.y, c0 = blockIdx.x * CH;
  const int j = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 15, rg = lane >> 4;
  const int slot = t * k + j, e = idx[slot];
  const float ws = w[slot];
  if (e >= 0 && e < E) {
    const float p = radial_exponent(theta, e, act);
    constexpr int kIt = CH / 4;
    Raw8<T> wv[kIt][NG];
#pragma unroll
    for (int it = 0; it < kIt; ++it) {
      const T* wr = wd + ((size_t)e * H + c0 + it * 4 + rg) * I;
#pragma unroll
      for (int u = 0; u < NG; ++u) {
        const int g = (u * 16 + c) * 8;
        if (g < I) wv[it][u].load(wr + g); else wv[it][u].zero();
      }
    }
    float gv[NG][8], h[NG][8];                                 // gate, then up -> h
    const float* gr = gu + (size_t)slot * 2 * I;
    float sq[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      const int g = (u * 16 + c) * 8;
#pragma unroll
      for (int q = 0; q < 8; ++q) gv[u][q] = h[u][q] = 0.f;
      if (g < I) {
        load8(gv[u], gr + g);
        load8(h[u], gr + I + g);
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) sq[q & 3] = fmaf(gv[u][q], gv[u][q], sq[q & 3]);
    }
    const float ss = sum64(sq);
    if constexpr (sizeof(T) == 4) {
      // fp32 layers: the math library and divisions, as in activate_f32_kernel
      const float r = act == BIBO_ACT_SILU ? 1.f : sqrtf(ss / (float)I + kNormSiluEps);            // moe.py:88
      const float gain = act == BIBO_ACT_SILU ? 1.f : powf(r, p);
#pragma unroll
      for (int u = 0; u < NG; ++u)
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const float z = gv[u][q] / r;
          h[u][q] = (float)((double)(z / (1.f + expf(-z))) * gain * h[u][q]);                       // SiLU(g/r) r^p up
        }
    } else {
      float rinv, gain;                                                                            // 1/r, r^p (moe.py:88-89)
      radial_row_scalars(ss, I, p, act, rinv, gain);
      const float nrl = -1.4426950408889634f * rinv, rgn = rinv * gain;
#pragma unroll
      for (int u = 0; u < NG; ++u)
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const float sig = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(gv[u][q] * nrl));
          h[u][q] *= gv[u][q] * rgn * sig;                                                          // SiLU(g/r) r^p up
        }
    }
#pragma unroll
    for (int it = 0; it < kIt; ++it) {
      float part_d[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < NG; ++u)
#pragma unroll
        for (int q = 0; q < 8; ++q) part_d[q & 3] = fmaf(wv[it][u].get(q), h[u][q], part_d[q & 3]);
      const float acc = sum64(part_d);
      if (c == 0) part[j][it * 4 + rg] = ws * acc;                                                 // moe.py:93
    }
  } else if (lane < CH) {                                      // +/-Identity (moe.py:95-99), or no expert at all
    float v = 0.f;
    if (e >= E && e < E + a.n_pos + a.n_neg) {
      const float xv = to_float(static_cast<const T*>(a.x)[(size_t)t * H + c0 + lane]);
      v = e < E + a.n_pos ? ws * xv : -ws * xv;
    }
    part[j][lane] = v;
  }
  __syncthreads();
  if (threadIdx.x < CH) {
    const size_t o = (size_t)t * H + c0 + threadIdx.x;
    float acc = 0.f;
    for (int i = 0; i < k; ++i) acc += part[i][threadIdx.x];
    if (a.residual != nullptr)
      acc = (a.round_block ? to_float(from_float<T>(acc)) : acc) + to_float(static_cast<const T*>(a.residual)[o]);
    out[o] = from_float<T>(acc);
  }
}

// gate_up_done: launch_router_gateup has run
template <typename T>
hipError_t launch_t(const T* x, const T* wgu, const T* wd, const float* theta, const int32_t* idx, const float* w,
                    const CombineArgs& a, int Tn, int H, int E, int k, int I, int act, float* gu, T* out, bool gate_up_done, hipStream_t s) {
  auto gateup = [&](auto ng) {
    hipLaunchKernelGGL((gateup_few_kernel<T, decltype(ng)::value>), dim3((2 * I + kGateRows - 1) / kGateRows, Tn * k), dim3(256), 0, s, x,
                       wgu, idx, k, H, 2 * I, E, gu);
  };
  using std::integral_constant;
  const int nh = (H + 127) / 128;
  if (gate_up_done) {
  } else if (nh <= 2) gateup(integral_constant<int, 2>{});
  else if (nh <= 4) gateup(integral_constant<int, 4>{});
  else if (nh <= 6) gateup(integral_constant<int, 6>{});
  else gateup(integral_constant<int, 8>{});
  auto down = [&](auto ng) {
    hipLaunchKernelGGL((down_few_kernel<T, decltype(ng)::value, 8>), dim3(H / 8, Tn), dim3(64 * k), 0, s, gu, wd, theta, w, idx, a, k, H,
                       E, I, act, out);
  };
  const int ni = (I + 127) / 128;
  if (ni <= 1) down(integral_constant<int, 1>{});
  else if (ni == 2) down(integral_constant<int, 2>{});
  else if (ni == 3) down(integral_constant<int, 3>{});
  else down(integral_constant<int, 4>{});
  return hipGetLastError();
}

}  // namespace

bool few_supported(int T, int H, int k, int I) {
  return T >= 1 && T * k <= kFewSlots && H % 8 == 0 && I % 8 == 0 && H <= 1024 && I <= 512;
}

hipError_t launch_experts_few(const void* x, const void* wgu, const void* wd, const float* theta, const int32_t* idx, const float* w,
                              const CombineArgs& a, int T, int H, int E, int k, int I, int dtype, int act, float* gu, void* out,
                              bool gate_up_done, hipStream_t s) {
  if (dtype == BIBO_DTYPE_BF16)
    return launch_t(static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(wgu), static_cast<const bf16_t*>(wd), theta, idx, w, a, T,
                    H, E, k, I, act, gu, static_cast<bf16_t*>(out), gate_up_done, s);
  return launch_t(static_cast<const float*>(x), static_cast<const float*>(wgu), static_cast<const float*>(wd), theta, idx, w, a, T, H, E,
                  k, I, act, gu, static_cast<float*>(out), gate_up_done, s);
}

}  // namespace bibo
