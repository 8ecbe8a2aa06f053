// RMSNorm in front of the MoE block, as the caller of the block applies it: BiBoRMSNorm.forward
// (src/modeling/norm.py:19-24) inside BiBoDecoderLayer._ffn_forward (src/modeling/layers.py:59-60).
//   out = weight * round_to_dtype(x * rsqrt(mean(x^2) + eps)),   statistics in fp32
// One wave per row; the row stays in registers between the two passes when it is short enough.
#include "common.h"

namespace bibo {
namespace {

constexpr int kNormMaxPerLane = 32;      // elements a lane keeps in registers (rows up to 2048 wide)

template <typename TIn>
__global__ __launch_bounds__(256) void rmsnorm_kernel(const TIn* __restrict__ x, Vec weight, float eps, int T, int H, TIn* __restrict__ out) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= T) return;
  const TIn* xr = x + (size_t)row * H;
  TIn* orow = out + (size_t)row * H;
  float v[kNormMaxPerLane];
  float ss = 0.f;
  const bool in_regs = H <= kNormMaxPerLane * kWave;
  if (in_regs) {
#pragma unroll
    for (int u = 0; u < kNormMaxPerLane; ++u) {
      const int c = u * kWave + lane;
      v[u] = (c < H) ? to_float(xr[c]) : 0.f;
      ss = fmaf(v[u], v[u], ss);
    }
  } else {
    for (int c = lane; c < H; c += kWave) { const float f = to_float(xr[c]); ss = fmaf(f, f, ss); }
  }
  ss = wave_sum(ss);
  const float rinv = rsqrtf(ss / (float)H + eps);                                   // norm.py:22-23
  if (in_regs) {
#pragma unroll
    for (int u = 0; u < kNormMaxPerLane; ++u) {
      const int c = u * kWave + lane;
      if (c < H) orow[c] = from_float<TIn>(weight[c] * to_float(from_float<TIn>(v[u] * rinv)));   // norm.py:24
    }
  } else {
    for (int c = lane; c < H; c += kWave)
      orow[c] = from_float<TIn>(weight[c] * to_float(from_float<TIn>(to_float(xr[c]) * rinv)));
  }
}

// bf16 rows of up to 2048 elements, H % 8 == 0, 16-byte aligned: 16-byte accesses, the row stays in registers
__global__ __launch_bounds__(256) void rmsnorm_bf16x8_kernel(const bf16_t* __restrict__ x, Vec weight, float eps, int T, int H, bf16_t* __restrict__ out) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= T) return;
  const int nchunk = H / 8;
  const bf16x8* xr = reinterpret_cast<const bf16x8*>(x + (size_t)row * H);
  bf16x8 v[4];
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int c = u * kWave + lane;
    if (c < nchunk) {
      v[u] = xr[c];
#pragma unroll
      for (int q = 0; q < 8; ++q) ss = fmaf((float)v[u][q], (float)v[u][q], ss);
    }
  }
  ss = wave_sum(ss);
  const float rinv = rsqrtf(ss / (float)H + eps);                                   // norm.py:22-23
  bf16x8* orow = reinterpret_cast<bf16x8*>(out + (size_t)row * H);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int c = u * kWave + lane;
    if (c < nchunk) {
      bf16x8 o;
      float nw[8];
      load8(weight, c * 8, nw);
#pragma unroll
      for (int q = 0; q < 8; ++q) o[q] = (bf16_t)(nw[q] * (float)(bf16_t)((float)v[u][q] * rinv));   // norm.py:24
      orow[c] = o;
    }
  }
}

// Depth mix of Block Attention Residuals (apply_attention_residual, exp/modeling_bibo.py:119-232, softmax scores,
// dense): candidates = the completed block representatives and the running prefix sum of a token; score of a
// candidate = rsqrt(mean(c^2) + eps) * <c, score_a * score_b> (norm weight and pseudo-query; their product in fp32); out = the
// candidates averaged with the softmax of their scores, fp32, rounded once.  With `normed`, the RMSNorm of the rounded row
// that the attention behind it reads (input_layernorm) leaves with it.  One wave per token, all N candidate rows
// requested at once and kept in registers (two 16-byte granules per lane: H <= 1024): bound by memory.
constexpr int kAttnResMaxCand = 8;
struct AttnResPtrs {
  const bf16_t* c[kAttnResMaxCand];
};

template <int N>
__global__ __launch_bounds__(256) void attn_res_kernel(AttnResPtrs cand, Vec score_a, Vec score_b, float eps, int T, int H,
                                                       bf16_t* __restrict__ out, Vec norm_w, float norm_eps,
                                                       bf16_t* __restrict__ normed) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= T) return;
  const int nchunk = H / 8;
  bf16x8 v[N][2];
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c = u * kWave + lane;
      if (c < nchunk) v[i][u] = reinterpret_cast<const bf16x8*>(cand.c[i] + (size_t)row * H)[c];
      else
#pragma unroll
        for (int q = 0; q < 8; ++q) v[i][u][q] = (bf16_t)0.f;
    }
  float score[N], ss[N], dot[N];
#pragma unroll
  for (int i = 0; i < N; ++i) ss[i] = dot[i] = 0.f;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int c = u * kWave + lane;
    float sw[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (c < nchunk) {
      load8(score_a, c * 8, sw);
      if (score_b.p != nullptr) {
        float sb[8];
        load8(score_b, c * 8, sb);
#pragma unroll
        for (int q = 0; q < 8; ++q) sw[q] *= sb[q];
      }
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const float f = (float)v[i][u][q];
        ss[i] = fmaf(f, f, ss[i]);
        dot[i] = fmaf(f, sw[q], dot[i]);
      }
  }
  float mx = -3.0e38f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    score[i] = wave_sum(dot[i]) * rsqrtf(wave_sum(ss[i]) / (float)H + eps);
    mx = fmaxf(mx, score[i]);
  }
  float den = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    score[i] = __expf(score[i] - mx);
    den += score[i];
  }
  const float inv = 1.f / den;
  bf16x8 o[2];
  float os = 0.f;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int c = u * kWave + lane;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float pr = score[i] * inv;
#pragma unroll
      for (int q = 0; q < 8; ++q) acc[q] = fmaf(pr, (float)v[i][u][q], acc[q]);
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      o[u][q] = (bf16_t)acc[q];
      os = fmaf((float)o[u][q], (float)o[u][q], os);
    }
    if (c < nchunk) reinterpret_cast<bf16x8*>(out + (size_t)row * H)[c] = o[u];
  }
  if (normed == nullptr) return;
  const float rinv = rsqrtf(wave_sum(os) / (float)H + norm_eps);                    // norm.py:22-23
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int c = u * kWave + lane;
    if (c < nchunk) {
      bf16x8 w;
      float nw[8];
      load8(norm_w, c * 8, nw);
#pragma unroll
      for (int q = 0; q < 8; ++q) w[q] = (bf16_t)(nw[q] * (float)(bf16_t)((float)o[u][q] * rinv));   // norm.py:24
      reinterpret_cast<bf16x8*>(normed + (size_t)row * H)[c] = w;
    }
  }
}

// The two sums behind an attention block (exp/modeling_bibo.py:526-531,640-648), 8 elements per thread: hs = attn_read +
// theta a (theta NULL: a), and prefix_out = prefix + a where the block has a prefix already.
__global__ __launch_bounds__(256) void carry_kernel(const bf16_t* __restrict__ attn_read, const bf16_t* __restrict__ a,
                                                    Vec theta, const bf16_t* __restrict__ prefix,
                                                    long long n8, int H8, bf16_t* __restrict__ hs, bf16_t* __restrict__ prefix_out) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const int c = (int)(i % H8);
  const bf16x8 av = reinterpret_cast<const bf16x8*>(a)[i], rv = reinterpret_cast<const bf16x8*>(attn_read)[i];
  float th[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};
  if (theta.p != nullptr) load8(theta, c * 8, th);
  bf16x8 o;
#pragma unroll
  for (int q = 0; q < 8; ++q) o[q] = (bf16_t)fmaf(th[q], (float)av[q], (float)rv[q]);
  reinterpret_cast<bf16x8*>(hs)[i] = o;
  if (prefix != nullptr) {
    const bf16x8 pv = reinterpret_cast<const bf16x8*>(prefix)[i];
#pragma unroll
    for (int q = 0; q < 8; ++q) o[q] = (bf16_t)((float)pv[q] + (float)av[q]);
    reinterpret_cast<bf16x8*>(prefix_out)[i] = o;
  }
}

// SiLU(gate) * up of rows [gate | up] of a dense SwiGLU (src/modeling/ffn/mlp.py:34-35), 8 elements per thread
__global__ __launch_bounds__(256) void silu_mul_kernel(const bf16_t* __restrict__ gu, long long n8, int I8, bf16_t* __restrict__ out) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const long long t = i / I8, c = i - t * I8;
  const bf16x8 g = reinterpret_cast<const bf16x8*>(gu)[t * 2 * I8 + c], u = reinterpret_cast<const bf16x8*>(gu)[t * 2 * I8 + I8 + c];
  bf16x8 o;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const float f = (float)g[q];
    o[q] = (bf16_t)(f / (1.f + __expf(-f)) * (float)u[q]);
  }
  reinterpret_cast<bf16x8*>(out)[i] = o;
}

}  // namespace

bool attn_res_supported(int H, int n_cand, int dtype) {
  return dtype == BIBO_DTYPE_BF16 && H % 8 == 0 && H <= 1024 && n_cand >= 1 && n_cand <= kAttnResMaxCand;
}

hipError_t launch_attn_res(const void* const* cands, int n_cand, Vec score_a, Vec score_b, float eps, int T, int H, void* out,
                           Vec norm_w, float norm_eps, void* normed, hipStream_t s) {
  if (T == 0) return hipSuccess;
  AttnResPtrs p;
  for (int i = 0; i < kAttnResMaxCand; ++i) p.c[i] = static_cast<const bf16_t*>(i < n_cand ? cands[i] : cands[0]);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((T + 3) / 4), dim3(256), 0, s, p, score_a, score_b, eps, T, H, static_cast<bf16_t*>(out), norm_w, norm_eps,
                       static_cast<bf16_t*>(normed));
  };
  switch (n_cand) {
    case 1: launch(attn_res_kernel<1>); break;
    case 2: launch(attn_res_kernel<2>); break;
    case 3: launch(attn_res_kernel<3>); break;
    case 4: launch(attn_res_kernel<4>); break;
    case 5: launch(attn_res_kernel<5>); break;
    case 6: launch(attn_res_kernel<6>); break;
    case 7: launch(attn_res_kernel<7>); break;
    case 8: launch(attn_res_kernel<8>); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_carry(const void* attn_read, const void* a, Vec theta, const void* prefix, int T, int H, void* hs,
                        void* prefix_out, hipStream_t s) {
  const long long n8 = (long long)T * H / 8;
  if (n8 == 0) return hipSuccess;
  hipLaunchKernelGGL(carry_kernel, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, s, static_cast<const bf16_t*>(attn_read),
                     static_cast<const bf16_t*>(a), theta, static_cast<const bf16_t*>(prefix), n8, H / 8, static_cast<bf16_t*>(hs),
                     static_cast<bf16_t*>(prefix_out));
  return hipGetLastError();
}

hipError_t launch_silu_mul(const void* gu, int T, int I, void* out, hipStream_t s) {
  const long long n8 = (long long)T * I / 8;
  if (n8 == 0) return hipSuccess;
  hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, s, static_cast<const bf16_t*>(gu), n8, I / 8,
                     static_cast<bf16_t*>(out));
  return hipGetLastError();
}

hipError_t launch_rmsnorm(const void* x, Vec weight, float eps, int T, int H, int dtype, void* out,
                          hipStream_t s) {
  if (T == 0) return hipSuccess;
  const int grid = (T + 3) / 4;
  const bool vec = dtype == BIBO_DTYPE_BF16 && (H % 8) == 0 && H <= 2048 &&
                   ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
  if (vec)
    hipLaunchKernelGGL(rmsnorm_bf16x8_kernel, dim3(grid), dim3(256), 0, s, static_cast<const bf16_t*>(x), weight, eps, T, H,
                       static_cast<bf16_t*>(out));
  else if (dtype == BIBO_DTYPE_BF16)
    hipLaunchKernelGGL(rmsnorm_kernel<bf16_t>, dim3(grid), dim3(256), 0, s, static_cast<const bf16_t*>(x), weight, eps, T,
                       H, static_cast<bf16_t*>(out));
  else
    hipLaunchKernelGGL(rmsnorm_kernel<float>, dim3(grid), dim3(256), 0, s, static_cast<const float*>(x), weight, eps, T,
                       H, static_cast<float*>(out));
  return hipGetLastError();
}

}  // namespace bibo
