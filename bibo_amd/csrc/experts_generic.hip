// Generic expert kernels: any H and I, bf16 or fp32 operands, fp32 arithmetic.  They serve shapes the bf16 MFMA
// tiles do not cover and fp32 modules, and double as an independent implementation the MFMA kernels are cross-checked
// against.  Two ways through them: grouped GEMMs on fp32 MFMAs (tile_f32.h) for sizes that are multiples of four, and one
// workgroup per routed row for the rest and for the stage entry points, which have no room for pre-activations.
// Follow BiBoFusedExperts.forward, src/modeling/ffn/moe.py:73-101 of the reference.
#include "tile_f32.h"

namespace bibo {
namespace {

__device__ __forceinline__ int find_expert(const int32_t* __restrict__ offsets, int E, int row, int* sh) {
  // offsets is non-decreasing; the owner is the last expert with offsets[e] <= row < offsets[e+1]
  const int tid = threadIdx.x;
  if (tid < E && offsets[tid] <= row && row < offsets[tid + 1]) *sh = tid;
  __syncthreads();
  return *sh;
}

// hidden[row, :] = r^p * SiLU(g/r) * up   (moe.py:84-92)
template <typename TIn>
__global__ __launch_bounds__(256) void gateup_generic_kernel(const TIn* __restrict__ x, const TIn* __restrict__ wgu,
                                                             const float* __restrict__ theta,
                                                             const int32_t* __restrict__ offsets,
                                                             const int32_t* __restrict__ perm_token, int H, int E,
                                                             int I, int act, TIn* __restrict__ hidden) {
  extern __shared__ float smem[];
  float* xs = smem;            // [H]
  float* gu = smem + H;        // [2I]
  __shared__ int sh_e;
  __shared__ float red[4];
  const int row = blockIdx.x;
  if (row >= offsets[E]) return;
  const int e = find_expert(offsets, E, row, &sh_e);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const TIn* xr = x + (size_t)perm_token[row] * H;                     // moe.py:81
  for (int h = tid; h < H; h += 256) xs[h] = to_float(xr[h]);
  __syncthreads();
  const TIn* wbase = wgu + (size_t)e * 2 * I * H;
  for (int j = wave; j < 2 * I; j += 4) {                              // moe.py:84
    const TIn* wrow = wbase + (size_t)j * H;
    float acc = 0.f;
    for (int h = lane; h < H; h += kWave) acc = fmaf(xs[h], to_float(wrow[h]), acc);
    acc = wave_sum(acc);
    if (lane == 0) gu[j] = acc;
  }
  __syncthreads();
  float ss = 0.f;
  for (int i = tid; i < I; i += 256) ss = fmaf(gu[i], gu[i], ss);
  ss = wave_sum(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  const float ms = ((red[0] + red[1]) + red[2]) + red[3];
  const float r = act == BIBO_ACT_SILU ? 1.f : sqrtf(ms / (float)I + kNormSiluEps);   // moe.py:88
  const float p = radial_exponent(theta, e, act);                      // moe.py:89
  const float gain = act == BIBO_ACT_SILU ? 1.f : powf(r, p);
  for (int i = tid; i < I; i += 256) {
    const float z = gu[i] / r;
    const float act = z / (1.f + expf(-z)) * gain;                     // SiLU(g/r) * r^p
    hidden[(size_t)row * I + i] = from_float<TIn>(act * gu[I + i]);    // * up (moe.py:92)
  }
}

// yw[slot, :] = w[slot] * (hidden[row, :] @ w_down[e]^T)   (moe.py:92-93)
template <typename TIn>
__global__ __launch_bounds__(256) void down_generic_kernel(const TIn* __restrict__ hidden, const TIn* __restrict__ wd,
                                                           const float* __restrict__ w,
                                                           const int32_t* __restrict__ offsets,
                                                           const int32_t* __restrict__ perm_slot, int H, int E, int I,
                                                           float* __restrict__ yw) {
  extern __shared__ float smem[];
  float* hs = smem;            // [I]
  __shared__ int sh_e;
  const int row = blockIdx.x;
  if (row >= offsets[E]) return;
  const int e = find_expert(offsets, E, row, &sh_e);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  for (int i = tid; i < I; i += 256) hs[i] = to_float(hidden[(size_t)row * I + i]);
  __syncthreads();
  const int slot = perm_slot[row];
  const float ws = w[slot];
  const TIn* wbase = wd + (size_t)e * H * I;
  for (int h = wave; h < H; h += 4) {
    const TIn* wrow = wbase + (size_t)h * I;
    float acc = 0.f;
    for (int i = lane; i < I; i += kWave) acc = fmaf(hs[i], to_float(wrow[i]), acc);
    acc = wave_sum(acc);
    if (lane == 0) yw[(size_t)slot * H + h] = ws * acc;
  }
}

// hidden[row, :] = r^p SiLU(g/r) up (moe.py:87-92) from the fp32 pre-activations gu [S, 2I], one wave per permuted row.
// Bound by memory (a row is read twice, the second time from L1): 4 rows per workgroup keep enough loads in flight.
template <typename TIn>
__global__ __launch_bounds__(256) void activate_f32_kernel(const float* __restrict__ gu, const float* __restrict__ theta,
                                                           const int32_t* __restrict__ offsets, int S, int E, int I, int act,
                                                           TIn* __restrict__ hidden) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= S) return;
  const int e = expert_of_row(offsets, E, row);
  if (e < 0) return;
  const float* g = gu + (size_t)row * 2 * I;
  float ss = 0.f;
  for (int c = lane * 4; c < I; c += 4 * kWave) {
    const floatx4 v = load4<float>(g + c);
#pragma unroll
    for (int q = 0; q < 4; ++q) ss = fmaf(v[q], v[q], ss);
  }
  ss = wave_sum(ss);
  const float r = act == BIBO_ACT_SILU ? 1.f : sqrtf(ss / (float)I + kNormSiluEps);   // moe.py:88
  const float gain = act == BIBO_ACT_SILU ? 1.f : powf(r, radial_exponent(theta, e, act));
  for (int c = lane * 4; c < I; c += 4 * kWave) {
    const floatx4 v = load4<float>(g + c), u = load4<float>(g + I + c);
    floatx4 h;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float z = v[q] / r;
      h[q] = (float)((double)(z / (1.f + expf(-z))) * gain * u[q]);    // SiLU(g/r) r^p up, rounded once
    }
    store4(hidden + (size_t)row * I + c, h);
  }
}

// out[t, :] = round(residual[t, :] + sum_j contribution(t, j))  in fp32, ascending j   (moe.py:93-101; the residual
// add of the caller, src/modeling/layers.py:62, when `residual` is given).  contribution = yw[t*k + j, :] for a GLU
// expert; with `idx` given, +/- w[t,j] * x[t, :] for a +/-Identity special (moe.py:95-99) and nothing for an index
// outside [0, E_glu + n_pos + n_neg) (no kernel wrote that slot's row).
template <typename TX>
__device__ __forceinline__ bool special_slot(const CombineArgs& a, size_t slot, int* sign) {
  *sign = 0;
  if (a.idx == nullptr) return false;
  const int e = a.idx[slot];
  if ((unsigned)e >= (unsigned)(a.E_glu + a.n_pos + a.n_neg)) return true;       // skipped
  if (e < a.E_glu) return false;
  *sign = e < a.E_glu + a.n_pos ? 1 : -1;
  return true;
}

// The workgroups of a combine kernel that sum rows, and whether this one is not of them but takes the balancing step: a launch less for a training
// forward (H = 512, T = 1111: 4 us of host time, 2 to 5 us on the GPU).
__device__ __forceinline__ bool balance_workgroup(const CombineArgs& a, unsigned& workgroups) {
  workgroups = gridDim.x - (a.balance.counts != nullptr ? 1u : 0u);
  if (blockIdx.x < workgroups) return false;
  if (threadIdx.x < kWave) balance_step(a.balance);
  return true;
}

template <typename TY, typename TOut>
__global__ __launch_bounds__(256) void combine_kernel(const TY* __restrict__ yw, CombineArgs a, int T, int H, int k,
                                                      TOut* __restrict__ out) {
  unsigned workgroups;
  if (balance_workgroup(a, workgroups)) return;
  const size_t n = (size_t)T * H;
  const TOut* x = static_cast<const TOut*>(a.x);
  const TOut* residual = static_cast<const TOut*>(a.residual);
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)workgroups * 256) {
    const size_t t = i / H, h = i - t * H;
    float acc = 0.f;
    for (int j = 0; j < k; ++j) {
      int sign;
      if (special_slot<TOut>(a, t * k + j, &sign)) {
        if (sign != 0) acc += (float)sign * a.w[t * k + j] * to_float(x[i]);
        continue;
      }
      acc += to_float(yw[(t * k + j) * H + h]);
    }
    if (residual != nullptr) acc = (a.round_block ? to_float(from_float<TOut>(acc)) : acc) + to_float(residual[i]);
    out[i] = from_float<TOut>(acc);
  }
}

// bf16 slot rows -> bf16 output, 8 columns (16 bytes) per thread, fp32 sum in ascending j
__global__ __launch_bounds__(256) void combine_bf16x8_kernel(const bf16_t* __restrict__ yw, CombineArgs a, int T, int H8,
                                                             int k, bf16_t* __restrict__ out) {
  unsigned workgroups;
  if (balance_workgroup(a, workgroups)) return;
  const size_t n = (size_t)T * H8;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)workgroups * 256) {
    const size_t t = i / H8, c = i - t * H8;
    float acc[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) acc[q] = 0.f;
    const bf16x8* src = reinterpret_cast<const bf16x8*>(yw) + (t * k) * H8 + c;
    for (int j = 0; j < k; ++j) {
      int sign;
      if (special_slot<bf16_t>(a, t * k + j, &sign)) {
        if (sign != 0) {
          const float sw = (float)sign * a.w[t * k + j];
          const bf16x8 xv = reinterpret_cast<const bf16x8*>(a.x)[i];
#pragma unroll
          for (int q = 0; q < 8; ++q) acc[q] += sw * (float)xv[q];
        }
        continue;
      }
      const bf16x8 v = src[(size_t)j * H8];
#pragma unroll
      for (int q = 0; q < 8; ++q) acc[q] += (float)v[q];
    }
    if (a.residual != nullptr) {
      const bf16x8 r = reinterpret_cast<const bf16x8*>(a.residual)[i];
#pragma unroll
      for (int q = 0; q < 8; ++q) acc[q] = (a.round_block ? (float)(bf16_t)acc[q] : acc[q]) + (float)r[q];
    }
    bf16x8 o;
#pragma unroll
    for (int q = 0; q < 8; ++q) o[q] = (bf16_t)acc[q];
    reinterpret_cast<bf16x8*>(out)[i] = o;
  }
}

// fp32 slot rows -> bf16 or fp32 output, 4 columns per thread: the decode-size combine, whose duration is one round trip of
// its loads, issues a quarter of the threads and all k loads of a thread at once.  Same sum as combine_kernel.
template <typename TOut>
__global__ __launch_bounds__(256) void combine_f32x4_kernel(const float* __restrict__ yw, CombineArgs a, int T, int H4,
                                                            int k, TOut* __restrict__ out) {
  unsigned workgroups;
  if (balance_workgroup(a, workgroups)) return;
  const TOut* x = static_cast<const TOut*>(a.x);
  const TOut* residual = static_cast<const TOut*>(a.residual);
  const size_t n = (size_t)T * H4;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)workgroups * 256) {
    const size_t t = i / H4, c = i - t * H4;
    floatx4 v[kMaxK];
    int sign[kMaxK];
    bool special[kMaxK];
    const floatx4* src = reinterpret_cast<const floatx4*>(yw) + (t * k) * H4 + c;
#pragma unroll
    for (int j = 0; j < kMaxK; ++j)
      if (j < k) {
        special[j] = special_slot<TOut>(a, t * k + j, &sign[j]);
        if (!special[j]) v[j] = src[(size_t)j * H4];
      }
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < kMaxK; ++j)
      if (j < k) {
        if (special[j]) {
          if (sign[j] != 0) {
            const float sw = (float)sign[j] * a.w[t * k + j];
            const floatx4 xv = load4<TOut>(x + i * 4);
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[q] += sw * xv[q];
          }
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[q] += v[j][q];
        }
      }
    if (residual != nullptr) {
      const floatx4 r = load4<TOut>(residual + i * 4);
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = (a.round_block ? to_float(from_float<TOut>(acc[q])) : acc[q]) + r[q];
    }
    store4(out + i * 4, floatx4{acc[0], acc[1], acc[2], acc[3]});
  }
}

}  // namespace

hipError_t launch_gateup_generic(const void* x, const void* wgu, const float* theta, const int32_t* offsets,
                                 const int32_t* perm_token, int T, int H, int E, int k, int I, int dtype, int act,
                                 void* hidden, hipStream_t s) {
  const int S = T * k;
  if (S == 0) return hipSuccess;
  const size_t shm = (size_t)(H + 2 * I) * sizeof(float);
  if (dtype == BIBO_DTYPE_BF16)
    hipLaunchKernelGGL(gateup_generic_kernel<bf16_t>, dim3(S), dim3(256), shm, s, static_cast<const bf16_t*>(x),
                       static_cast<const bf16_t*>(wgu), theta, offsets, perm_token, H, E, I, act,
                       static_cast<bf16_t*>(hidden));
  else
    hipLaunchKernelGGL(gateup_generic_kernel<float>, dim3(S), dim3(256), shm, s, static_cast<const float*>(x),
                       static_cast<const float*>(wgu), theta, offsets, perm_token, H, E, I, act,
                       static_cast<float*>(hidden));
  return hipGetLastError();
}

hipError_t launch_down_generic(const void* hidden, const void* wd, const float* w, const int32_t* offsets,
                               const int32_t* perm_slot, int T, int H, int E, int k, int I, int dtype, float* yw,
                               hipStream_t s) {
  const int S = T * k;
  if (S == 0) return hipSuccess;
  const size_t shm = (size_t)I * sizeof(float);
  if (dtype == BIBO_DTYPE_BF16)
    hipLaunchKernelGGL(down_generic_kernel<bf16_t>, dim3(S), dim3(256), shm, s, static_cast<const bf16_t*>(hidden),
                       static_cast<const bf16_t*>(wd), w, offsets, perm_slot, H, E, I, yw);
  else
    hipLaunchKernelGGL(down_generic_kernel<float>, dim3(S), dim3(256), shm, s, static_cast<const float*>(hidden),
                       static_cast<const float*>(wd), w, offsets, perm_slot, H, E, I, yw);
  return hipGetLastError();
}

bool tile_f32_supported(int H, int I) { return H % 4 == 0 && I % 4 == 0; }

// The experts of the generic family as three launches: gu = x W_gate_up^T (fp32, [S, 2I], permuted rows), the activation,
// yw[slot] = w[slot] hidden W_down^T.  `gu` may share its memory with `yw`.  At T = 2048, H = 768, E = 64, k = 6, I = 384 in
// fp32 the row kernels took 5088 + 2688 us: every routed row read its expert's 3.5 MB through one CU.
template <typename TIn>
static hipError_t launch_experts_tiled_t(const TIn* x, const TIn* wgu, const TIn* wd, const float* theta, const float* w,
                                         const int32_t* offsets, const int32_t* perm_slot, const int32_t* perm_token, int S,
                                         int H, int E, int I, int act, float* gu, TIn* hidden, float* yw, hipStream_t s) {
  hipError_t err = launch_ggemm_f32<TIn, TIn, false, true, false>(x, perm_token, wgu, offsets, nullptr, nullptr, S, H, 2 * I, E, gu, s);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(activate_f32_kernel<TIn>, dim3((S + 3) / 4), dim3(256), 0, s, gu, theta, offsets, S, E, I, act, hidden);
  return launch_ggemm_f32<TIn, TIn, false, false, true>(hidden, nullptr, wd, offsets, perm_slot, w, S, I, H, E, yw, s);
}

hipError_t launch_experts_tiled(const void* x, const void* wgu, const void* wd, const float* theta, const float* w,
                                const int32_t* offsets, const int32_t* perm_slot, const int32_t* perm_token, int T, int H,
                                int E, int k, int I, int dtype, int act, float* gu, void* hidden, float* yw, hipStream_t s) {
  const int S = T * k;
  if (S == 0) return hipSuccess;
  if (dtype == BIBO_DTYPE_BF16)
    return launch_experts_tiled_t(static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(wgu), static_cast<const bf16_t*>(wd), theta,
                                  w, offsets, perm_slot, perm_token, S, H, E, I, act, gu, static_cast<bf16_t*>(hidden), yw, s);
  return launch_experts_tiled_t(static_cast<const float*>(x), static_cast<const float*>(wgu), static_cast<const float*>(wd), theta, w,
                                offsets, perm_slot, perm_token, S, H, E, I, act, gu, static_cast<float*>(hidden), yw, s);
}

hipError_t launch_combine(const void* yw, int yw_is_bf16, const CombineArgs& a, int T, int H, int k, int dtype,
                          void* out, hipStream_t s) {
  const size_t n = (size_t)T * H;
  if (n == 0) return a.balance.counts != nullptr ? launch_balance_step(a.balance, s) : hipSuccess;
  const int more = a.balance.counts != nullptr ? 1 : 0;
  const int grid = (int)((n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536);
  if (yw_is_bf16) {
    if (dtype != BIBO_DTYPE_BF16) return hipErrorInvalidValue;
    if ((H % 8) == 0 && ((reinterpret_cast<uintptr_t>(yw) | reinterpret_cast<uintptr_t>(out) |
                          reinterpret_cast<uintptr_t>(a.residual) | reinterpret_cast<uintptr_t>(a.x)) & 15) == 0) {
      const size_t n8 = n / 8;
      const int g8 = (int)((n8 + 255) / 256 < 65536 ? (n8 + 255) / 256 : 65536);
      hipLaunchKernelGGL(combine_bf16x8_kernel, dim3(g8 + more), dim3(256), 0, s, static_cast<const bf16_t*>(yw), a, T, H / 8, k,
                         static_cast<bf16_t*>(out));
    } else
      hipLaunchKernelGGL((combine_kernel<bf16_t, bf16_t>), dim3(grid + more), dim3(256), 0, s,
                         static_cast<const bf16_t*>(yw), a, T, H, k, static_cast<bf16_t*>(out));
  } else {
    const bool vec = (H % 4) == 0 && ((reinterpret_cast<uintptr_t>(yw) | reinterpret_cast<uintptr_t>(out) |
                                       reinterpret_cast<uintptr_t>(a.residual) | reinterpret_cast<uintptr_t>(a.x)) & 15) == 0;
    const size_t n4 = n / 4;
    const int g4 = (int)((n4 + 255) / 256 < 65536 ? (n4 + 255) / 256 : 65536);
    const float* yp = static_cast<const float*>(yw);
    if (dtype == BIBO_DTYPE_BF16) {
      bf16_t* op = static_cast<bf16_t*>(out);
      if (vec) hipLaunchKernelGGL(combine_f32x4_kernel<bf16_t>, dim3(g4 + more), dim3(256), 0, s, yp, a, T, H / 4, k, op);
      else hipLaunchKernelGGL((combine_kernel<float, bf16_t>), dim3(grid + more), dim3(256), 0, s, yp, a, T, H, k, op);
    } else {
      float* op = static_cast<float*>(out);
      if (vec) hipLaunchKernelGGL(combine_f32x4_kernel<float>, dim3(g4 + more), dim3(256), 0, s, yp, a, T, H / 4, k, op);
      else hipLaunchKernelGGL((combine_kernel<float, float>), dim3(grid + more), dim3(256), 0, s, yp, a, T, H, k, op);
    }
  }
  return hipGetLastError();
}

}  // namespace bibo
