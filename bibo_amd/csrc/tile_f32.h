// Grouped GEMMs in fp32 arithmetic for the generic family (fp32 operands, and bf16 sizes no bf16 tile divides), gfx950.
//
// v_mfma_f32_32x32x2_f32 / 16x16x4_f32 multiply fp32 operands at 154 TFLOP/s (what a library product of 4096 x 8192 x 8192
// reaches on this chip), twice what scalar FMAs could; at that rate one CU needs 38 GB/s for a 64 x 64 tile, far below
// what L2 delivers, so small tiles are enough and several workgroups per CU hide the latency of plain register loads.
// Operands are widened to fp32 on their way to LDS, so one kernel serves both operand types.
//
// LDS layouts of a K step of 32:
//   K-contiguous operand (rows of K elements in memory): [rows][32], 128-byte rows; 16-byte granule c of row r sits at
//     c ^ ((r >> 1) & 7), so 16 consecutive rows read without bank conflicts.  A lane reads a granule (4 consecutive k)
//     and feeds its four elements to four MFMAs.
//   K-major operand (element (k, n) at k * ld + n): [32][columns] as it lies; a lane reads one element per MFMA, 32 lanes
//     on 128 consecutive bytes.
// Both sides use the same k for the same MFMA (the order of the K elements inside a step does not matter otherwise).
//
// How ggemm_f32_kernel sums a dot product: chains of eight products inside the MFMAs, a step's four chains in fp32, the steps in
// fp64.  One chain over all of K, which the accumulators would form by themselves, is as far from the exact result as the square
// root of its length says: the layer at H = 768, I = 384 was off by 8.4e-7 (2-norm), one routed row at a time, whose dot products
// are 64 partial sums and a tree, by 1.81e-7, this by 1.49e-7, and by no more than one row at a time from H = 64 to 1024.  The sums
// cost 80 vector instructions beside the 16 MFMAs of a step: T = 2048, H = 768, E = 64, k = 6, I = 384 takes 323 us and took 292
// (319 us with fp32 in the place of fp64, 336 with fp64 sums of every sixteen products).  120 registers keep four workgroups on a
// CU, which is what hides one's sums behind the others' MFMAs: a chain goes into its sum as soon as it ends.
#pragma once

#include "stripe.h"

namespace bibo {
namespace {

constexpr int kFK = 32;        // K elements per step

template <typename T> __device__ __forceinline__ floatx4 load4(const T* p);
template <> __device__ __forceinline__ floatx4 load4<float>(const float* p) { return *reinterpret_cast<const floatx4*>(p); }
template <> __device__ __forceinline__ floatx4 load4<bf16_t>(const bf16_t* p) {
  const bf16x4 v = *reinterpret_cast<const bf16x4*>(p);
  return floatx4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}
__device__ __forceinline__ void store4(float* p, floatx4 v) { *reinterpret_cast<floatx4*>(p) = v; }
__device__ __forceinline__ void store4(bf16_t* p, floatx4 v) {
  *reinterpret_cast<bf16x4*>(p) = bf16x4{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
}

__device__ __forceinline__ int fswz(int row, int c) { return row * kFK + ((c ^ ((row >> 1) & 7)) << 2); }

// out[dst(r), n] = scale(r) * sum_k A[src(r), k] W[e](k, n) for the rows r of expert e.  src(r) = a_index[r] (GATHER) or
// r; dst(r) = out_index[r] and scale(r) = out_scale[out_index[r]] (SCATTER; out_scale == NULL: 1) or r and 1.  W[e] is
// [N, K] (K-contiguous) or, with W_KM, [K, N].  K, N multiples of 4, rows 16-byte (bf16: 8-byte) aligned.
// BM = 64: 64 rows x 64 columns, 2 x 2 waves of 32x32 tiles.  BM = 16 (few rows per expert): 16 rows x 64 columns, four
// waves along the columns, 16x16 tiles: a quarter of the MFMA time per streamed weight byte, which is what counts there.
template <typename TA, typename TW, bool W_KM, bool GATHER, bool SCATTER, int BM>
__global__ __launch_bounds__(256, 4) void ggemm_f32_kernel(const TA* __restrict__ A, const int32_t* __restrict__ a_index,
                                                        const TW* __restrict__ W, const int32_t* __restrict__ offsets,
                                                        const int32_t* __restrict__ out_index,
                                                        const float* __restrict__ out_scale, int K, int N, int E, int nblk_n,
                                                        float* __restrict__ out) {
  static_assert(BM == 64 || (BM == 16 && !W_KM), "tile shapes");
  constexpr int BN = 64;
  constexpr int A_PER = BM == 64 ? 2 : 1, W_PER = 2;            // granules of four elements per thread and step
  __shared__ __attribute__((aligned(16))) float As[2][BM * kFK];
  __shared__ __attribute__((aligned(16))) float Ws[2][BN * kFK];
  __shared__ int dst_s[BM];
  __shared__ float scale_s[BM];

  const TileMap tm = make_tile_map(offsets, E, BM);
  const int total = tm.total * nblk_n;
  const int flat = xcd_tile(blockIdx.x, total);
  if (flat >= total) return;
  const int tile = flat / nblk_n, nb = flat - tile * nblk_n;
  int e, row0, rows;
  find_tile(tm, tile, e, row0, rows);
  e = __builtin_amdgcn_readfirstlane(e);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int n0 = nb * BN;
  if (tid < BM) {
    const int r = row0 + min(tid, rows - 1);
    const int d = SCATTER ? out_index[r] : r;
    dst_s[tid] = d;
    scale_s[tid] = SCATTER && out_scale != nullptr ? out_scale[d] : 1.f;
  }
  const TA* arow[A_PER];
  int ac = tid & 7;
  const bool a_live = BM == 64 || tid < BM * 8;
#pragma unroll
  for (int i = 0; i < A_PER; ++i) {
    const int r = row0 + min((tid >> 3) + 32 * i, rows - 1);     // rows past the end repeat the last one
    arow[i] = A + (size_t)(GATHER ? a_index[r] : r) * K;
  }
  const TW* wbase = W + (size_t)e * K * N;
  floatx4 ra[A_PER], rw[W_PER];
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < A_PER; ++i) ra[i] = a_live && k0 + ac * 4 < K ? load4<TA>(arow[i] + k0 + ac * 4) : zero;
#pragma unroll
    for (int i = 0; i < W_PER; ++i) {
      const int g = tid + 256 * i;
      if constexpr (W_KM) {
        const int kr = k0 + g / (BN / 4), n = n0 + (g % (BN / 4)) * 4;
        rw[i] = kr < K && n < N ? load4<TW>(wbase + (size_t)kr * N + n) : zero;
      } else {
        const int n = n0 + (g >> 3), k = k0 + (g & 7) * 4;
        rw[i] = n < N && k < K ? load4<TW>(wbase + (size_t)n * K + k) : zero;
      }
    }
  };
  auto store = [&](int st) {
#pragma unroll
    for (int i = 0; i < A_PER; ++i)
      if (a_live) *reinterpret_cast<floatx4*>(&As[st][fswz((tid >> 3) + 32 * i, ac)]) = ra[i];
#pragma unroll
    for (int i = 0; i < W_PER; ++i) {
      const int g = tid + 256 * i;
      *reinterpret_cast<floatx4*>(&Ws[st][W_KM ? g * 4 : fswz(g >> 3, g & 7)]) = rw[i];
    }
  };
  const int nsteps = (K + kFK - 1) / kFK;
  load(0);
  store(0);
  __syncthreads();
  if constexpr (BM == 64) {
    const int wm = wave & 1, wn = wave >> 1, l32 = lane & 31, h = lane >> 5;
    const int n = n0 + wn * 32 + l32;
    floatx16 none, part;
    double sum[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) { none[i] = 0.f; sum[i] = 0.; }
    for (int s = 0; s < nsteps; ++s) {
      if (s + 1 < nsteps) load((s + 1) * kFK);
      const float* as = As[s & 1];
      const float* ws = Ws[s & 1];
#pragma unroll
      for (int ks = 0; ks < kFK / 8; ++ks) {
        const floatx4 a = *reinterpret_cast<const floatx4*>(as + fswz(wm * 32 + l32, 2 * ks + h));
        floatx4 b;
        if constexpr (W_KM) {
#pragma unroll
          for (int q = 0; q < 4; ++q) b[q] = ws[(8 * ks + 4 * h + q) * BN + wn * 32 + l32];
        } else {
          b = *reinterpret_cast<const floatx4*>(ws + fswz(wn * 32 + l32, 2 * ks + h));
        }
        floatx16 acc = none;
#pragma unroll
        for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q], b[q], acc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) part[i] = ks == 0 ? acc[i] : part[i] + acc[i];
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        sum[i] += (double)part[i];
        asm volatile("" : "+v"(sum[i]));   // here: moved behind the barrier it keeps 64 more registers alive
      }
      if (s + 1 < nsteps) store((s + 1) & 1);
      __syncthreads();
    }
    // lane = column lane % 32, register i = row 8 (i / 4) + 4 (lane / 32) + i % 4: a store covers 128 bytes of two rows
    if (n < N) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int m = wm * 32 + acc_row(i, lane);
        if (m < rows) out[(size_t)dst_s[m] * N + n] = (float)(scale_s[m] * sum[i]);
      }
    }
  } else {
    const int l16 = lane & 15, g4 = lane >> 4;
    double sum[4] = {0., 0., 0., 0.};
    for (int s = 0; s < nsteps; ++s) {
      if (s + 1 < nsteps) load((s + 1) * kFK);
      const float* as = As[s & 1];
      const float* ws = Ws[s & 1];
      floatx4 part[2][2];
#pragma unroll
      for (int ks = 0; ks < kFK / 16; ++ks) {
        const floatx4 a = *reinterpret_cast<const floatx4*>(as + fswz(l16, 4 * ks + g4));
        const floatx4 b = *reinterpret_cast<const floatx4*>(ws + fswz(wave * 16 + l16, 4 * ks + g4));
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          part[ks][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[2 * c], b[2 * c], zero, 0, 0, 0);
          part[ks][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[2 * c + 1], b[2 * c + 1], part[ks][c], 0, 0, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[i] += (double)((part[0][0][i] + part[0][1][i]) + (part[1][0][i] + part[1][1][i]));
      if (s + 1 < nsteps) store((s + 1) & 1);
      __syncthreads();
    }
    const int n = n0 + wave * 16 + l16;
    if (n < N) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = 4 * g4 + i;
        if (m < rows) out[(size_t)dst_s[m] * N + n] = (float)(scale_s[m] * sum[i]);
      }
    }
  }
}

// 16-row tiles up to this many rows per expert on average: a 64-row tile multiplies up to 63 rows that are not there, a 16-row tile
// streams its weights four times as often, from L2.  Layer times in fp32, 64-row -> 16-row tiles: H = 768, I = 384, E = 64, k = 6:
// 116 -> 80 us at 9 rows, 117 -> 116 at 31, 213 -> 199 at 96, 221 -> 223 at 111, 326 -> 343 at 192; H = 1024, I = 512, k = 8: 175 -> 128
// at 10, 311 -> 281 at 80, 322 -> 321 at 96, 347 -> 369 at 112; H = 192, I = 88, E = 16, k = 3: 34 -> 30 at 96, 49 -> 44 at 384.  (Where
// the rows just fill 64, e.g. 36 to 40 at H = 768, the 64-row tiles are 2 % ahead.)
constexpr int kFewRows = 96;

template <typename TA, typename TW, bool W_KM, bool GATHER, bool SCATTER>
hipError_t launch_ggemm_f32(const TA* A, const int32_t* a_index, const TW* W, const int32_t* offsets, const int32_t* out_index,
                            const float* out_scale, int S, int K, int N, int E, float* out, hipStream_t s) {
  auto grid = [&](int BM, int nblk_n) {
    const long long tiles = (long long)(S / BM + E < S ? S / BM + E : S) * nblk_n;
    return dim3((unsigned)(((tiles + 7) & ~7ll) + 8));
  };
  const int nblk = (N + 63) / 64;
  if constexpr (!W_KM) {
    if ((long long)S <= (long long)kFewRows * E) {
      hipLaunchKernelGGL((ggemm_f32_kernel<TA, TW, false, GATHER, SCATTER, 16>), grid(16, nblk), dim3(256), 0, s, A, a_index, W,
                         offsets, out_index, out_scale, K, N, E, nblk, out);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((ggemm_f32_kernel<TA, TW, W_KM, GATHER, SCATTER, 64>), grid(64, nblk), dim3(256), 0, s, A, a_index, W,
                     offsets, out_index, out_scale, K, N, E, nblk, out);
  return hipGetLastError();
}

// dW[e][n][m] = sum over the rows r of expert e of P[srcP(r)][n] Q[srcQ(r)][m]; srcP(r) = index[r] (GATHER_P) or r, likewise
// Q.  Both operands K-major (the contraction runs over rows).  Workgroup = 64 x 64 of dW, 2 x 2 waves.  N, M multiples
// of 4.  Rows past the expert's end count as zeros.
template <typename TP, typename TQ, typename TOut, bool GATHER_P, bool GATHER_Q>
__global__ __launch_bounds__(256) void wgrad_f32_kernel(const TP* __restrict__ P, const TQ* __restrict__ Q,
                                                        const int32_t* __restrict__ index, const int32_t* __restrict__ offsets,
                                                        int N, int M, int E, int nblk_n, int nblk_m, TOut* __restrict__ dW) {
  constexpr int B = 64;
  __shared__ __attribute__((aligned(16))) float Ps[2][B * kFK];
  __shared__ __attribute__((aligned(16))) float Qs[2][B * kFK];
  const int per_e = nblk_n * nblk_m;
  const int item = xcd_tile(blockIdx.x, E * per_e);
  if (item >= E * per_e) return;
  const int e = item / per_e, rest = item - e * per_e;
  const int n0 = (rest / nblk_m) * B, m0 = (rest % nblk_m) * B;
  const int lo = offsets[e], hi = offsets[e + 1];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int kr = tid >> 4, c4 = (tid & 15) * 4;          // this thread's rows kr, kr + 16 of a step, four columns
  const bool p_live = n0 + c4 < N, q_live = m0 + c4 < M;
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  floatx4 rp[2], rq[2];
  int ix[2];
  auto lookup = [&](int r0) {                            // row indices of a gathered operand, one step ahead of its loads
    if constexpr (GATHER_P || GATHER_Q) {
#pragma unroll
      for (int i = 0; i < 2; ++i) ix[i] = r0 + kr + 16 * i < hi ? index[r0 + kr + 16 * i] : 0;
    }
  };
  auto load = [&](int r0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = r0 + kr + 16 * i;
      const bool live = r < hi;
      rp[i] = live && p_live ? load4<TP>(P + (size_t)(GATHER_P ? ix[i] : r) * N + n0 + c4) : zero;
      rq[i] = live && q_live ? load4<TQ>(Q + (size_t)(GATHER_Q ? ix[i] : r) * M + m0 + c4) : zero;
    }
  };
  auto store = [&](int st) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      *reinterpret_cast<floatx4*>(&Ps[st][(kr + 16 * i) * B + c4]) = rp[i];
      *reinterpret_cast<floatx4*>(&Qs[st][(kr + 16 * i) * B + c4]) = rq[i];
    }
  };
  const int wm = wave & 1, wn = wave >> 1, l32 = lane & 31, h = lane >> 5;
  floatx16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  const int nsteps = (hi - lo + kFK - 1) / kFK;
  if (nsteps > 0) {
    lookup(lo);
    load(lo);
    lookup(lo + kFK);
    store(0);
    __syncthreads();
    for (int s = 0; s < nsteps; ++s) {
      if (s + 1 < nsteps) {
        load(lo + (s + 1) * kFK);
        lookup(lo + (s + 2) * kFK);
      }
      const float* ps = Ps[s & 1] + wm * 32 + l32;
      const float* qs = Qs[s & 1] + wn * 32 + l32;
#pragma unroll
      for (int k = 0; k < kFK; k += 2)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ps[(k + h) * B], qs[(k + h) * B], acc, 0, 0, 0);
      if (s + 1 < nsteps) store((s + 1) & 1);
      __syncthreads();
    }
  }
  const int m = m0 + wn * 32 + l32;
  if (m < M) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int n = n0 + wm * 32 + acc_row(i, lane);
      if (n < N) dW[((size_t)e * N + n) * M + m] = from_float<TOut>(acc[i]);
    }
  }
}

template <typename TP, typename TQ, typename TOut, bool GATHER_P, bool GATHER_Q>
hipError_t launch_wgrad_f32(const TP* P, const TQ* Q, const int32_t* index, const int32_t* offsets, int N, int M, int E, TOut* dW,
                            hipStream_t s) {
  const int nblk_n = (N + 63) / 64, nblk_m = (M + 63) / 64;
  const unsigned grid = (unsigned)((E * nblk_n * nblk_m + 7) & ~7);
  hipLaunchKernelGGL((wgrad_f32_kernel<TP, TQ, TOut, GATHER_P, GATHER_Q>), dim3(grid), dim3(256), 0, s, P, Q, index, offsets, N, M,
                     E, nblk_n, nblk_m, dW);
  return hipGetLastError();
}

// expert of a permuted row, by the wave that owns the row: one offset per lane and a ballot.  -1: the row lies behind the
// E experts that have weights.
__device__ __forceinline__ int expert_of_row(const int32_t* __restrict__ offsets, int E, int row) {
  const int lane = lane_id();
  const int my_off = offsets[min(lane, E)];
  const int end = E < kWave ? __shfl(my_off, E, kWave) : offsets[E];
  if (row >= end) return -1;
  return __popcll(__ballot(lane < E && my_off <= row)) - 1;
}

}  // namespace
}  // namespace bibo
