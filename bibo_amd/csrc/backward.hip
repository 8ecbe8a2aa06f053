// Backward pass of the sparse-MoE block, bf16, gfx950: the gradients torch.autograd derives for the reference's
// eager layer (src/modeling/ffn/moe.py:46-101,157-183, src/modeling/ffn/router.py:25-47) with the selection held
// fixed.  For a routed row (token t, expert e, combine weight w) the forward is
//     gu = W_gate_up[e] x_t,  r = sqrt(mean(g^2) + eps),  h = r^p SiLU(g / r) u,  y = W_down[e] h,  out_t += w y
// and the backward, for the upstream gradient d_t of out_t:
//     dh' = W_down[e]^T d_t            (grouped GEMM over the TRANSPOSED down weights)
//     dw  = <dh', h>,  dh = w dh'      (gradient of the combine weight; moe.py:93)
//     (dg, du, dtheta) from dh         (Radial NormSiLU backward, moe.py:87-92)
//     dx_t += W_gate_up[e]^T [dg, du]  (grouped GEMM over the TRANSPOSED gate/up weights)
//     dW_down[e] += (w d_t) h^T,  dW_gate_up[e] += [dg, du] x_t^T   (grouped GEMMs that contract over an expert's rows)
//     dlogit from dw (router.py:41-47), dW_router += dlogit^T x, dx += dlogit W_router.
// Every GEMM here runs on LDS-DMA stages and MFMAs.  The pre-activations are recomputed with the forward's
// operand layout (both operands contiguous along the contraction).  The input gradients contract over the middle
// dimension of the weight tensors and the weight gradients over the ROWS of row-major activations: those operands go
// to LDS as they lie in memory and are read through transposing LDS reads (kmajor.h), so nothing is transposed in
// memory and an expert's rows need no padding: a K stage that runs past an expert's last row reads a row of zeros.
#include "kmajor.h"

namespace bibo {
namespace {

constexpr int kBwdBK = 64;   // K elements per LDS stage of the GEMMs here: whole 128-byte lines per row

// ---- grouped GEMM: out[dst(r), n] = sum_k A[src(r), k] W[e][n, k] for the rows r of expert e ------------------
// src(r) = a_index[r] (GATHER) or r; dst(r) = out_index[r] (SCATTER) or r.  r runs over permuted rows.
template <int MT, int NTW, int WM, bool GATHER, bool SCATTER>
__global__ __launch_bounds__(256 * WM) void ggemm_kernel(const bf16_t* __restrict__ A, const int32_t* __restrict__ a_index,
                                                         const bf16_t* __restrict__ W,
                                                         const int32_t* __restrict__ offsets,
                                                         const int32_t* __restrict__ out_index, int K, int N, int E,
                                                         int nblk_n, bf16_t* __restrict__ out) {
  using S = Stripe<MT, NTW, WM, kBwdBK>;
  constexpr int BM = S::BM;
  constexpr int BN = S::BN;
  __shared__ __attribute__((aligned(16))) bf16_t st0[S::kStageElems];
  __shared__ __attribute__((aligned(16))) bf16_t st1[S::kStageElems];
  __shared__ int dst_s[BM];

  const TileMap tm = make_tile_map(offsets, E, BM);
  const int total = tm.total * nblk_n;
  const int flat = xcd_tile(blockIdx.x, total);
  if (flat >= total) return;
  const int tile = flat / nblk_n, nb = flat - tile * nblk_n;
  int e, row0, rows;
  find_tile(tm, tile, e, row0, rows);

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wn = wave & 3, wm = wave >> 2;
  if (tid < BM) {
    const int r = row0 + min(tid, rows - 1);
    dst_s[tid] = SCATTER ? out_index[r] : r;
  }
  const int chunk = S::dma_chunk(tid);
  StripeLoader<S> ld;
#pragma unroll
  for (int i = 0; i < S::A_PER; ++i) {
    const int r = row0 + min(S::dma_row(tid) + i * S::kRowsPerInstr, rows - 1);   // rows past the end re-read the last one
    const int src = GATHER ? a_index[r] : r;
    ld.a_src[i] = A + (size_t)src * K + chunk * 8;
  }
  const int n0 = nb * BN;
  ld.b_src = W + ((size_t)e * N + n0 + S::dma_row(tid)) * K + chunk * 8;
  ld.bstep = (size_t)S::kRowsPerInstr * K;
  ld.issue_stage(0, st0);
  floatx16 acc[MT][NTW];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < NTW; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mt][j][i] = 0.f;
  auto frag_row = [&](int j) { return (wn * NTW + j) * 32; };
  stripe_mainloop_dma<MT, NTW, WM, S::BK, true>(acc, ld, K, st0, st1, wm, frag_row);

  // Epilogue (accumulators transposed: lane = row, four consecutive columns per register quad): 32 rows at a time
  // through a wave-private LDS tile, out as 16-byte row segments.
  const int mbase = wm * MT * 32;
  const int n = lane & 31, hh = lane >> 5;
  constexpr int kOutCols = NTW * 32;
  constexpr int kOutStride = kOutCols + 8;          // +16 bytes staggers the rows over the banks
  static_assert((4 * WM / 2) * 32 * kOutStride <= S::kStageElems, "output staging does not fit a stage buffer");
  __syncthreads();                       // every wave is done reading the stage buffers
  bf16_t* otile = (wave < 4 * WM / 2 ? st0 : st1) + (wave % (4 * WM / 2)) * (32 * kOutStride);
  constexpr int kGranPerRow = kOutCols / 8;
  const int colbase = n0 + wn * kOutCols;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int j = 0; j < NTW; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        bf16x4 hv;
#pragma unroll
        for (int r = 0; r < 4; ++r) hv[r] = (bf16_t)acc[mt][j][4 * q + r];
        *reinterpret_cast<bf16x4*>(otile + n * kOutStride + j * 32 + 8 * q + 4 * hh) = hv;
      }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
    for (int g = lane; g < 32 * kGranPerRow; g += kWave) {
      const int ml = g / kGranPerRow, c = g - ml * kGranPerRow;
      const int m = mbase + mt * 32 + ml;
      if (m < rows)
        *reinterpret_cast<u32x4*>(out + (size_t)dst_s[m] * N + colbase + c * 8) =
            *reinterpret_cast<const u32x4*>(otile + ml * kOutStride + c * 8);
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_wave_barrier();
  }
}

template <int NTW, bool GATHER, bool SCATTER>
hipError_t launch_ggemm_t(const bf16_t* A, const int32_t* a_index, const bf16_t* W, const int32_t* offsets,
                          const int32_t* out_index, int S_rows, int K, int N, int E, bf16_t* out, hipStream_t s) {
  constexpr int MT = 2, WM = 2;
  using St = Stripe<MT, NTW, WM, kBwdBK>;
  const int nblk_n = N / St::BN;
  const int tiles = (S_rows / St::BM + E) * nblk_n;
  const int grid = ((tiles + 7) & ~7) + 8;
  hipLaunchKernelGGL((ggemm_kernel<MT, NTW, WM, GATHER, SCATTER>), dim3(grid), dim3(256 * WM), 0, s, A, a_index, W,
                     offsets, out_index, K, N, E, nblk_n, out);
  return hipGetLastError();
}

template <bool GATHER, bool SCATTER>
hipError_t launch_ggemm(const bf16_t* A, const int32_t* a_index, const bf16_t* W, const int32_t* offsets,
                        const int32_t* out_index, int S_rows, int K, int N, int E, bf16_t* out, hipStream_t s) {
  if (N % 384 == 0) return launch_ggemm_t<3, GATHER, SCATTER>(A, a_index, W, offsets, out_index, S_rows, K, N, E, out, s);
  if (N % 256 == 0) return launch_ggemm_t<2, GATHER, SCATTER>(A, a_index, W, offsets, out_index, S_rows, K, N, E, out, s);
  return launch_ggemm_t<1, GATHER, SCATTER>(A, a_index, W, offsets, out_index, S_rows, K, N, E, out, s);
}

// 256-row tiles stream an expert's weights through LDS half as often as 128-row tiles, and the workgroups of a launch run in rounds of one
// per CU (256 on this chip): the tall tiles pay when their rounds, weighted by 1.75, are fewer.  A round of them takes 1.4 to 1.5 times as long
// where both heights need one, and what the weight leaves out is not worth a call: dh' GEMM, lower -> taller tiles, us, E = 64, k = 6 and
// rounds in brackets: H = 768, I = 384: 19.4 -> 28.5 (T = 2048, 1 and 1), 21.9 -> 31.4 (4096, 1 and 1), 35.0 -> 31.8 (5000, 2 and 1),
// 39.8 -> 36.3 (8192, 2 and 1), 59.7 -> 61.6 (12,000, 3 and 2: stays low), 79.9 -> 68.7 (16,384, 4 and 2); H = 512, I = 256: 23.4 -> 20.4 (8192);
// H = 1024, I = 512: 45.6 -> 38.7 (4000), 77.3 -> 65.1 (8192); H = 640, I = 128: 16.2 -> 16.4 (8192).  Only for experts that hold 192 rows on
// average (a 256-row tile is then at least half full where it matters).
inline bool tall_tiles(int S_rows, int E, long long tiles_short, long long tiles_tall) {
  constexpr long long kCUs = 256;
  const long long rs = (tiles_short + kCUs - 1) / kCUs, rt = (tiles_tall + kCUs - 1) / kCUs;
  return (long long)S_rows >= 192ll * E && rt * 7 < rs * 4;
}

template <int NTW, bool GATHER, bool SCATTER>
hipError_t launch_dgrad_t(const bf16_t* A, const int32_t* a_index, const bf16_t* W, const int32_t* offsets,
                          const int32_t* out_index, int S_rows, int K, int N, int E, bf16_t* out, hipStream_t s) {
  constexpr int BN = kSubW * NTW;
  const int nblk_n = N / BN;
  // an expert's last tile is ragged: about half a tile per expert on top of the full ones
  const bool tall = tall_tiles(S_rows, E, (long long)(S_rows / 128 + E / 2) * nblk_n, (long long)(S_rows / 256 + E / 2) * nblk_n);
  const int tiles = (S_rows / (tall ? 256 : 128) + E) * nblk_n;
  const int grid = ((tiles + 7) & ~7) + 8;
  if (tall)
    hipLaunchKernelGGL((dgrad_kmajor_kernel<4, NTW, GATHER, SCATTER>), dim3(grid), dim3(512), 0, s, A, a_index, W, offsets,
                       out_index, K, N, E, nblk_n, out);
  else
    hipLaunchKernelGGL((dgrad_kmajor_kernel<2, NTW, GATHER, SCATTER>), dim3(grid), dim3(512), 0, s, A, a_index, W, offsets,
                       out_index, K, N, E, nblk_n, out);
  return hipGetLastError();
}

// out[dst(r)] = A[src(r)] W[e] with W [E, K, N] as stored (kmajor.h)
template <bool GATHER, bool SCATTER>
hipError_t launch_dgrad(const bf16_t* A, const int32_t* a_index, const bf16_t* W, const int32_t* offsets,
                        const int32_t* out_index, int S_rows, int K, int N, int E, bf16_t* out, hipStream_t s) {
  if (N % 384 == 0) return launch_dgrad_t<3, GATHER, SCATTER>(A, a_index, W, offsets, out_index, S_rows, K, N, E, out, s);
  if (N % 256 == 0) return launch_dgrad_t<2, GATHER, SCATTER>(A, a_index, W, offsets, out_index, S_rows, K, N, E, out, s);
  return launch_dgrad_t<1, GATHER, SCATTER>(A, a_index, W, offsets, out_index, S_rows, K, N, E, out, s);
}

// How many 128-column sub-tiles a workgroup takes of an extent.
inline int sub_tiles(int n) { return n % 384 == 0 ? 3 : n % 256 == 0 ? 2 : 1; }

// dx of every slot and both weight gradients (kmajor.h: backward_gemms_kernel).  256-row tiles, which stream the other operand half as
// often, from 128 rows per expert on, where the average expert fills a row tile of the lower ones and begins another, if the launch is several
// rounds of workgroups, whose last one the three products share.  Lower -> taller tiles, us, E = 64, k = 6 and rows per expert in brackets:
// H = 768, I = 384: 56 -> 59 (122), 60.5 -> 59.6 (131), 70 -> 63 (159), 79 -> 67 (192), 189 -> 151 (768); H = 512, I = 256: 31.6 -> 28.8 (131),
// 100 -> 86 (768); H = 768, I = 128: 29.6 -> 24.7 (131); H = 1024, I = 512, k = 8: 106 -> 95 (100), 122 -> 102 (150), 260 -> 211 (512).  In
// launches of one round and a bit (H = 512, I = 256, E = 9, k = 2): 13.9 -> 18.6 (494), 30.8 -> 33.1 (1333).
// Tall launches address rows by 32-bit offsets (kmajor.h: SMALL): from the first token of x and d_out, from the first row of a chunk in the
// others.
hipError_t launch_backward_gemms(BackwardGemms g, int T, int S, int chunk, int slots, hipStream_t s) {
  const int H = g.H, I = g.I, E = g.E, nh = sub_tiles(H), ni = sub_tiles(I), bh = kSubW * nh, bi = kSubW * ni;
  auto pad8 = [](long long n) { return (int)((n + 7) & ~7ll); };
  auto dx = [&](int rows) { return ((long long)S / rows + E) * (H / bh); };
  auto gu = [&](int rows) { return (long long)slots * (2 * I / rows) * (H / bh); };
  auto down = [&](int rows) { return (long long)slots * (H / rows) * (I / bi); };
  const long long widest = (long long)sizeof(bf16_t) * (H > 2 * I ? H : 2 * I);
  const bool near = T * widest < kNoRow && chunk * widest < kNoRow;
  const bool tall = near && (long long)S >= 128ll * E && dx(128) + gu(128) + down(128) > 3 * kCUs;
  const int rows = tall ? 256 : 128;                     // (2 I is a multiple of both: backward_supported)
  g.tall_d = tall && H % 256 == 0;
  g.n_dx = pad8(dx(rows));
  g.n_gu = pad8(gu(rows));
  const int n_d = pad8(down(g.tall_d ? 256 : 128));
  const dim3 grid((unsigned)(g.n_dx + g.n_gu + n_d));
  using std::integral_constant;
  auto launch = [&](auto hc, auto ic) {
    constexpr int NH = decltype(hc)::value, NI = decltype(ic)::value;
    if (tall) hipLaunchKernelGGL((backward_gemms_kernel<NH, NI, true>), grid, dim3(512), 0, s, g);
    else hipLaunchKernelGGL((backward_gemms_kernel<NH, NI, false>), grid, dim3(512), 0, s, g);
  };
  auto by_i = [&](auto hc) {
    if (ni == 3) launch(hc, integral_constant<int, 3>{});
    else if (ni == 2) launch(hc, integral_constant<int, 2>{});
    else launch(hc, integral_constant<int, 1>{});
  };
  if (nh == 3) by_i(integral_constant<int, 3>{});
  else if (nh == 2) by_i(integral_constant<int, 2>{});
  else by_i(integral_constant<int, 1>{});
  return hipGetLastError();
}

// ---- Radial NormSiLU backward (moe.py:87-92), one wave per permuted row ----------------------------------------
// h = r^p a u, a = SiLU(z) = z s, s = sigmoid(z), z = g / r, a' = s (1 + z (1 - s)); with q = dh u:
//   du = dh r^p a;  dg = q r^(p-1) a' + g / (I r) sum_i q_i (p r^(p-1) a_i - r^(p-2) a'_i g_i);
//   dtheta (the row's share) = p'(theta) ln r sum_i q_i r^p a_i;  dw = <dh', h>, dh = w dh'.
// `hidden` receives w h, the row the down projection's weight gradient contracts with d_out.
// act = SiLU: h = SiLU(g) u, dg = q a'(g), no theta.  Rows of I <= kActMaxI elements.
// Bound by its vector instructions: the divisions are IEEE ones and the row has three sums besides that of its squares.  T = 8192, k = 6, I = 384:
// 57 us for 226 MB, 4 TB/s; on the reciprocal unit, with two sums, 40 us.  That costs precision: a quotient off by an ulp in 14 of 525 rows
// of one element where these are the nearest floats, and gradients that are other numbers by 1e-4 of their norm.
constexpr int kActMaxI = 512;   // one 16-byte granule of the row per lane

__global__ __launch_bounds__(256) void act_bwd_kernel(const bf16_t* __restrict__ gu, const bf16_t* __restrict__ dhp,
                                                      const float* __restrict__ w, const float* __restrict__ theta,
                                                      const int32_t* __restrict__ offsets,
                                                      const int32_t* __restrict__ perm_slot, int S, int E, int I, int act,
                                                      bf16_t* __restrict__ dgu, bf16_t* __restrict__ hidden,
                                                      float* __restrict__ dw_slot, float* __restrict__ dtheta_row,
                                                      uint32_t* __restrict__ zero_words, int n_zero_words,
                                                      int* __restrict__ plan, int n_routed, int chunk, int slots) {
  // (the first workgroup also clears the row of zeros the weight-gradient kernels read past an expert's last row and,
  // with its first wave, lists the row chunks those kernels work through)
  if (blockIdx.x == 0) {
    for (int i = threadIdx.x; i < n_zero_words; i += 256) zero_words[i] = 0u;
    if (threadIdx.x < kWave) wgrad_plan(offsets, n_routed, chunk, slots, plan);
  }
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= S) return;
  // the row's values are requested first: nothing below that decides about the row depends on them
  const bool live = lane * 8 < I;
  bf16x8 gv, uv, dv;
#pragma unroll
  for (int q = 0; q < 8; ++q) gv[q] = uv[q] = dv[q] = (bf16_t)0.f;
  if (live) {
    gv = *reinterpret_cast<const bf16x8*>(gu + (size_t)row * 2 * I + lane * 8);
    uv = *reinterpret_cast<const bf16x8*>(gu + (size_t)row * 2 * I + I + lane * 8);
    dv = *reinterpret_cast<const bf16x8*>(dhp + (size_t)row * I + lane * 8);
  }
  const int slot = perm_slot[row];
  // expert of the row: offsets[e] <= row < offsets[e + 1], one offset per lane (E <= 64) and a ballot
  const int my_off = offsets[min(lane, E)];
  const int end = E < kWave ? __shfl(my_off, E, kWave) : offsets[E];
  if (row >= end) return;                                      // E = GLU experts: rows behind theirs have no activation
  const int e = __popcll(__ballot(lane < E && my_off <= row)) - 1;
  const float ws = w[slot];
  float g[8], u[8], d[8];
  float ss = 0.f;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    g[q] = (float)gv[q]; u[q] = (float)uv[q]; d[q] = (float)dv[q];
    ss = fmaf(g[q], g[q], ss);
  }
  ss = wave_sum(ss);
  const bool radial = act != BIBO_ACT_SILU;
  float p = 0.f, rinv = 1.f, gain = 1.f;
  if (radial) {
    p = radial_exponent(theta, e, act);
    radial_row_scalars(ss, I, p, act, rinv, gain);             // 1 / r and r^p
  }
  const float r = 1.f / rinv;
  float dot_h = 0.f, sum_qa = 0.f, inner = 0.f;
  float a_[8], ad_[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const float z = g[q] * rinv;
    const float s = 1.f / (1.f + __expf(-z));
    a_[q] = z * s;
    ad_[q] = s * (1.f + z * (1.f - s));
    dot_h = fmaf(d[q], gain * a_[q] * u[q], dot_h);
    const float qq = ws * d[q] * u[q];
    sum_qa = fmaf(qq, a_[q], sum_qa);
    inner = fmaf(qq, gain * rinv * (p * a_[q] - ad_[q] * z), inner);    // p r^(p-1) a - r^(p-2) a' g = r^(p-1) (p a - a' z)
  }
  dot_h = wave_sum(dot_h);
  sum_qa = wave_sum(sum_qa);
  inner = wave_sum(inner);
  if (live) {
    bf16x8 og, ou, oh;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float dh = ws * d[q];
      float dg = dh * u[q] * gain * rinv * ad_[q];
      if (radial) dg = fmaf(g[q] * rinv / (float)I, inner, dg);
      og[q] = (bf16_t)dg;
      ou[q] = (bf16_t)(dh * gain * a_[q]);
      oh[q] = (bf16_t)(ws * gain * a_[q] * u[q]);              // w h: the weight gradient's operand (moe.py:92-93)
    }
    *reinterpret_cast<bf16x8*>(dgu + (size_t)row * 2 * I + lane * 8) = og;
    *reinterpret_cast<bf16x8*>(dgu + (size_t)row * 2 * I + I + lane * 8) = ou;
    *reinterpret_cast<bf16x8*>(hidden + (size_t)row * I + lane * 8) = oh;
  }
  if (lane == 0) {
    dw_slot[slot] = dot_h;
    const float dp = act == BIBO_ACT_RADIAL_TANH ? 1.f - p * p : p * (1.f - p);
    dtheta_row[row] = radial ? dp * __logf(r) * gain * sum_qa : 0.f;
  }
}

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// dlogit of slot j of a token (router.py:31,41-47) from the scores s, weights w and weight gradients dw of its slots, the sums in ascending order
template <int K>
__device__ __forceinline__ float weight_to_score_grad(float dw, float w, float sum, float dot, int norm_mode) {
  if (K > 1 && norm_mode == BIBO_NORM_SUM) return (dw - dot) / (sum + 1e-20f);
  if (K > 1 && norm_mode == BIBO_NORM_SOFTMAX) return w * (dw - dot);
  return dw;
}
__device__ __forceinline__ float score_of(float logit) { return 1.f / (1.f + __expf(-logit)); }

// dW_router[e, c] = sum over the rows r of expert e of dl[slot(r)] x[token(r), c], in two steps.  Step 1: a block takes the z-th of
// kDwrSplit equal row ranges of row chunk g of the plan (kmajor.h: an expert's rows, cut where an expert holds many) and `width` columns
// (dwr_width); 32 threads share a row, 256 columns at a time, the eight partial sums meet in LDS in a fixed order -> part[g][z][c] fp32.
// Step 2 adds the ranges of an expert's chunks in order.  A row's token and dl go through LDS, 256 rows at a time: as loads of each of
// its threads they were three of four load instructions, 16 cycles of a CU's address unit each.
constexpr int kDwrSplit = 8, kDwrRows = 4, kDwrTurns = 4;
struct DwrShared {
  float red[8][256], d[256];
  int token[256];
};
template <typename SlotGrad>
__device__ __forceinline__ void dwr_block(DwrShared& sh, const bf16_t* __restrict__ x, SlotGrad slot_grad, const int* __restrict__ plan,
                                          const int32_t* __restrict__ perm_slot, const int32_t* __restrict__ perm_token, int H, int width,
                                          int block, float* __restrict__ part) {
  const int across = (H + width - 1) / width, range = block / across;
  const int g = range / kDwrSplit, z = range % kDwrSplit, c0 = (block - range * across) * width, c1 = min(c0 + width, H);
  if (g >= plan[0]) return;
  const int tid = threadIdx.x, cg = tid & 31, rl = tid >> 5;
  const int lo_e = plan[4 + 4 * g + 1], n = plan[4 + 4 * g + 2] - lo_e;
  const int per = (n + kDwrSplit - 1) / kDwrSplit;
  const int lo = lo_e + min(z * per, n), hi = lo_e + min((z + 1) * per, n);
  float acc[kDwrTurns][8];
#pragma unroll
  for (int i = 0; i < kDwrTurns; ++i)
#pragma unroll
    for (int q = 0; q < 8; ++q) acc[i][q] = 0.f;
  for (int r0 = lo; r0 < hi; r0 += 256) {
    const int rows = min(hi - r0, 256);
    __syncthreads();                                            // the rows before have been read
    if (tid < rows) {
      sh.token[tid] = perm_token[r0 + tid];
      sh.d[tid] = slot_grad(perm_slot[r0 + tid]);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kDwrTurns; ++i) {
      const int c = c0 + i * 256 + cg * 8;
      if (c >= c1) continue;
      const bf16_t* const xc = x + c;
      auto add = [&](float d, const bf16x8& v) {
#pragma unroll
        for (int q = 0; q < 8; ++q) acc[i][q] = fmaf(d, (float)v[q], acc[i][q]);
      };
      int r = rl;
      for (; r + 8 * (kDwrRows - 1) < rows; r += 8 * kDwrRows) {     // several rows on their way together
        bf16x8 v[kDwrRows];
#pragma unroll
        for (int u = 0; u < kDwrRows; ++u) v[u] = *reinterpret_cast<const bf16x8*>(xc + (size_t)sh.token[r + 8 * u] * H);
#pragma unroll
        for (int u = 0; u < kDwrRows; ++u) add(sh.d[r + 8 * u], v[u]);
      }
      for (; r < rows; r += 8) add(sh.d[r], *reinterpret_cast<const bf16x8*>(xc + (size_t)sh.token[r] * H));
    }
  }
#pragma unroll
  for (int i = 0; i < kDwrTurns; ++i) {
    if (c0 + i * 256 >= c1) break;
    __syncthreads();                                            // the sums before have been read
#pragma unroll
    for (int q = 0; q < 8; ++q) sh.red[rl][cg * 8 + q] = acc[i][q];
    __syncthreads();
    const int col = c0 + i * 256 + tid;
    if (col < c1)
      part[((size_t)g * kDwrSplit + z) * H + col] = ((sh.red[0][tid] + sh.red[1][tid]) + (sh.red[2][tid] + sh.red[3][tid])) +
                                                    ((sh.red[4][tid] + sh.red[5][tid]) + (sh.red[6][tid] + sh.red[7][tid]));
  }
}

// Columns of a block: all turns, fewer where less than two blocks a CU would come of it, which then read for longer than the rest of their
// launch takes.  All columns in a block -> this, backward pass, us: T = 16384, H = 4096, four experts: 953 -> 621; 8192, 2048, eight: 256 -> 213;
// 8192, 1536, four: 267 -> 205; 300, 1024, sixteen: 72 -> 69; with +/-Identity experts 8192, 2048, nine: 262 -> 226.  Half as many blocks at
// least, or twice as many: the same within 1 %.
constexpr int kDwrLeast = 512;
int dwr_blocks(int slots, int H, int width) { return slots * kDwrSplit * ((H + width - 1) / width); }
int dwr_width(int slots, int H) {
  int width = 256 * kDwrTurns;
  while (width > 256 && dwr_blocks(slots, H, width) < kDwrLeast) width /= 2;
  return width;
}

// where +/-Identity experts make a slot's gradient a dot product, which token_bwd_kernel works out
__global__ __launch_bounds__(256) void dwr_partial_kernel(const bf16_t* __restrict__ x, const float* __restrict__ dl, const int* __restrict__ plan,
                                                          const int32_t* __restrict__ perm_slot, const int32_t* __restrict__ perm_token,
                                                          int H, int width, float* __restrict__ part) {
  __shared__ DwrShared sh;
  dwr_block(sh, x, [&](int slot) { return dl[slot]; }, plan, perm_slot, perm_token, H, width, blockIdx.x, part);
}

// Everything per token behind the experts, one wave per token and run of up to 512 columns (`parts` runs of equal length):
//   +/-Identity slots (moe.py:95-99): dw = +/- <d_out[t], x[t]>, their share of dx is +/- w d_out[t];
//   router (router.py:31,41-47; w_router == NULL: none): lane j < k turns the gradients of the combine weights into dlogit of
//     slot j, the sums over a token's slots in ascending j;
//   dx[t, c] = sum_j (dx row of slot j + dl[t, j] W_router[idx[t, j], c]).
// A slot whose expert id lies outside [0, E + n_pos + n_neg) (padding in a caller's indices, which the forward pass skips) has no
// dx row and no combine-weight gradient: it is left out and its dw_slot entry set to zero.  Every wave of a token works out the k
// scalars, the first one stores them (without DWR).  Bound by reading the slots' dx rows (T = 8192, H = 768, k = 6: 75 MB), which are requested
// before the indices that decide about them are back.  K = k at compile time, and no load under a condition: the compiler
// drains all loads where a branch around one ends (k at run time: 26 us at that size, 21 like this).
// DWR: the first nb_dwr workgroups are dwr_partial_kernel's (the ranges of a chunk next to each other) and work out
// dl of their rows' slots themselves, so that they need not wait for this launch.  Both launches -> this one, us: 40.0 -> 31.4 (T = 8192, H = 768,
// k = 6), 20.4 -> 13.2 (6000, 512, 6), 29.3 -> 25.7 (4000, 1024, 8); with 256 columns a workgroup, each of which
// works dl out again, 35.3, 14.0 and 28.8; with dl from workgroups behind the GEMMs' 32.6, 15.0 and 26.9, and 1 to 7 more in the GEMMs.  (1111, 512, 2,
// sixteen experts: 8.7 -> 5.0 with 256 columns, which dwr_width takes there.)  Neither dl nor dw_slot is written then: every slot must be an
// expert's with weights (E is all there is, the indices the router's), whose dw_slot entry act_bwd_kernel has left.
template <int K, bool DWR>
__global__ __launch_bounds__(256) void token_bwd_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ d_out,
                                                        const bf16_t* __restrict__ dxs, const float* __restrict__ logits,
                                                        const int32_t* __restrict__ idx, const float* __restrict__ w,
                                                        const bf16_t* __restrict__ w_router, int T, int H, int E, int n_pos,
                                                        int n_neg, int norm_mode, int parts, float* __restrict__ dw_slot,
                                                        float* __restrict__ dl, bf16_t* __restrict__ dx, int nb_dwr, int dwr_cols,
                                                        const int* __restrict__ plan, const int32_t* __restrict__ perm_slot,
                                                        const int32_t* __restrict__ perm_token, float* __restrict__ dwr_part) {
  if constexpr (DWR) {
    __shared__ DwrShared sh;
    if (blockIdx.x < (unsigned)nb_dwr) {
      dwr_block(sh, x, [&](int slot) {
        const int t = slot / K, mine = slot - t * K;
        float s[K], dw[K], wj[K], sum = 0.f, dot = 0.f;
#pragma unroll
        for (int j = 0; j < K; ++j) {
          s[j] = logits[(size_t)t * E + min((unsigned)idx[t * K + j], (unsigned)E - 1u)];
          dw[j] = dw_slot[t * K + j];
          wj[j] = w[t * K + j];
        }
        float s_ = 0.f, dw_ = 0.f, w_ = 0.f;
#pragma unroll
        for (int j = 0; j < K; ++j) {
          s[j] = score_of(s[j]);
          sum += s[j];
          dot = fmaf(dw[j], wj[j], dot);
          if (j == mine) { s_ = s[j]; dw_ = dw[j]; w_ = wj[j]; }
        }
        return weight_to_score_grad<K>(dw_, w_, sum, dot, norm_mode) * s_ * (1.f - s_);
      }, plan, perm_slot, perm_token, H, dwr_cols, blockIdx.x, dwr_part);
      return;
    }
  }
  const int lane = threadIdx.x & 63;
  const int unit = __builtin_amdgcn_readfirstlane((blockIdx.x - (DWR ? nb_dwr : 0)) * 4 + (threadIdx.x >> 6));
  const int t = unit / parts, part = unit - t * parts;
  if (t >= T) return;
  const int Et = E + n_pos + n_neg, gran = H / 8, run = (gran + parts - 1) / parts;
  const int c = part * run + lane, cc = min(c, gran - 1);
  const bool mine = lane < run && c < gran;
  const bf16x8* const dtok = reinterpret_cast<const bf16x8*>(d_out) + (size_t)t * gran;
  // lane j < k: slot j.  Loads are waited for in the order of their requests: the indices first, then the rows, which do not need them.
  const int sl = t * K + min(lane, K - 1);
  int e_ = idx[sl];
  const float w_ = w[sl];
  float dw_ = dw_slot[sl], s_ = 0.f;
  bf16x8 v[K], r[K];
  const bf16x8* const rows = reinterpret_cast<const bf16x8*>(dxs) + (size_t)t * K * gran + cc;
#pragma unroll
  for (int j = 0; j < K; ++j) v[j] = rows[(size_t)j * gran];
  __builtin_amdgcn_sched_barrier(0);
  if (e_ >= Et) e_ = -1;
  if (e_ < 0 || e_ >= E) dw_ = 0.f;
  if (w_router != nullptr) {
    const float logit = logits[(size_t)t * Et + max(e_, 0)];
#pragma unroll
    for (int j = 0; j < K; ++j)
      r[j] = reinterpret_cast<const bf16x8*>(w_router)[(size_t)max(__builtin_amdgcn_readlane(e_, j), 0) * gran + cc];
    s_ = score_of(logit);
  }
  if (__ballot(e_ >= E) != 0ull) {
    float dot = 0.f;
    for (int g = lane; g < gran; g += kWave) {
      const bf16x8 xv = reinterpret_cast<const bf16x8*>(x)[(size_t)t * gran + g];
      const bf16x8 dv = dtok[g];
#pragma unroll
      for (int q = 0; q < 8; ++q) dot = fmaf((float)dv[q], (float)xv[q], dot);
    }
    dot = wave_sum(dot);
    if (e_ >= E) dw_ = e_ < E + n_pos ? dot : -dot;
  }
  float dl_ = 0.f;
  if (w_router != nullptr) {
    float sum = 0.f, dot = 0.f;
#pragma unroll
    for (int j = 0; j < K; ++j) {
      sum += lane_value(s_, j);
      dot = fmaf(lane_value(dw_, j), lane_value(w_, j), dot);
    }
    dl_ = weight_to_score_grad<K>(dw_, w_, sum, dot, norm_mode) * s_ * (1.f - s_);
  }
  if (!DWR && part == 0 && lane < K) {
    if (e_ < 0 || e_ >= E) dw_slot[t * K + lane] = dw_;
    if (w_router != nullptr) dl[t * K + lane] = dl_;
  }
  if (!mine) return;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < K; ++j) {
    const int e = __builtin_amdgcn_readlane(e_, j);
    if (e < 0) continue;
    if (e >= E) {
      const float wj = lane_value(w_, j);
      const bf16x8 dv = dtok[c];
#pragma unroll
      for (int q = 0; q < 8; ++q) acc[q] = fmaf(e < E + n_pos ? wj : -wj, (float)dv[q], acc[q]);
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) acc[q] += (float)v[j][q];
    }
    if (w_router != nullptr) {
      const float dj = lane_value(dl_, j);
#pragma unroll
      for (int q = 0; q < 8; ++q) acc[q] = fmaf(dj, (float)r[j][q], acc[q]);
    }
  }
  bf16x8 o;
#pragma unroll
  for (int q = 0; q < 8; ++q) o[q] = (bf16_t)acc[q];
  reinterpret_cast<bf16x8*>(dx)[(size_t)t * gran + c] = o;
}

// The last launch of the backward pass: every sum that ends one, by ranges of workgroups.
//   [0, nb_w): the partial tiles of the experts that were cut into chunks (kmajor.h) -> dW_down, dW_gate_up;
//   [nb_w, nb_w + E): dtheta[e] = the sum of the theta shares of expert e's rows, chunk by chunk of the plan and the
//     chunks in order (no atomics: the same bits on every call);
//   from nb_w + E on (when dwr != nullptr): the router's weight gradient [Et, H] = the sum over an expert's chunks
//     of dwr_partial_kernel's partial rows.
__global__ __launch_bounds__(256) void backward_sums_kernel(int nb_w, const float* __restrict__ part_a,
                                                            const float* __restrict__ part_b, const int* __restrict__ plan,
                                                            int slots, int NMa, int NMb, int E, int Et,
                                                            void* __restrict__ dWa, void* __restrict__ dWb, int f32,
                                                            const float* __restrict__ dtheta_row, float* __restrict__ dtheta,
                                                            const float* __restrict__ dwr_part, int H,
                                                            void* __restrict__ dwr) {
  const int block = blockIdx.x;
  if (block < nb_w) {
    wgrad_reduce_block(block, part_a, part_b, plan, slots, NMa, NMb, E, dWa, dWb, f32);
    return;
  }
  const int* experts = plan + 4 + 4 * (slots + Et);            // {first chunk, chunks, ., .} per expert
  if (block < nb_w + E) {
    __shared__ float red[4];
    const int e = block - nb_w;
    const int first = experts[4 * e], chunks = experts[4 * e + 1];
    float total = 0.f;
    for (int c = 0; c < chunks; ++c) {
      const int* entry = plan + 4 + 4 * (first + c);
      float acc = 0.f;
      for (int r = entry[1] + threadIdx.x; r < entry[2]; r += 256) acc += dtheta_row[r];
      acc = wave_sum(acc);
      __syncthreads();
      if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
      __syncthreads();
      total += (red[0] + red[1]) + (red[2] + red[3]);
    }
    if (threadIdx.x == 0) dtheta[e] = total;
    return;
  }
  if (dwr == nullptr) return;
  const int i = (block - nb_w - E) * 256 + threadIdx.x;         // element of [Et, H]
  if (i >= Et * H) return;
  const int e = i / H, c = i - e * H;
  const int first = experts[4 * e], chunks = experts[4 * e + 1];
  float acc = 0.f;
  for (int j = 0; j < chunks * kDwrSplit; ++j) acc += dwr_part[((size_t)first * kDwrSplit + j) * H + c];
  if (f32) static_cast<float*>(dwr)[i] = acc;
  else static_cast<bf16_t*>(dwr)[i] = (bf16_t)acc;
}

// zero n 4-byte words (a kernel rather than a memset node, so that the call can be captured into a graph)
__global__ void zero_words_kernel(uint32_t* __restrict__ p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0u;
}

void zero_bytes(void* p, size_t bytes, hipStream_t s) {          // bytes is a multiple of 4
  const size_t n = bytes / 4;
  if (n == 0) return;
  const unsigned grid = (unsigned)((n + 255) / 256 < 2048 ? (n + 255) / 256 : 2048);
  hipLaunchKernelGGL(zero_words_kernel, dim3(grid), dim3(256), 0, s, static_cast<uint32_t*>(p), n);
}

}  // namespace

bool backward_supported(int H, int I, int k, int dtype) {
  return dtype == BIBO_DTYPE_BF16 && H >= 128 && H % 128 == 0 && I >= 128 && I % 128 == 0 && I <= kActMaxI &&
         k <= kMaxK;
}

int backward_dwr_split() { return kDwrSplit; }

// a row of zeros as wide as the widest weight-gradient operand: what a K stage reads past an expert's last row
// The sums over an expert's rows (weight-gradient GEMMs, router weight gradient, theta gradient) cut an expert with more
// rows than this into chunks (kmajor.h): one and a half times the average over all E routed experts, so that evenly
// routed tokens leave every expert in one piece, and at least 512.
int backward_chunk_rows(int S_rows, int E) {
  const long long c = (3ll * S_rows / (2ll * E) + 31) & ~31ll;
  return (int)(c < 512 ? 512 : c);
}
// chunks over all experts, at most
int backward_chunk_slots(int S_rows, int E) { return S_rows / backward_chunk_rows(S_rows, E) + E; }
// fp32 partial tiles of the cut experts, dW_down's and dW_gate_up's, one slot per chunk each
size_t backward_wgrad_part_bytes(int S_rows, int H, int E, int I) {
  return (size_t)backward_chunk_slots(S_rows, E) * 3 * I * H * sizeof(float);
}
// the list of chunks (kmajor.h: WgradPlan): a header, a 16-byte entry per chunk and two per expert
size_t backward_plan_bytes(int S_rows, int E) { return 16 + (size_t)(backward_chunk_slots(S_rows, E) + 2 * E) * 16; }

size_t backward_zero_row_bytes(int H, int I) { return (size_t)(H > 2 * I ? H : 2 * I) * sizeof(bf16_t); }

// The launches after routing and permutation.  Buffers (bf16 unless noted): gu [S,2I], dhp [S,I], dgu [S,2I],
// hidden [S,I], dxs [S,H], zrow [max(H, 2I)] (cleared by act_bwd_kernel), dw_slot [S] f32, dl [S] f32, dtheta_row [S] f32,
// dwr_part [backward_chunk_slots(), backward_dwr_split(), H] f32.
hipError_t launch_backward(const void* x, const void* d_out, const void* w_router, const void* wgu, const void* wd,
                           const float* theta, const float* logits, const int32_t* idx, const float* w,
                           const int32_t* offsets, const int32_t* perm_slot, const int32_t* perm_token, int T, int H, int E,
                           int n_pos, int n_neg, int k, int I, int norm_mode, int act, const BackwardBuffers& b, void* dx,
                           void* d_w_router, void* d_wgu, void* d_wd, float* d_theta, int grad_f32,
                           hipStream_t s, const void* gu_saved) {
  const size_t gb = grad_f32 ? sizeof(float) : sizeof(bf16_t);      // bytes per element of the weight gradients
  // E = GLU experts (with weights); the router and the permutation know Et experts, the +/-Identity ones last
  const int Et = E + n_pos + n_neg;
  const int S = T * k;
  const int slots = backward_chunk_slots(S, Et);      // row chunks of the plan, at most
  const bf16_t* xp = static_cast<const bf16_t*>(x);
  const bf16_t* dop = static_cast<const bf16_t*>(d_out);
  const bf16_t* wrp = static_cast<const bf16_t*>(w_router);
  const bf16_t* wgup = static_cast<const bf16_t*>(wgu);
  const bf16_t* wdp = static_cast<const bf16_t*>(wd);
  // the pre-activations: a training forward's, or recomputed below into the workspace
  const bf16_t* gu = gu_saved != nullptr ? static_cast<const bf16_t*>(gu_saved) : static_cast<const bf16_t*>(b.gu);
  bf16_t* dhp = static_cast<bf16_t*>(b.dhp);
  bf16_t* dgu = static_cast<bf16_t*>(b.dgu);
  bf16_t* hidden = static_cast<bf16_t*>(b.hidden);
  bf16_t* dxs = static_cast<bf16_t*>(b.dxs);
  bf16_t* zrow = static_cast<bf16_t*>(b.zrow);
  hipError_t err = hipSuccess;
  if (S == 0) {
    zero_bytes(d_theta, (size_t)E * sizeof(float), s);
    if (d_w_router != nullptr) zero_bytes(d_w_router, (size_t)Et * H * gb, s);
    zero_bytes(d_wgu, (size_t)E * 2 * I * H * gb, s);
    zero_bytes(d_wd, (size_t)E * H * I * gb, s);
    return hipGetLastError();
  }
  // pre-activations again (moe.py:84): x W_gate_up^T, both contiguous along H - by the first phase of the forward
  // pass's fused kernel where it takes the shape (its ring of weight stages is the faster main loop)
  if (gu_saved != nullptr)
    err = hipSuccess;
  else if ((fused_supported(H, I, BIBO_DTYPE_BF16) || fused_wide_supported(H, I, BIBO_DTYPE_BF16)) && (long long)T * H < (1LL << 31))
    err = launch_gateup_raw(xp, wgup, offsets, perm_token, T, H, E, k, I, b.gu, split_columns(S, E, H, I), false, s);
  else
    err = launch_ggemm<true, false>(xp, perm_token, wgup, offsets, nullptr, S, H, 2 * I, E, static_cast<bf16_t*>(b.gu), s);
  if (err != hipSuccess) return err;
  // dh' = d W_down: contracts over H, the middle dimension of w_down [E, H, I]
  err = launch_dgrad<true, false>(dop, perm_token, wdp, offsets, nullptr, S, H, I, E, dhp, s);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(act_bwd_kernel, dim3((S + 3) / 4), dim3(256), 0, s, gu, dhp, w, theta, offsets, perm_slot, S, E, I, act,
                     dgu, hidden, b.dw_slot, b.dtheta_row, reinterpret_cast<uint32_t*>(zrow),
                     (int)(backward_zero_row_bytes(H, I) / 4), b.wgrad_plan, Et, backward_chunk_rows(S, Et), slots);
  // dx of every slot, in slot order: [dg, du] W_gate_up, contracts over the 2I rows of w_gate_up [E, 2I, H].  Weight gradients,
  // contracted over each expert's rows: dW_down[e] = d^T (w h) (d gathered by token, `hidden` already carries w), dW_gate_up[e] =
  // [dg, du]^T x (x gathered by token)
  float* part_gu = b.wgrad_part + (size_t)slots * H * I;
  BackwardGemms gemms{xp, dop, dgu, hidden, wgup, zrow, offsets, perm_slot, perm_token, b.wgrad_plan, dxs, d_wgu, d_wd, part_gu,
                      b.wgrad_part, H, I, E, grad_f32, 0, 0, false};
  if ((err = launch_backward_gemms(gemms, T, S, backward_chunk_rows(S, Et), slots, s)) != hipSuccess) return err;
  const bool with_router = w_router != nullptr;      // else: the experts alone, the caller owns the routing
  const bool merged = with_router && E == Et;        // the router's partial sums beside the tokens: their slots are the experts'
  const int parts = (H / 8 + kWave - 1) / kWave;     // runs of columns a lane each
  const int dwr_cols = dwr_width(slots, H), nb_dwr = dwr_blocks(slots, H, dwr_cols);
  auto token_bwd = [&](auto kc, auto with_dwr) {
    constexpr bool DWR = decltype(with_dwr)::value;
    hipLaunchKernelGGL((token_bwd_kernel<decltype(kc)::value, DWR>), dim3((unsigned)(((long long)T * parts + 3) / 4) + (DWR ? nb_dwr : 0)), dim3(256),
                       0, s, xp, dop, dxs, logits, idx, w, wrp, T, H, E, n_pos, n_neg, norm_mode, parts, b.dw_slot, b.dl,
                       static_cast<bf16_t*>(dx), nb_dwr, dwr_cols, b.wgrad_plan, perm_slot, perm_token, b.dwr_part);
  };
  auto token_launch = [&](auto kc) {
    if (merged) token_bwd(kc, std::true_type());
    else token_bwd(kc, std::false_type());
  };
  static_assert(kMaxK == 8, "a case per k");
  using std::integral_constant;
  switch (k) {
    case 1: token_launch(integral_constant<int, 1>{}); break;
    case 2: token_launch(integral_constant<int, 2>{}); break;
    case 3: token_launch(integral_constant<int, 3>{}); break;
    case 4: token_launch(integral_constant<int, 4>{}); break;
    case 5: token_launch(integral_constant<int, 5>{}); break;
    case 6: token_launch(integral_constant<int, 6>{}); break;
    case 7: token_launch(integral_constant<int, 7>{}); break;
    default: token_launch(integral_constant<int, 8>{});
  }
  if (with_router && !merged)
    hipLaunchKernelGGL(dwr_partial_kernel, dim3(nb_dwr), dim3(256), 0, s, xp, b.dl, b.wgrad_plan, perm_slot, perm_token, H, dwr_cols, b.dwr_part);
  // the sums that end the pass: cut experts' partial tiles, dtheta, the router's weight gradient
  const int nb_w = (int)(((size_t)2 * I * H / 4 + 255) / 256);
  const int nb_r = with_router ? (Et * H + 255) / 256 : 0;
  hipLaunchKernelGGL(backward_sums_kernel, dim3(nb_w + E + nb_r), dim3(256), 0, s, nb_w, b.wgrad_part, part_gu, b.wgrad_plan,
                     slots, H * I, 2 * I * H, E, Et, d_wd, d_wgu, grad_f32, b.dtheta_row,
                     d_theta, b.dwr_part, H, with_router ? d_w_router : nullptr);
  return hipGetLastError();
}

}  // namespace bibo
