// Kernel 1: fused router.  fp32 logits x @ w_router^T, canonical sigmoid, selection on score + bias
// (ties to the lowest expert index), gather of the unbiased scores, normalisation.
// Follows BiBoMoERouter.forward, src/modeling/ffn/router.py:25-51 of the reference.
#include "few.h"

namespace bibo {
namespace {

constexpr int kRowPad = kMaxE + 1;   // LDS row stride (floats): lane = token reads are conflict-free

// Integer key of a score whose unsigned order is the order of the floats (-0 counts as +0): the row-wide maximum
// is then one v_max_u32 per butterfly step instead of a compare-and-select on (value, expert) pairs under exec
// masks, which cost this selection 3.5 us per workgroup.
__device__ __forceinline__ unsigned order_key(float v) {
  const unsigned u = __float_as_uint(v + 0.f);
  return u ^ ((unsigned)((int)u >> 31) | 0x80000000u);
}
__device__ __forceinline__ float key_value(unsigned key) {
  return __uint_as_float((key & 0x80000000u) ? key ^ 0x80000000u : ~key);
}

template <int kCtrl>
__device__ __forceinline__ unsigned dpp_u32(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, 0xf, 0xf, false);
}
// 16-lane butterfly on DPP row operations (a DPP row is exactly one token's 16 lanes): swap within pairs, swap
// pairs within quads, mirror within 8 lanes, mirror within 16 lanes.  Every lane ends with the row's result.
__device__ __forceinline__ unsigned row_max_u32(unsigned v) {
  v = max(v, dpp_u32<0xB1>(v));
  v = max(v, dpp_u32<0x4E>(v));
  v = max(v, dpp_u32<0x141>(v));
  return max(v, dpp_u32<0x140>(v));
}
__device__ __forceinline__ unsigned row_min_u32(unsigned v) {
  v = min(v, dpp_u32<0xB1>(v));
  v = min(v, dpp_u32<0x4E>(v));
  v = min(v, dpp_u32<0x141>(v));
  return min(v, dpp_u32<0x140>(v));
}

// Cooperative selection: 16 lanes per token, lane `seg` owns experts 4*seg .. 4*seg+3.  k rounds of
// "best remaining candidate": the row's largest key, then the lowest expert index among the lanes that hold it,
// which is the tie rule (equal floats have equal keys).  All 16 lanes end every round with the same winner.
// Returns the bit mask of the chosen experts.
__device__ __forceinline__ unsigned long long select_mask16(const float (&v)[4], int seg, int rounds, float* kth,
                                                            float* kth1) {
  unsigned key[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) key[q] = order_key(v[q]);
  unsigned taken = 0;
  unsigned long long mask = 0;
  for (int r = 0; r < rounds; ++r) {
    unsigned bk = 0, be = kMaxE;                     // a taken expert counts as key 0, below every score's key
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const unsigned kq = ((taken >> q) & 1) ? 0u : key[q];
      if (kq > bk) { bk = kq; be = seg * 4 + q; }    // strict: the lower expert of the lane keeps an equal key
    }
    const unsigned mk = row_max_u32(bk);
    be = row_min_u32(bk == mk ? be : (unsigned)kMaxE);
    be &= kMaxE - 1;
    if ((int)(be >> 2) == seg) taken |= 1u << (be & 3);
    mask |= 1ull << be;
    if (kth != nullptr) { if (r == rounds - 2) *kth = key_value(mk); if (r == rounds - 1) *kth1 = key_value(mk); }
  }
  return mask;
}

// Selection for the tokens of one workgroup whose scores sit in LDS rows `sc` (stride kRowPad):
// thread = (token tid>>4, segment tid&15); needs blockDim.x >= 16 * ntok_max.  Lane j < k of a token's 16 then
// owns output j (the j-th chosen expert in ascending order): it gathers the unbiased score, the row adds the scores
// up one after the other in that order (a serial scan over lanes, so the sum has the bits of the sequential loop),
// and every lane normalises and stores its own weight.
// Returns the bit mask of the experts chosen for this thread's token (0 for a token past the end).
__device__ __forceinline__ unsigned long long select_tokens16(const float* __restrict__ sc,
                                                              const float* __restrict__ bias_s, int E, int k,
                                                              int norm_mode, int t0, int ntok, int32_t* __restrict__ idx,
                                                              float* __restrict__ w, float* __restrict__ gap) {
  const int tid = threadIdx.x;
  const int tl = tid >> 4, seg = tid & 15;
  const bool live = tl < ntok;                       // whole 16-lane groups are live or not
  const float* row = sc + (live ? tl : 0) * kRowPad;
  float v[4], u[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int e = seg * 4 + q;
    u[q] = (e < E) ? row[e] : -INFINITY;
    v[q] = (e < E) ? row[e] + bias_s[e] : -INFINITY;                      // router.py:38
  }
  const unsigned long long mask = select_mask16(v, seg, k, nullptr, nullptr);
  float g_hi = 0.f, g_lo = 0.f;
  if (gap != nullptr && k < E) select_mask16(u, seg, k + 1, &g_hi, &g_lo);   // router.py:33-36, unbiased scores
  const bool mine = seg < k;                                              // this lane owns output `seg`
  unsigned long long m = mask;
#pragma unroll
  for (int j = 0; j < kMaxK - 1; ++j)
    if (j < seg) m &= m - 1;                                              // drop the `seg` lowest chosen experts
  const int e = mine ? __ffsll((long long)m) - 1 : 0;                     // ascending expert order
  const float raw = mine ? row[e] : 0.f;                                  // UNBIASED score, router.py:41
  // running sum in ascending j, one lane after the other: lane j ends with ((raw_0 + raw_1) + ...) + raw_j
  auto scan = [&](float x) {
    float s = x;
#pragma unroll
    for (int j = 1; j < kMaxK; ++j) {
      const float prev = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s), 0x111, 0xf, 0xf, false));
      if (seg == j && j < k) s = prev + x;                                // row_shr:1, lane j reads lane j-1
    }
    return __shfl(s, (tid & 48) + k - 1, kWave);                          // the whole sum, from lane k-1 of the row
  };
  float wv = raw;                                                         // router.py:46-47
  if (k > 1 && norm_mode == BIBO_NORM_SOFTMAX) {                          // router.py:42-43
    const float mx = key_value(row_max_u32(mine ? order_key(raw) : 0u));
    const float ex = mine ? expf(raw - mx) : 0.f;
    wv = ex / scan(ex);
  } else if (k > 1 && norm_mode == BIBO_NORM_SUM) {                       // router.py:44-45
    wv = raw / (scan(raw) + kSumNormEps);
  }
  if (live && mine) {
    const size_t o = (size_t)(t0 + tl) * k + seg;
    idx[o] = e;
    w[o] = wv;
  }
  if (live && seg == 0 && gap != nullptr) gap[t0 + tl] = (k < E) ? (g_hi - g_lo) : 0.f;
  return live ? mask : 0ull;
}

// Histogram of the selections of this workgroup's TOK tokens (16 threads each), for the permutation kernel.
template <int TOK>
__device__ __forceinline__ void write_chunk_hist(unsigned long long mask, int32_t* __restrict__ chunk_hist, unsigned long long* mask_s) {
  const int tid = threadIdx.x;
  if ((tid & 15) == 0) mask_s[tid >> 4] = mask;
  __syncthreads();
  if (tid < kMaxE) {
    int c = 0;
#pragma unroll
    for (int t = 0; t < TOK; ++t) c += (int)((mask_s[t] >> tid) & 1ull);
    chunk_hist[blockIdx.x * kMaxE + tid] = c;
  }
}

// ---- MFMA router: bf16, H % 128 == 0 ------------------------------------------------------------
// One workgroup = TOK tokens (16 or 32), TOK/16 x 4 waves: wave (tm, en) owns the 16x16 logits tile of
// token tile tm and expert tile en over the whole K, so no partial sums cross waves and the fp32
// accumulation order is fixed.  x rows and w_router rows travel global -> LDS by LDS-DMA in K chunks of
// 128 elements (256-byte rows, one instruction fetches four whole rows per wave), double-buffered:
// fetching w_router straight into registers costs a CU about 37 GB/s, the DMA path twice that, and
// every workgroup needs all of w_router.  Granule c of row r sits at position c ^ (r & 15).
constexpr int kRouterKC = 128;                       // K elements per chunk
constexpr int kRouterGran = kRouterKC / 8;           // 16-byte granules per chunk row

typedef __attribute__((address_space(3))) void router_lds_void;
typedef const __attribute__((address_space(1))) void router_gbl_void;

// Everything after the logits of a TOK-token workgroup: canonical sigmoid on the accumulator registers, selection,
// weights, and the workgroup's histogram of selected experts.  Wave (tm, en) holds the 16x16 logits tile of token
// tile tm and expert tile en: lane = column (expert) lane%16, rows (tokens) 4*(lane/16)+i.
template <int TOK>
__device__ __forceinline__ void router_finish(const floatx4& acc, float* sc, const float* bias_s, int T, int E, int k,
                                              int norm_mode, int t0, float* __restrict__ logits, int32_t* __restrict__ idx,
                                              float* __restrict__ w, float* __restrict__ gap,
                                              int32_t* __restrict__ chunk_hist, unsigned long long* mask_s) {
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int tm = wave >> 2, en = wave & 3;
  const int r16 = lane & 15, kc = lane >> 4;
  const int ntok = min(TOK, T - t0);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int tl = tm * 16 + kc * 4 + i, e = en * 16 + r16;
    if (tl < ntok && e < E) {
      const float lg = acc[i];
      if (logits != nullptr) logits[(size_t)(t0 + tl) * E + e] = lg;
      sc[tl * kRowPad + e] = sigmoid32_canonical(lg);          // router.py:31
    }
  }
  __syncthreads();
  const unsigned long long mask = select_tokens16(sc, bias_s, E, k, norm_mode, t0, ntok, idx, w, gap);
  if (chunk_hist != nullptr) write_chunk_hist<TOK>(mask, chunk_hist, mask_s);
}

// ---- generic router: any H, bf16 or fp32 inputs, fp32 arithmetic ---------------------------------
// One workgroup = 16 tokens x 64 experts, wave en = expert tile en.  K chunks of 64 elements, widened to fp32, pass through
// LDS; the next three are on their way to registers meanwhile (with a few tokens the kernel is one workgroup and its loads'
// latency).  v_mfma_f32_16x16x4_f32 with k ascending: one logit is one chain of FMAs over ascending h, bit for bit (checked
// against scalar FMAs, which took 16 us for H = 768 at one wave per SIMD where the MFMA chain takes 2.6).
// VEC: rows are 16-byte (bf16: 8-byte) aligned and H % 4 == 0.
constexpr int kGenTokens = 16;
constexpr int kGenKC = 64;
constexpr int kGenAhead = 3;

template <typename TIn, bool VEC>
__global__ __launch_bounds__(256) void router_f32_kernel(const TIn* __restrict__ x, const TIn* __restrict__ wr,
                                                         const float* __restrict__ bias, int T, int H, int E, int k,
                                                         int norm_mode, float* __restrict__ logits, int32_t* __restrict__ idx,
                                                         float* __restrict__ w, float* __restrict__ gap,
                                                         int32_t* __restrict__ chunk_hist) {
  constexpr int kStride = kGenKC + 4;                          // floats: 16 rows of a 16-byte read hit distinct banks
  __shared__ __attribute__((aligned(16))) float xs[kGenTokens * kStride];
  __shared__ __attribute__((aligned(16))) float ws[kMaxE * kStride];
  __shared__ float sc[kGenTokens * kRowPad];
  __shared__ float bias_s[kMaxE];
  const int tid = threadIdx.x;
  const int t0 = blockIdx.x * kGenTokens;
  if (tid < kMaxE) bias_s[tid] = (tid < E) ? bias[tid] : 0.f;
  // fill side: thread = granule tid % 16 (four elements) of rows tid / 16 + 16 i; row group 0 = the tokens, 1 .. 4 = w_router
  const int fr = tid >> 4, fc = (tid & 15) * 4;
  const TIn* src[5];
  bool live[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const int e = fr + 16 * (i - 1);
    live[i] = i == 0 || e < E;
    src[i] = i == 0 ? x + (size_t)min(t0 + fr, T - 1) * H : wr + (size_t)min(e, E - 1) * H;
  }
  floatx4 r[kGenAhead][5];
  auto load = [&](auto set, int h0) {
    constexpr int st = decltype(set)::value;
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      r[st][i] = floatx4{0.f, 0.f, 0.f, 0.f};
      if constexpr (VEC) {
        if (live[i] && h0 + fc < H) r[st][i] = load4<TIn>(src[i] + h0 + fc);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (live[i] && h0 + fc + q < H) r[st][i][q] = to_float(src[i][h0 + fc + q]);
      }
    }
  };
  const int lane = tid & 63, r16 = lane & 15, g4 = lane >> 4;
  const float* xrow = xs + r16 * kStride + g4;                 // A: token r16, k = 4 m + g4
  const float* wrow = ws + ((tid >> 6) * 16 + r16) * kStride + g4;
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  auto chunk = [&](auto set, int h0) {
    constexpr int st = decltype(set)::value;
    *reinterpret_cast<floatx4*>(xs + fr * kStride + fc) = r[st][0];
#pragma unroll
    for (int i = 1; i < 5; ++i) *reinterpret_cast<floatx4*>(ws + (fr + 16 * (i - 1)) * kStride + fc) = r[st][i];
    __syncthreads();
    if (h0 + kGenAhead * kGenKC < H) load(set, h0 + kGenAhead * kGenKC);
#pragma unroll
    for (int m = 0; m < kGenKC; m += 4) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xrow[m], wrow[m], acc, 0, 0, 0);
    __syncthreads();
  };
  using std::integral_constant;
  load(integral_constant<int, 0>{}, 0);
  load(integral_constant<int, 1>{}, kGenKC);
  load(integral_constant<int, 2>{}, 2 * kGenKC);
  for (int h0 = 0; h0 < H; h0 += kGenAhead * kGenKC) {
    chunk(integral_constant<int, 0>{}, h0);
    if (h0 + kGenKC < H) chunk(integral_constant<int, 1>{}, h0 + kGenKC);
    if (h0 + 2 * kGenKC < H) chunk(integral_constant<int, 2>{}, h0 + 2 * kGenKC);
  }
  __shared__ unsigned long long mask_s[kGenTokens];
  router_finish<kGenTokens>(acc, sc, bias_s, T, E, k, norm_mode, t0, logits, idx, w, gap, chunk_hist, mask_s);
}

template <int TOK>
__global__ __launch_bounds__(TOK * 16) void router_mfma_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ wr,
                                                               const float* __restrict__ bias, int T, int H, int E,
                                                               int k, int norm_mode, float* __restrict__ logits,
                                                               int32_t* __restrict__ idx, float* __restrict__ w,
                                                               float* __restrict__ gap,
                                                               int32_t* __restrict__ chunk_hist) {
  constexpr int kThreads = TOK * 16;
  constexpr int kRows = TOK + kMaxE;                 // stage rows: tokens first, then experts
  constexpr int kPer = kRows * kRouterGran / kThreads;   // load instructions per thread and chunk
  static_assert(kRows * kRouterGran % kThreads == 0, "stage does not divide over the threads");
  __shared__ __attribute__((aligned(16))) bf16_t st0[kRows * kRouterKC];
  __shared__ __attribute__((aligned(16))) bf16_t st1[kRows * kRouterKC];
  __shared__ float sc[TOK * kRowPad];
  __shared__ float bias_s[kMaxE];
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int t0 = blockIdx.x * TOK;
  if (tid < kMaxE) bias_s[tid] = (tid < E) ? bias[tid] : 0.f;

  // thread t of load instruction i fills granule i*kThreads + t = (row, position t % 16) and fetches logical
  // granule (t % 16) ^ (row % 16) of that row
  const bf16_t* src[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int row = (i * kThreads + tid) / kRouterGran;
    const int c = (tid & (kRouterGran - 1)) ^ (row & 15);
    src[i] = (row < TOK ? x + (size_t)min(t0 + row, T - 1) * H : wr + (size_t)min(row - TOK, E - 1) * H) + c * 8;
  }
  auto issue = [&](int k0, bf16_t* st) {
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      __builtin_amdgcn_global_load_lds((router_gbl_void*)(src[i] + k0), (router_lds_void*)(st + (i * kThreads + wave * 64) * 8),
                                       16, 0, 0);
  };
  const int tm = wave >> 2, en = wave & 3;
  const int r16 = lane & 15, kc = lane >> 4;         // fragment row, 8-wide k chunk of a 32-wide step
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const bf16_t* st) {
    const bf16_t* arow = st + (tm * 16 + r16) * kRouterKC;
    const bf16_t* brow = st + (TOK + en * 16 + r16) * kRouterKC;
#pragma unroll
    for (int s = 0; s < kRouterKC / 32; ++s) {
      const int pos = ((s * 4 + kc) ^ r16) * 8;      // both rows are r16 mod 16
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(arow + pos);
      const bf16x8 b = *reinterpret_cast<const bf16x8*>(brow + pos);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
    }
  };
  issue(0, st0);
  for (int k0 = 0; k0 < H; k0 += 2 * kRouterKC) {
    __builtin_amdgcn_s_waitcnt(0);                   // vmcnt(0): this thread's transfers have landed
    __syncthreads();
    if (k0 + kRouterKC < H) issue(k0 + kRouterKC, st1);
    multiply(st0);
    if (k0 + kRouterKC < H) {
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      if (k0 + 2 * kRouterKC < H) issue(k0 + 2 * kRouterKC, st0);
      multiply(st1);
    }
  }
  __shared__ unsigned long long mask_s[TOK];
  router_finish<TOK>(acc, sc, bias_s, T, E, k, norm_mode, t0, logits, idx, w, gap, chunk_hist, mask_s);
}

// The same for calls of at most one workgroup per CU, which are a chain of memory latencies, one a chunk with two stages: here the first
// six chunks of the rows and of w_router are requested up front (further ones as stages fall free), so that a workgroup waits for
// one round trip and then for its bytes.  120 KB of LDS: one workgroup a CU.
constexpr int kRouterRing = 6, kRingLeast = 128;
__global__ __launch_bounds__(256) void router_ring_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ wr,
                                                          const float* __restrict__ bias, int T, int H, int E, int k, int norm_mode,
                                                          float* __restrict__ logits, int32_t* __restrict__ idx,
                                                          float* __restrict__ w, float* __restrict__ gap,
                                                          int32_t* __restrict__ chunk_hist) {
  constexpr int TOK = 16, kThreads = TOK * 16, kRows = TOK + kMaxE, kPer = kRows * kRouterGran / kThreads;
  constexpr int kElems = kRows * kRouterKC;
  __shared__ __attribute__((aligned(16))) bf16_t st0[kElems];
  __shared__ __attribute__((aligned(16))) bf16_t st1[kElems];
  __shared__ __attribute__((aligned(16))) bf16_t st2[kElems];
  __shared__ __attribute__((aligned(16))) bf16_t st3[kElems];
  __shared__ __attribute__((aligned(16))) bf16_t st4[kElems];
  __shared__ __attribute__((aligned(16))) bf16_t st5[kElems];
  __shared__ float sc[TOK * kRowPad];
  __shared__ float bias_s[kMaxE];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int t0 = blockIdx.x * TOK;
  const float my_bias = tid < E ? bias[tid] : 0.f;
  const bf16_t* src[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int row = (i * kThreads + tid) / kRouterGran;
    const int c = (tid & (kRouterGran - 1)) ^ (row & 15);
    src[i] = (row < TOK ? x + (size_t)min(t0 + row, T - 1) * H : wr + (size_t)min(row - TOK, E - 1) * H) + c * 8;
  }
  auto stage = [&](auto ic) -> bf16_t* {
    constexpr int i = decltype(ic)::value;
    if constexpr (i == 0) return st0; else if constexpr (i == 1) return st1; else if constexpr (i == 2) return st2;
    else if constexpr (i == 3) return st3; else if constexpr (i == 4) return st4; else return st5;
  };
  auto issue = [&](int chunk, bf16_t* st) {
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      __builtin_amdgcn_global_load_lds((router_gbl_void*)(src[i] + chunk * kRouterKC), (router_lds_void*)(st + (i * kThreads + wave * 64) * 8),
                                       16, 0, 0);
  };
  const int r16 = lane & 15, kc = lane >> 4;
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  const int nchunks = H / kRouterKC;
  using std::integral_constant;
  for_each<kRouterRing>([&](auto ic) { if (decltype(ic)::value < nchunks) issue(decltype(ic)::value, stage(ic)); });
  for (int c0 = 0; c0 < nchunks; c0 += kRouterRing)
    for_each<kRouterRing>([&](auto ic) {
      const int c = c0 + decltype(ic)::value;
      if (c >= nchunks) return;
      switch (min(nchunks - 1 - c, kRouterRing - 1)) {         // chunks that may still be on their way
        case 0: sync_keep_loads<0>(); break;
        case 1: sync_keep_loads<kPer>(); break;
        case 2: sync_keep_loads<2 * kPer>(); break;
        case 3: sync_keep_loads<3 * kPer>(); break;
        case 4: sync_keep_loads<4 * kPer>(); break;
        default: sync_keep_loads<5 * kPer>();
      }
      const bf16_t* st = stage(ic);
      const bf16_t* arow = st + r16 * kRouterKC;
      const bf16_t* brow = st + (TOK + wave * 16 + r16) * kRouterKC;
#pragma unroll
      for (int s = 0; s < kRouterKC / 32; ++s) {
        const int pos = ((s * 4 + kc) ^ r16) * 8;
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(arow + pos);
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(brow + pos);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
      }
      if (c + kRouterRing < nchunks) {
        __builtin_amdgcn_s_waitcnt(0xc07f);                    // this wave's reads of the stage have returned
        __builtin_amdgcn_s_barrier();
        issue(c + kRouterRing, stage(ic));
      }
    });
  if (tid < kMaxE) bias_s[tid] = my_bias;
  __shared__ unsigned long long mask_s[TOK];
  router_finish<TOK>(acc, sc, bias_s, T, E, k, norm_mode, t0, logits, idx, w, gap, chunk_hist, mask_s);
}

constexpr int kNormRouterMaxH = 1024, kNormGran = kNormRouterMaxH / 8 / kWave;

// A token's routing with the first pass of its experts behind it, for the few-token kernels: every workgroup works out the routing of its
// slot's token for itself and goes on to blocks of 32 rows of the slot's gate/up weights.  All of w_router (98 KB at E = 64, H = 768) comes
// from L2 to each workgroup at once (behind a norm three of 24 go out after the first wait at H = 768), and a launch and the gap behind it are saved.  One
// workgroup a CU at most (the LDS holds w_router), so with more slots each takes more blocks.  Kernels of a layer, router + gate/up launch
// -> this, weights from HBM, us: H = 768, I = 384, k = 6: 16.7 -> 14.7 (T = 1), 21.1 -> 19.4 (4), 26.5 -> 25.8 (8); H = 512, I = 256:
// 13.3 -> 10.6 (1), 18.1 -> 17.7 (8); H = 1024, I = 512, k = 8: 22.0 -> 17.4 (1), 30.8 -> 26.0 (4).  The host is through sooner too: the
// layer of one token at H = 768 takes 12.2 us instead of 15.6.  Same products in the same order as router_mfma_kernel and
// gateup_few_kernel.  Grid (blocks of rows shared out, T k); NG = H / 128.
// TN (the type of the norm's weights; void: no norm): the token's row goes through the block's input RMSNorm first, in every wave, with the
// arithmetic and the summation order of router_norm_mfma_kernel; the first workgroup of a token leaves it in `xn`.
// Kernels of norm + layer + sum, norm and router in a launch of their own -> this, us: H = 768, I = 384: 17.6 -> 13.3 (T = 1), 24.2 -> 19.2 (4),
// 28.2 -> 26.1 (8); H = 512, I = 256: 15.2 -> 11.5, 17.1 -> 13.0, 19.4 -> 16.6; H = 1024, I = 512, k = 8: 20.7 -> 16.5 (1), 32.7 -> 26.3 (4).
template <int NG, typename TN>
__global__ __launch_bounds__(256) void router_gateup_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ wr,
                                                            const float* __restrict__ bias, int Et, int k, int norm_mode,
                                                            float* __restrict__ logits, int32_t* __restrict__ idx,
                                                            float* __restrict__ w, const bf16_t* __restrict__ wgu, int E, int I2,
                                                            float* __restrict__ gu, const void* __restrict__ norm_weight, float eps,
                                                            bf16_t* __restrict__ xn) {
  constexpr bool kNorm = !std::is_same_v<TN, void>;
  constexpr int H = NG * kRouterKC, kGran = H / 8;
  __shared__ __attribute__((aligned(16))) bf16_t ws[kMaxE * H];
  __shared__ __attribute__((aligned(16))) bf16_t xs[H];
  __shared__ float sc[16 * kRowPad];
  __shared__ float bias_s[kMaxE];
  __shared__ int32_t idx_s[kMaxK];
  __shared__ float w_s[kMaxK];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int slot = blockIdx.y, t = slot / k, j = slot - t * k;
  const bf16_t* xr = x + (size_t)t * H;
  const bool first = blockIdx.x == 0 && j == 0;
  bf16x8 row[kNormGran];                               // granules u*64 + lane
  float nw[kNormGran][8];
  if constexpr (kNorm) {
#pragma unroll
    for (int u = 0; u < kNormGran; ++u) {
      const int c = min(u * kWave + lane, kGran - 1);
      row[u] = *reinterpret_cast<const bf16x8*>(xr + c * 8);
      TN v[8];
      if constexpr (sizeof(TN) == 2) *reinterpret_cast<bf16x8*>(v) = reinterpret_cast<const bf16x8*>(norm_weight)[c];
      else
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = static_cast<const TN*>(norm_weight)[c * 8 + q];
#pragma unroll
      for (int q = 0; q < 8; ++q) nw[u][q] = (float)v[q];
    }
  }
  // chunk-major stages as in router_mfma_kernel: granule c of a row sits at position c ^ (row & 15)
#pragma unroll
  for (int c = 0; c < NG; ++c)
#pragma unroll
    for (int i = 0; i < kMaxE / 16; ++i) {
      const int row = i * 16 + (tid >> 4), g = (tid & 15) ^ (row & 15);
      __builtin_amdgcn_global_load_lds((router_gbl_void*)(wr + (size_t)min(row, Et - 1) * H + c * kRouterKC + g * 8),
                                       (router_lds_void*)(ws + ((c * kMaxE + i * 16) * 16 + wave * 64) * 8), 16, 0, 0);
    }
  const int c16 = tid & 15, rg = tid >> 4;
  Raw8<bf16_t> xv[NG];
  if constexpr (kNorm) {
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < kNormGran; ++u)
      if (u * kWave + lane < kGran)
#pragma unroll
        for (int q = 0; q < 8; ++q) ss = fmaf((float)row[u][q], (float)row[u][q], ss);
    ss = wave_sum(ss);
    const float rinv = rsqrtf(ss / (float)H + eps);                                               // norm.py:22-23
#pragma unroll
    for (int u = 0; u < kNormGran; ++u) {
      const int c = u * kWave + lane;
      if (wave == u && c < kGran) {
        bf16x8 o;
#pragma unroll
        for (int q = 0; q < 8; ++q) o[q] = (bf16_t)(nw[u][q] * (float)(bf16_t)((float)row[u][q] * rinv));    // norm.py:24
        *reinterpret_cast<bf16x8*>(xs + c * 8) = o;
        if (first) *reinterpret_cast<bf16x8*>(xn + (size_t)t * H + c * 8) = o;
      }
    }
  } else {
#pragma unroll
    for (int u = 0; u < NG; ++u) xv[u].load(xr + (u * 16 + c16) * 8);
    if (tid < kGran) *reinterpret_cast<bf16x8*>(xs + tid * 8) = *reinterpret_cast<const bf16x8*>(xr + tid * 8);
  }
  if (tid < kMaxE) bias_s[tid] = tid < Et ? bias[tid] : 0.f;
  __builtin_amdgcn_s_waitcnt(0);                               // vmcnt(0): this thread's transfers of w_router have landed
  __syncthreads();
  if constexpr (kNorm) {
#pragma unroll
    for (int u = 0; u < NG; ++u) xv[u].v = *reinterpret_cast<const bf16x8*>(xs + (u * 16 + c16) * 8);
  }
  const int r16 = lane & 15, kc = lane >> 4;
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < NG; ++c)
#pragma unroll
    for (int s = 0; s < kRouterKC / 32; ++s) {
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(xs + c * kRouterKC + (s * 4 + kc) * 8);    // sixteen times the token's row
      const bf16x8 b = *reinterpret_cast<const bf16x8*>(ws + (c * kMaxE + wave * 16 + r16) * kRouterKC + ((s * 4 + kc) ^ r16) * 8);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
    }
  router_finish<16>(acc, sc, bias_s, 1, Et, k, norm_mode, 0, first && logits != nullptr ? logits + (size_t)t * Et : nullptr, idx_s, w_s,
                    nullptr, nullptr, nullptr);
  __syncthreads();
  if (first && tid < k) {
    idx[(size_t)t * k + tid] = idx_s[tid];
    w[(size_t)t * k + tid] = w_s[tid];
  }
  const int e = __builtin_amdgcn_readfirstlane(idx_s[j]);
  if ((unsigned)e >= (unsigned)E) return;                      // no GLU expert
  for (int row = blockIdx.x * kGateRows; row < I2; row += gridDim.x * kGateRows)
    gateup_rows<bf16_t, NG>(xv, wgu + (size_t)e * I2 * H, row + rg, c16, H, I2, gu + (size_t)slot * I2);
}

// ---- MFMA router with the block's input RMSNorm in front (the caller's seam) ----------------------
// out = h + moe(post_attention_layernorm(h)) (src/modeling/layers.py:57-64) needs the normalised rows twice: as the
// router's operand and as the rows the expert kernels gather.  This kernel reads the raw rows once: all H elements of
// its TOK rows arrive in LDS by LDS-DMA, one wave per row computes BiBoRMSNorm (src/modeling/norm.py:19-24) with the
// arithmetic and the summation order of rmsnorm_bf16x8_kernel (so both produce the same bits), writes the normalised
// row back to LDS in place and to `xn` in memory, and the logits are then multiplied from the resident rows while
// w_router streams through two LDS stages, two chunks a round trip, the first two requested in front of the rows.  A wave's four rows pass
// through the norm side by side and leave for memory behind the products: one row after the other and a chunk a round trip the whole seam
// took, us: H = 768, I = 384, k = 6: T = 16: 38.5 -> 37.7, 64: 43.2 -> 41.9, 2049: 66.0 -> 64.6, 6000: 127.2 -> 125.7; H = 512, I = 256, T = 512:
// 30.9 -> 29.7 (all with the sums over a wave in common.h, which are 0.2 to 0.8 of it).  x rows are stored as H/128 chunks of
// [TOK][128], granule c of a chunk row r at position c ^ (r & 15).
// What the selection needs lies where the rows were: 80 KB of LDS at TOK = 32 and H = 768, so that two workgroups share a CU and one's
// round trips pass behind the other's arithmetic (one a CU: 30.0 -> 21.7 us at T = 16384, 26.9 -> 19.9 at 12000).  RING: six chunks of
// w_router requested behind the rows, as in router_ring_kernel (H = 512, T = 1024: 10.8 -> 9.5 us; H = 768: 12.2 -> 11.4;
// T = 16: 9.8 -> 10.8, so not there).  The chunks arrive together, not behind the norm's arithmetic: the first use of the norm's weights,
// registers whose loads are older, is compiled into a wait for everything (H = 768, T = 2049: 10.2 us, where router_ring_kernel takes 8 without
// the norm).
template <int TOK>
constexpr int kNormTail = (TOK * kRowPad + kMaxE) * (int)sizeof(float) + TOK * (int)sizeof(unsigned long long);

template <int TOK, typename TN, bool RING>
__global__ __launch_bounds__(TOK * 16) void router_norm_mfma_kernel(const bf16_t* __restrict__ h, const TN* __restrict__ nw,
                                                                    float eps, const bf16_t* __restrict__ wr,
                                                                    const float* __restrict__ bias, int T, int H, int E,
                                                                    int k, int norm_mode, bf16_t* __restrict__ xn,
                                                                    float* __restrict__ logits, int32_t* __restrict__ idx,
                                                                    float* __restrict__ w, float* __restrict__ gap,
                                                                    int32_t* __restrict__ chunk_hist) {
  constexpr int kThreads = TOK * 16;
  constexpr int kWPer = kMaxE * kRouterGran / kThreads;      // w_router load instructions per thread and chunk
  extern __shared__ __attribute__((aligned(16))) bf16_t xs[];                 // [H/128][TOK][128]
  constexpr int kRingElems = RING ? kMaxE * kRouterKC : 8;
  __shared__ __attribute__((aligned(16))) bf16_t wst0[kMaxE * kRouterKC];
  __shared__ __attribute__((aligned(16))) bf16_t wst1[kMaxE * kRouterKC];
  __shared__ __attribute__((aligned(16))) bf16_t wst2[kRingElems];
  __shared__ __attribute__((aligned(16))) bf16_t wst3[kRingElems];
  __shared__ __attribute__((aligned(16))) bf16_t wst4[kRingElems];
  __shared__ __attribute__((aligned(16))) bf16_t wst5[kRingElems];
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int t0 = blockIdx.x * TOK;
  const int nchunks = H / kRouterKC;
  const int ngran = H / 8;
  const float my_bias = tid < E ? bias[tid] : 0.f;
  TN wv[kNormGran][8];                                 // the norm's weights of this lane's granules u*64 + lane, for all of the wave's rows
#pragma unroll
  for (int u = 0; u < kNormGran; ++u) {
    const int c = min(u * kWave + lane, ngran - 1);
    if constexpr (sizeof(TN) == 2) *reinterpret_cast<bf16x8*>(wv[u]) = reinterpret_cast<const bf16x8*>(nw)[c];
    else
#pragma unroll
      for (int q = 0; q < 8; ++q) wv[u][q] = nw[c * 8 + q];
  }
  __builtin_amdgcn_sched_barrier(0);                   // requested in front of w_router and of the rows

  // w_router chunk loads: thread t of instruction i fills granule i*kThreads + t = (row, position t % 16)
  const bf16_t* wsrc[kWPer];
#pragma unroll
  for (int i = 0; i < kWPer; ++i) {
    const int row = (i * kThreads + tid) / kRouterGran;
    wsrc[i] = wr + (size_t)min(row, E - 1) * H + ((tid & (kRouterGran - 1)) ^ (row & 15)) * 8;
  }
  auto issue_w = [&](int k0, bf16_t* st) {
#pragma unroll
    for (int i = 0; i < kWPer; ++i)
      __builtin_amdgcn_global_load_lds((router_gbl_void*)(wsrc[i] + k0), (router_lds_void*)(st + (i * kThreads + wave * 64) * 8),
                                       16, 0, 0);
  };
  auto stage = [&](auto ic) -> bf16_t* {
    constexpr int i = decltype(ic)::value;
    if constexpr (i == 0) return wst0; else if constexpr (i == 1) return wst1; else if constexpr (i == 2) return wst2;
    else if constexpr (i == 3) return wst3; else if constexpr (i == 4) return wst4; else return wst5;
  };
  if constexpr (!RING) {
    issue_w(0, wst0);
    if (nchunks > 1) issue_w(kRouterKC, wst1);
  }
  // the raw rows: instruction i is chunk i of every row (TOK * 16 granules = one per thread)
  {
    const int row = tid >> 4;
    const bf16_t* src = h + (size_t)min(t0 + row, T - 1) * H + ((tid & 15) ^ (row & 15)) * 8;
    for (int i = 0; i < nchunks; ++i)
      __builtin_amdgcn_global_load_lds((router_gbl_void*)(src + i * kRouterKC),
                                       (router_lds_void*)(xs + (i * kThreads + wave * 64) * 8), 16, 0, 0);
  }
  if constexpr (RING) {
    for_each<kRouterRing>([&](auto ic) { if (decltype(ic)::value < nchunks) issue_w(decltype(ic)::value * kRouterKC, stage(ic)); });
    switch (min(nchunks, kRouterRing)) {               // the rows have arrived
      case 1: sync_keep_loads<kWPer>(); break;
      case 2: sync_keep_loads<2 * kWPer>(); break;
      case 3: sync_keep_loads<3 * kWPer>(); break;
      case 4: sync_keep_loads<4 * kWPer>(); break;
      case 5: sync_keep_loads<5 * kWPer>(); break;
      default: sync_keep_loads<6 * kWPer>();
    }
  } else {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  // RMSNorm, one wave per row, four rows per wave, which pass through each step side by side (one after the other their reads wait for the
  // writes of the row before); lane takes logical granules u*64 + lane of the row.  They leave for memory behind the products, whose waits for
  // w_router would be for them too.
  bf16x8 v[4][kNormGran];
  {
    float rinv[4];
    auto place = [&](int j, int u) {
      const int c = u * kWave + lane, r = wave * 4 + j;
      return xs + (((c >> 4) * TOK + r) * kRouterGran + ((c & 15) ^ (r & 15))) * 8;
    };
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int u = 0; u < kNormGran; ++u)
        if (u * kWave + lane < ngran) v[j][u] = *reinterpret_cast<const bf16x8*>(place(j, u));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float ss = 0.f;
#pragma unroll
      for (int u = 0; u < kNormGran; ++u)
        if (u * kWave + lane < ngran)
#pragma unroll
          for (int q = 0; q < 8; ++q) ss = fmaf((float)v[j][u][q], (float)v[j][u][q], ss);
      rinv[j] = ss;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) rinv[j] = rsqrtf(wave_sum(rinv[j]) / (float)H + eps);       // norm.py:22-23
#pragma unroll
    for (int u = 0; u < kNormGran; ++u) {
      const int c = u * kWave + lane;
      if (c < ngran)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
          for (int q = 0; q < 8; ++q) v[j][u][q] = (bf16_t)((float)wv[u][q] * (float)(bf16_t)((float)v[j][u][q] * rinv[j]));   // norm.py:24
          *reinterpret_cast<bf16x8*>(place(j, u)) = v[j][u];
        }
    }
  }
  const int tm = wave >> 2, en = wave & 3;
  const int r16 = lane & 15, kc = lane >> 4;
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const bf16_t* xa, const bf16_t* st) {
    const bf16_t* arow = xa + (tm * 16 + r16) * kRouterKC;
    const bf16_t* brow = st + (en * 16 + r16) * kRouterKC;
#pragma unroll
    for (int s = 0; s < kRouterKC / 32; ++s) {
      const int pos = ((s * 4 + kc) ^ r16) * 8;
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(arow + pos);
      const bf16x8 b = *reinterpret_cast<const bf16x8*>(brow + pos);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
    }
  };
  if constexpr (RING) {
    for (int c0 = 0; c0 < nchunks; c0 += kRouterRing)
      for_each<kRouterRing>([&](auto ic) {
        const int c = c0 + decltype(ic)::value;
        if (c >= nchunks) return;
        if (c == 0) __builtin_amdgcn_s_waitcnt(0xc07f);          // this wave's normalised rows are in LDS
        switch (min(nchunks - 1 - c, kRouterRing - 1)) {         // chunks that may still be on their way
          case 0: sync_keep_loads<0>(); break;
          case 1: sync_keep_loads<kWPer>(); break;
          case 2: sync_keep_loads<2 * kWPer>(); break;
          case 3: sync_keep_loads<3 * kWPer>(); break;
          case 4: sync_keep_loads<4 * kWPer>(); break;
          default: sync_keep_loads<5 * kWPer>();
        }
        multiply(xs + (size_t)c * TOK * kRouterKC, stage(ic));
        if (c + kRouterRing < nchunks) {
          __builtin_amdgcn_s_waitcnt(0xc07f);                    // this wave's reads of the stage have returned
          __builtin_amdgcn_s_barrier();
          issue_w((c + kRouterRing) * kRouterKC, stage(ic));
        }
      });
  } else {
    for (int c0 = 0; c0 < nchunks; c0 += 2) {            // two chunks a round trip; the first two are requested in front of the rows
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();                                   // first pass: also the normalised rows of the other waves
      multiply(xs + (size_t)c0 * TOK * kRouterKC, wst0);
      if (c0 + 1 < nchunks) multiply(xs + (size_t)(c0 + 1) * TOK * kRouterKC, wst1);
      if (c0 + 2 < nchunks) {
        __syncthreads();
        issue_w((c0 + 2) * kRouterKC, wst0);
        if (c0 + 3 < nchunks) issue_w((c0 + 3) * kRouterKC, wst1);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int u = 0; u < kNormGran; ++u) {
      const int c = u * kWave + lane, t = t0 + wave * 4 + j;
      if (c < ngran && t < T) *reinterpret_cast<bf16x8*>(xn + (size_t)t * H + c * 8) = v[j][u];
    }
  // the rows' LDS holds what is left to do: scores, bias, selections
  __syncthreads();
  float* sc = reinterpret_cast<float*>(xs);
  float* bias_s = sc + TOK * kRowPad;
  unsigned long long* mask_s = reinterpret_cast<unsigned long long*>(bias_s + kMaxE);
  if (tid < kMaxE) bias_s[tid] = my_bias;
  router_finish<TOK>(acc, sc, bias_s, T, E, k, norm_mode, t0, logits, idx, w, gap, chunk_hist, mask_s);
}

// ---- MFMA router for H % 32 == 0 but not % 128: operands straight to registers, K split over 4 waves ----
constexpr int kMfmaTokens = 16;

__global__ __launch_bounds__(256) void router_mfma_split_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ wr,
                                                                const float* __restrict__ bias, int T, int H, int E,
                                                                int k, int norm_mode, float* __restrict__ logits,
                                                                int32_t* __restrict__ idx, float* __restrict__ w,
                                                                float* __restrict__ gap, int32_t* __restrict__ chunk_hist) {
  __shared__ float part[4 * kMfmaTokens * kRowPad];
  __shared__ float sc[kMfmaTokens * kRowPad];
  __shared__ float bias_s[kMaxE];
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int t0 = blockIdx.x * kMfmaTokens;
  if (tid < kMaxE) bias_s[tid] = (tid < E) ? bias[tid] : 0.f;

  const int r16 = lane & 15, kc = lane >> 4;                 // fragment row, 8-wide k chunk
  const bf16_t* xa = x + (size_t)min(t0 + r16, T - 1) * H + kc * 8;
  const bf16_t* wb[4];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) wb[nt] = wr + (size_t)min(nt * 16 + r16, E - 1) * H + kc * 8;
  floatx4 acc[4];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) acc[nt] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int nsteps = H / 32;
  constexpr int kU = 8;                                      // K steps whose loads are issued together (160 VGPRs)
  for (int s0 = wave; s0 < nsteps; s0 += 4 * kU) {
    bf16x8 a[kU], b[kU][4];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int s = s0 + 4 * u;
      if (s < nsteps) {
        a[u] = *reinterpret_cast<const bf16x8*>(xa + s * 32);
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) b[u][nt] = *reinterpret_cast<const bf16x8*>(wb[nt] + s * 32);
      }
    }
#pragma unroll
    for (int u = 0; u < kU; ++u)
      if (s0 + 4 * u < nsteps) {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], b[u][nt], acc[nt], 0, 0, 0);
      }
  }
  // D layout of the 16x16 tile: lane holds column (expert) lane%16, rows (tokens) 4*(lane/16)+i
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      part[(wave * kMfmaTokens + kc * 4 + i) * kRowPad + nt * 16 + r16] = acc[nt][i];
  __syncthreads();
  const int ntok = min(kMfmaTokens, T - t0);
  for (int i = tid; i < kMfmaTokens * kMaxE; i += 256) {
    const int tl = i >> 6, e = i & 63;
    if (tl < ntok && e < E) {
      const int o = tl * kRowPad + e;
      const float lg = ((part[o] + part[kMfmaTokens * kRowPad + o]) + part[2 * kMfmaTokens * kRowPad + o]) +
                       part[3 * kMfmaTokens * kRowPad + o];
      if (logits != nullptr) logits[(size_t)(t0 + tl) * E + e] = lg;
      sc[o] = sigmoid32_canonical(lg);                       // router.py:31
    }
  }
  __syncthreads();
  const unsigned long long mask = select_tokens16(sc, bias_s, E, k, norm_mode, t0, ntok, idx, w, gap);
  __shared__ unsigned long long mask_s[kMfmaTokens];
  if (chunk_hist != nullptr) write_chunk_hist<kMfmaTokens>(mask, chunk_hist, mask_s);
}

}  // namespace

bool router_norm_supported(int H, int dtype, const void* h, const void* w_router, const void* xn) {
  const bool aligned = ((reinterpret_cast<uintptr_t>(h) | reinterpret_cast<uintptr_t>(w_router) |
                         reinterpret_cast<uintptr_t>(xn)) & 15) == 0;
  return dtype == BIBO_DTYPE_BF16 && (H % kRouterKC) == 0 && H <= kNormRouterMaxH && aligned;
}

// the kernel's TOK whole rows sit in dynamic LDS: allowed once per device, for the widest rows it takes
template <int TOK, typename TN, bool RING>
hipError_t allow_dynamic_lds() {
  static LdsLimitOnce once;
  return once.raise(reinterpret_cast<const void*>(&router_norm_mfma_kernel<TOK, TN, RING>), (int)(TOK * kNormRouterMaxH * sizeof(bf16_t)));
}

// RMSNorm + router in one launch (see router_norm_mfma_kernel); `xn` receives the normalised rows.
hipError_t launch_router_norm(const void* h, Vec norm_weight, float eps, const void* w_router, const float* bias,
                              int T, int H, int E, int k, int norm_mode, void* xn, float* logits, int32_t* idx, float* w,
                              int32_t* chunk_hist, int* hist_tokens, hipStream_t s) {
  if (hist_tokens != nullptr) *hist_tokens = 0;
  if (T == 0) return hipSuccess;
  const bf16_t* hp = static_cast<const bf16_t*>(h);
  const bf16_t* wp = static_cast<const bf16_t*>(w_router);
  bf16_t* xp = static_cast<bf16_t*>(xn);
  auto launch = [&](auto tok, auto ring, auto* nw) -> hipError_t {
    constexpr int TOK = decltype(tok)::value;
    constexpr bool RING = decltype(ring)::value;
    using TN = std::remove_const_t<std::remove_pointer_t<decltype(nw)>>;
    const hipError_t e = allow_dynamic_lds<TOK, TN, RING>();
    if (e != hipSuccess) return e;
    const size_t rows = (size_t)TOK * H * sizeof(bf16_t), lds = rows > (size_t)kNormTail<TOK> ? rows : (size_t)kNormTail<TOK>;
    hipLaunchKernelGGL((router_norm_mfma_kernel<TOK, TN, RING>), dim3((T + TOK - 1) / TOK), dim3(TOK * 16), lds, s, hp, nw, eps, wp, bias, T, H, E, k, norm_mode, xp, logits, idx, w, nullptr, chunk_hist);
    return hipGetLastError();
  };
  auto typed = [&](auto tok, auto ring) {
    return norm_weight.bf16 ? launch(tok, ring, static_cast<const bf16_t*>(norm_weight.p))
                            : launch(tok, ring, static_cast<const float*>(norm_weight.p));
  };
  using std::integral_constant;
  const hipError_t e = T >= 32 * 256 ? typed(integral_constant<int, 32>(), std::false_type())
                       : T >= kRingLeast && T <= 16 * kCUs ? typed(integral_constant<int, 16>(), std::true_type())
                                        : typed(integral_constant<int, 16>(), std::false_type());
  if (e != hipSuccess) return e;
  if (hist_tokens != nullptr && chunk_hist != nullptr) *hist_tokens = T >= 32 * 256 ? 32 : 16;
  return hipSuccess;
}

bool router_gateup_supported(int T, int H, int k, int I, int dtype, const void* x, const void* w_router) {
  return dtype == BIBO_DTYPE_BF16 && H % kRouterKC == 0 && H <= 8 * kRouterKC && T >= 1 &&
         ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w_router)) & 15) == 0;
}

hipError_t launch_router_gateup(const void* x, const void* w_router, const float* bias, int T, int H, int Et, int k, int norm_mode,
                                float* logits, int32_t* idx, float* w, const void* wgu, int E, int I, float* gu, Vec norm_weight, float eps,
                                void* xn, hipStream_t s) {
  const int blocks = (2 * I + kGateRows - 1) / kGateRows, most = kCUs / (T * k), each = (blocks + most - 1) / most;
  auto typed = [&](auto ng, auto* tn) {
    using TN = std::remove_pointer_t<decltype(tn)>;
    hipLaunchKernelGGL((router_gateup_kernel<decltype(ng)::value, TN>), dim3((blocks + each - 1) / each, T * k), dim3(256), 0, s,
                       static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w_router), bias, Et, k, norm_mode, logits, idx, w,
                       static_cast<const bf16_t*>(wgu), E, 2 * I, gu, norm_weight.p, eps, static_cast<bf16_t*>(xn));
  };
  auto launch = [&](auto ng) {
    if (xn == nullptr) typed(ng, static_cast<void*>(nullptr));
    else if (norm_weight.bf16) typed(ng, static_cast<bf16_t*>(nullptr));
    else typed(ng, static_cast<float*>(nullptr));
  };
  using std::integral_constant;
  switch (H / kRouterKC) {
    case 1: launch(integral_constant<int, 1>{}); break;
    case 2: launch(integral_constant<int, 2>{}); break;
    case 3: launch(integral_constant<int, 3>{}); break;
    case 4: launch(integral_constant<int, 4>{}); break;
    case 5: launch(integral_constant<int, 5>{}); break;
    case 6: launch(integral_constant<int, 6>{}); break;
    case 7: launch(integral_constant<int, 7>{}); break;
    case 8: launch(integral_constant<int, 8>{}); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_router(const void* x, const void* w_router, const float* bias, int T, int H, int E, int k, int dtype,
                         int norm_mode, float* logits, int32_t* idx, float* w, float* gap, int32_t* chunk_hist,
                         int* hist_tokens, hipStream_t s) {
  if (hist_tokens != nullptr) *hist_tokens = 0;
  if (T == 0) return hipSuccess;
  const bool aligned = ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w_router)) & 15) == 0;
  if (dtype == BIBO_DTYPE_BF16 && (H % kRouterKC) == 0 && aligned) {
    // 32 tokens per workgroup halve the w_router traffic per token; below 256 workgroups' worth of tokens the
    // smaller tile keeps more CUs busy
    if (T >= 32 * 256)
      hipLaunchKernelGGL(router_mfma_kernel<32>, dim3((T + 31) / 32), dim3(512), 0, s, static_cast<const bf16_t*>(x),
                         static_cast<const bf16_t*>(w_router), bias, T, H, E, k, norm_mode, logits, idx, w, gap,
                         chunk_hist);
    else if (T >= kRingLeast && T <= 16 * kCUs && H >= kRouterRing * kRouterKC)
      // us, two stages -> ring: 9.3 -> 8.0 (H = 768, T = 128), 8.6 -> 7.6 (2049), 9.2 -> 8.0 (4096); 10.7 -> 8.9 (H = 1024, T = 128 to
      // 2049), 11.0 -> 9.0 (4096).  Few workgroups have the memory to themselves and only pay the larger launch: 5.6 -> 6.4 (H = 768,
      // T = 16), 6.7 -> 7.4 (H = 1024); four chunks and fewer gain 0.3 at most.
      hipLaunchKernelGGL(router_ring_kernel, dim3((T + 15) / 16), dim3(256), 0, s, static_cast<const bf16_t*>(x),
                         static_cast<const bf16_t*>(w_router), bias, T, H, E, k, norm_mode, logits, idx, w, gap,
                         chunk_hist);
    else
      hipLaunchKernelGGL(router_mfma_kernel<16>, dim3((T + 15) / 16), dim3(256), 0, s, static_cast<const bf16_t*>(x),
                         static_cast<const bf16_t*>(w_router), bias, T, H, E, k, norm_mode, logits, idx, w, gap,
                         chunk_hist);
    if (hist_tokens != nullptr && chunk_hist != nullptr) *hist_tokens = T >= 32 * 256 ? 32 : 16;
  } else if (dtype == BIBO_DTYPE_BF16 && (H % 32) == 0 && aligned) {
    chunk_hist = T < 32 * 256 ? chunk_hist : nullptr;   // (one per 16 tokens: too many to add up for larger batches)
    const int grid = (T + kMfmaTokens - 1) / kMfmaTokens;
    hipLaunchKernelGGL(router_mfma_split_kernel, dim3(grid), dim3(256), 0, s, static_cast<const bf16_t*>(x),
                       static_cast<const bf16_t*>(w_router), bias, T, H, E, k, norm_mode, logits, idx, w, gap, chunk_hist);
    if (hist_tokens != nullptr && chunk_hist != nullptr) *hist_tokens = kMfmaTokens;
  } else {
    chunk_hist = T < 32 * 256 ? chunk_hist : nullptr;
    const dim3 grid((T + kGenTokens - 1) / kGenTokens);
    const bool vec = aligned && H % 4 == 0;
    auto launch = [&](auto kernel, auto* xp) {
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, xp, static_cast<decltype(xp)>(w_router), bias, T, H, E, k, norm_mode,
                         logits, idx, w, gap, chunk_hist);
    };
    if (dtype == BIBO_DTYPE_BF16) {
      const bf16_t* xp = static_cast<const bf16_t*>(x);
      if (vec) launch(router_f32_kernel<bf16_t, true>, xp); else launch(router_f32_kernel<bf16_t, false>, xp);
    } else {
      const float* xp = static_cast<const float*>(x);
      if (vec) launch(router_f32_kernel<float, true>, xp); else launch(router_f32_kernel<float, false>, xp);
    }
    if (hist_tokens != nullptr && chunk_hist != nullptr) *hist_tokens = kGenTokens;
  }
  return hipGetLastError();
}

}  // namespace bibo
