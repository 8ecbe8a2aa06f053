// Grouped GEMMs in fp32 arithmetic for the generic family (fp32 operands, and bf16 sizes no bf16 tile divides), gfx950.
//
// Two kernels: ggemm_f32_kernel on fp32 MFMAs (154 TFLOP/s) for experts with few rows, ggemm_split_kernel and wgrad_split_kernel on bf16
// MFMAs, sixteen times as fast, which multiply three bf16 parts of every number where the other multiplies the number: six products for one.
//
// How a dot product is summed.  One chain over all of K, which the accumulators would form by themselves, is as far from the exact result
// as the square root of its length says: the layer at H = 768, I = 384 was off by 8.4e-7 (2-norm), one routed row at a time, whose dot
// products are 64 partial sums and a tree, by 1.81e-7.  ggemm_f32_kernel: chains of eight products inside the MFMAs, a step's four chains in
// fp32, the steps in fp64: 1.49e-7.  ggemm_split_kernel: a step inside the MFMAs, which add eight products at a time and round once, the
// small products first; the steps in fp64, every other one with its sign turned: 1.15e-7, and nowhere from H = 64 to 1024 more than the other
// (the three products of nine that are left out are below 2^-26 of theirs).
//
// LDS layout of ggemm_f32_kernel's K step of 32: [rows][32], 128-byte rows; 16-byte granule c of row r sits at c ^ ((r >> 1) & 7), so 16
// consecutive rows read without bank conflicts.  A lane reads a granule (4 consecutive k) and feeds its four elements to four MFMAs, the
// same k on both sides (the order of the K elements inside a step does not matter otherwise).  Operands are widened to fp32 on their way.
#pragma once

#include "kmajor.h"

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
// 16 rows x 64 columns, four waves along the columns, 16x16 tiles: few rows per expert, where what counts is the MFMA time per
// streamed weight byte.
template <typename TA, typename TW, bool GATHER, bool SCATTER>
__global__ __launch_bounds__(256, 4) void ggemm_f32_kernel(const TA* __restrict__ A, const int32_t* __restrict__ a_index,
                                                        const TW* __restrict__ W, const int32_t* __restrict__ offsets,
                                                        const int32_t* __restrict__ out_index,
                                                        const float* __restrict__ out_scale, int K, int N, int E, int nblk_n,
                                                        float* __restrict__ out) {
  constexpr int BM = 16, BN = 64, W_PER = 2;                     // granules of four elements of W per thread and step
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
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int n0 = nb * BN;
  if (tid < BM) {
    const int r = row0 + min(tid, rows - 1);
    const int d = SCATTER ? out_index[r] : r;
    dst_s[tid] = d;
    scale_s[tid] = SCATTER && out_scale != nullptr ? out_scale[d] : 1.f;
  }
  const int ac = tid & 7;
  const bool a_live = tid < BM * 8;
  const int ar = row0 + min(tid >> 3, rows - 1);                 // rows past the end repeat the last one
  const TA* const arow = A + (size_t)(GATHER ? a_index[ar] : ar) * K;
  const TW* wbase = W + (size_t)e * K * N;
  floatx4 ra, rw[W_PER];
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  auto load = [&](int k0) {
    ra = a_live && k0 + ac * 4 < K ? load4<TA>(arow + k0 + ac * 4) : zero;
#pragma unroll
    for (int i = 0; i < W_PER; ++i) {
      const int g = tid + 256 * i, n = n0 + (g >> 3), k = k0 + (g & 7) * 4;
      rw[i] = n < N && k < K ? load4<TW>(wbase + (size_t)n * K + k) : zero;
    }
  };
  auto store = [&](int st) {
    if (a_live) *reinterpret_cast<floatx4*>(&As[st][fswz(tid >> 3, ac)]) = ra;
#pragma unroll
    for (int i = 0; i < W_PER; ++i) {
      const int g = tid + 256 * i;
      *reinterpret_cast<floatx4*>(&Ws[st][fswz(g >> 3, g & 7)]) = rw[i];
    }
  };
  const int nsteps = (K + kFK - 1) / kFK;
  load(0);
  store(0);
  __syncthreads();
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

// ---- the same on bf16 MFMAs --------------------------------------------------------------------------------------------
// An fp32 number is the sum of three bf16 numbers (8 bits of mantissa each and the signs of the rests), so a product of two is nine
// bf16 products, of which the three smallest lie below 2^-24 of it.  The other six cost 6 x 16 cycles of the MFMA pipe per 16 x 16 x 32
// block where fp32 MFMAs take 256.  A bf16 operand is its own one part.  What bounds a 128 x 128 tile's step of 32: 1536 cycles of MFMAs,
// as many of LDS reads, about 1200 of vector instructions (11 for two numbers' parts, and the fp64 sums), which therefore go between the
// MFMAs; apart from them the waves of a workgroup did one after the other (159 us where it is 131 now).  T = 2048, H = 768, E = 64, k = 6,
// I = 384: gate/up 228 -> 133 us, down 120 -> 78, the layer 325 -> 250 (collected bits and turned signs are 4 of it); bf16 operands,
// T = 3000, H = 520, I = 296: 199 -> 58, 110 -> 42.

template <typename T> struct Planes { static constexpr int n = 3; typedef floatx4 raw; };
template <> struct Planes<bf16_t> { static constexpr int n = 1; typedef bf16x4 raw; };
__device__ __forceinline__ floatx4 widen4(floatx4 v) { return v; }
__device__ __forceinline__ floatx4 widen4(bf16x4 v) { return floatx4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]}; }
// Plane p of four consecutive elements, which v holds less the planes before it, to LDS; v keeps the rest.  A number whose lowest bit lies
// below 2^-133, bf16's smallest subnormal, is not the sum of three parts (all others are: the rest behind two parts has eight bits at
// most).  The rest then is an fp32 subnormal with some of its low 16 bits set, which no other third part has: `rests` collects them.
// NEG: of their negatives.
template <int P, bool NEG = false>
__device__ __forceinline__ void put_plane(bf16_t* to, floatx4& v, unsigned& rests) {
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  if constexpr (P == 2) {
    rests |= __float_as_uint(v[0]) | __float_as_uint(v[1]);
    rests |= __float_as_uint(v[2]) | __float_as_uint(v[3]);
  }
  if constexpr (NEG && P == 0) v = -v;
  const u32x2 u = {__builtin_bit_cast(unsigned, bf16x2{(bf16_t)v[0], (bf16_t)v[1]}), __builtin_bit_cast(unsigned, bf16x2{(bf16_t)v[2], (bf16_t)v[3]})};
  *reinterpret_cast<u32x2*>(to) = u;
  if constexpr (P < 2) {
    v[0] -= __uint_as_float(u[0] << 16);
    v[1] -= __uint_as_float(u[0] & 0xffff0000u);
    v[2] -= __uint_as_float(u[1] << 16);
    v[3] -= __uint_as_float(u[1] & 0xffff0000u);
  }
}
template <int P, bool NEG = false>
__device__ __forceinline__ void put_plane(bf16_t* to, bf16x4& v, unsigned&) { *reinterpret_cast<bf16x4*>(to) = NEG ? -v : v; }
__device__ __forceinline__ bool bits_lost(unsigned rests) { return (rests & 0xffffu) != 0; }

// Element offset of the four k from 4 c on of row r in a [rows][32] plane: 64-byte rows, 16-byte granules as in the stripe layout.
__device__ __forceinline__ int aswz(int r, int c) { return r * kFK + (((c >> 1) ^ ((r >> 2) & 3)) << 3) + ((c & 1) << 2); }
// Element offset of columns 4 c on of row k in a K-major [32][BN] plane.  The four k rows that one transposing read touches lie in four
// different 64-byte quarters of the bank period.
template <int BN>
__device__ __forceinline__ int kswz(int k, int c) {
  static_assert(BN == 64 || BN == 128, "one or two bank periods per two rows");
  return k * BN + (((c >> 1) ^ (BN == 128 ? (k & 3) << 2 : (k & 2) << 1)) << 3) + ((c & 1) << 2);
}
// The fragment of k16 step ks of the 32 columns from nbase on (kmajor.h has the lanes of ds_read_b64_tr_b16).
template <int BN>
__device__ __forceinline__ bf16x8 kplane_frag(const bf16_t* plane, int lane, int nbase, int ks) {
  const int r = lane & 15, g16 = lane >> 4;
  const int k = 16 * ks + 8 * (g16 >> 1) + (r >> 2), c = (nbase + 16 * (g16 & 1)) / 4 + (r & 3);
  const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(plane + kswz<BN>(k, c)));
  const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(plane + kswz<BN>(k + 4, c)));
  typedef short v8i16 __attribute__((ext_vector_type(8)));
  return __builtin_bit_cast(bf16x8, v8i16{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
}

// f(0), f(1), .. f(N - 1) with the index as a constant
template <typename F, int... Is>
__device__ __forceinline__ void for_each(F f, std::integer_sequence<int, Is...>) { (f(std::integral_constant<int, Is>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void for_each(F f) { for_each(f, std::make_integer_sequence<int, N>{}); }

// WM x WN waves, each 32 rows x 32 NTW columns.
template <int WM, int WN, int NTW, typename TA, typename TW, bool W_KM, bool GATHER, bool SCATTER>
__global__ __launch_bounds__(64 * WM * WN, 2) void ggemm_split_kernel(const TA* __restrict__ A, const int32_t* __restrict__ a_index,
                                                                      const TW* __restrict__ W, const int32_t* __restrict__ offsets,
                                                                      const int32_t* __restrict__ out_index,
                                                                      const float* __restrict__ out_scale, int K, int N, int E,
                                                                      int nblk_n, float* __restrict__ out) {
  constexpr int BM = 32 * WM, BN = 32 * NTW * WN, kThreads = 64 * WM * WN, PA = Planes<TA>::n, PW = Planes<TW>::n;
  constexpr int A_PER = BM * 8 / kThreads, W_PER = BN * 8 / kThreads;
  __shared__ __attribute__((aligned(16))) bf16_t As[2][PA * BM * kFK];
  __shared__ __attribute__((aligned(16))) bf16_t Ws[2][PW * BN * kFK];
  __shared__ int dst_s[BM];
  __shared__ float scale_s[BM];
  const TileMap tm = make_tile_map(offsets, E, BM);
  const int total = tm.total * nblk_n;
  const int flat = xcd_tile(blockIdx.x, total);
  if (flat >= total) return;
  const int tile = flat / nblk_n, n0 = (flat - tile * nblk_n) * BN;
  int e, row0, rows;
  find_tile(tm, tile, e, row0, rows);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  if (tid < BM) {
    const int r = row0 + min(tid, rows - 1);
    const int d = SCATTER ? out_index[r] : r;
    dst_s[tid] = d;
    scale_s[tid] = SCATTER && out_scale != nullptr ? out_scale[d] : 1.f;
  }
  typedef typename Planes<TA>::raw RawA;
  typedef typename Planes<TW>::raw RawW;
  RawA ra[2][A_PER];                                             // two steps on their way to LDS
  RawW rw[2][W_PER];
  const int ac = tid & 7, ar = tid >> 3;
  const TA* arow[A_PER];
#pragma unroll
  for (int i = 0; i < A_PER; ++i) {
    const int r = row0 + min(ar + kThreads / 8 * i, rows - 1);    // rows past the end repeat the last one
    arow[i] = A + (size_t)(GATHER ? a_index[r] : r) * K;
  }
  const TW* wbase = W + (size_t)e * K * N;
  // Columns past N repeat the last ones and are not stored; k past K are zeros (TAIL: the last, partial step).
  auto load = [&](auto set_c, auto tail_c, int k0) {
    constexpr int set = decltype(set_c)::value;
    constexpr bool tail = decltype(tail_c)::value;
    const int k = tail ? min(k0 + ac * 4, K - 4) : k0 + ac * 4;
    const bool live = !tail || k0 + ac * 4 < K;
#pragma unroll
    for (int i = 0; i < A_PER; ++i) {
      ra[set][i] = *reinterpret_cast<const RawA*>(arow[i] + k);
      if (!live) ra[set][i] = RawA{};
    }
#pragma unroll
    for (int i = 0; i < W_PER; ++i) {
      if constexpr (W_KM) {
        const int g = tid + kThreads * i, kr = k0 + g / (BN / 4), n = min(n0 + g % (BN / 4) * 4, N - 4);
        rw[set][i] = *reinterpret_cast<const RawW*>(wbase + (size_t)(tail ? min(kr, K - 1) : kr) * N + n);
        if (tail && kr >= K) rw[set][i] = RawW{};
      } else {
        const int n = min(n0 + ar + kThreads / 8 * i, N - 1);
        rw[set][i] = *reinterpret_cast<const RawW*>(wbase + (size_t)n * K + k);
        if (!live) rw[set][i] = RawW{};
      }
    }
  };
  unsigned rests = 0;
  // one plane of one of a thread's A_PER + W_PER quadruples to its stage
  auto put = [&](auto set_c, auto q_c) {
    constexpr int set = decltype(set_c)::value, q = decltype(q_c)::value;
    if constexpr (q < A_PER * PA) {
      constexpr int i = q / PA, p = q % PA;
      put_plane<p, set == 1>(As[set] + p * (BM * kFK) + aswz(ar + kThreads / 8 * i, ac), ra[set][i], rests);
    } else if constexpr (q < A_PER * PA + W_PER * PW) {
      constexpr int i = (q - A_PER * PA) / PW, p = (q - A_PER * PA) % PW;
      const int g = tid + kThreads * i;
      put_plane<p>(Ws[set] + p * (BN * kFK) + (W_KM ? kswz<BN>(g / (BN / 4), g % (BN / 4)) : aswz(ar + kThreads / 8 * i, ac)), rw[set][i], rests);
    }
  };
  const int wm = wave % WM, wn = wave / WM, l32 = lane & 31, h = lane >> 5;
  const bool busy = wm * 32 < rows;                              // a wave without rows only loads
  double sum[NTW][16];
  floatx16 none;
#pragma unroll
  for (int i = 0; i < 16; ++i) none[i] = 0.f;
#pragma unroll
  for (int j = 0; j < NTW; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) sum[j][i] = 0.;
  auto afrag = [&](int st, int p, int ks) {
    return *reinterpret_cast<const bf16x8*>(As[st] + p * (BM * kFK) + aswz(wm * 32 + l32, 2 * (2 * ks + h)));
  };
  auto wfrag = [&](int st, int p, int j, int ks) {
    const bf16_t* plane = Ws[st] + p * (BN * kFK);
    const int nb = (wn * NTW + j) * 32;
    if constexpr (W_KM) return kplane_frag<BN>(plane, lane, nb, ks);
    else return *reinterpret_cast<const bf16x8*>(plane + aswz(nb + l32, 2 * (2 * ks + h)));
  };
  // What a bf16 MFMA adds to a sum much smaller than itself cuts off that sum's bits below its own towards minus infinity (0.12 of a last
  // place on average; fp32 MFMAs round to nearest).  Over the steps, and over the k rows of a token, that adds up: d_x of 98 tokens, H = 536,
  // I = 400, E = 64, k = 8, was off by 2.14e-7 where fp32 MFMAs are by 2.05e-7, of 2 experts by 1.76e-7 and 1.84e-7.  So every other step
  // multiplies the negatives of A's rows and is subtracted.
  // Step s multiplies stage st = s % 2.  Between its MFMAs, two at a time, go the next step's planes from registers to the other stage and
  // the previous step's sums into the fp64 ones: vector instructions that would otherwise wait for the MFMA pipe and it for them.
  floatx16 acc[2][NTW];
  constexpr int kSmall = PA * PW == 9 ? 5 : PA * PW == 3 ? 2 : 0, kChunks = 2 * kSmall + 2, kPuts = A_PER * PA + W_PER * PW;
  auto step = [&](auto st_c) {
    constexpr int st = decltype(st_c)::value;
    bf16x8 a[2][PA], b[2][NTW][PW];
    auto read = [&](auto ks_c) {
      constexpr int ks = decltype(ks_c)::value;
#pragma unroll
      for (int p = 0; p < PA; ++p) a[ks][p] = afrag(st, p, ks);
#pragma unroll
      for (int j = 0; j < NTW; ++j)
#pragma unroll
        for (int p = 0; p < PW; ++p) b[ks][j][p] = wfrag(st, p, j, ks);
    };
    using std::integral_constant;
    read(integral_constant<int, 0>{});
    auto chunk = [&](auto c_c) {
      constexpr int c = decltype(c_c)::value;
      if constexpr (c == (kSmall > 2 ? 2 : 0)) read(integral_constant<int, 1>{});
      // products: the small ones of both k16 steps first, while the sum they enter is small itself (what is rounded at the sum's own size
      // are the four blocks of eight high products)
      constexpr int ks = c < 2 * kSmall ? c / (kSmall > 0 ? kSmall : 1) : c - 2 * kSmall;
      constexpr int q = c < 2 * kSmall ? c % (kSmall > 0 ? kSmall : 1) : kSmall;
      constexpr int pa = PA == 3 && PW == 3 ? (q == 0 ? 2 : q == 1 ? 0 : q == 2 ? 1 : q == 3 ? 1 : 0) : PA == 3 ? (q < 2 ? 2 - q : 0) : 0;
      constexpr int pw = PA == 3 && PW == 3 ? (q == 0 ? 0 : q == 1 ? 2 : q == 2 ? 1 : q == 3 ? 0 : q == 4 ? 1 : 0) : PW == 3 ? (q < 2 ? 2 - q : 0) : 0;
#pragma unroll
      for (int j = 0; j < NTW; ++j) acc[st][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[ks][pa], b[ks][j][pw], c == 0 ? none : acc[st][j], 0, 0, 0);
      constexpr int kP = (kPuts + kChunks - 1) / kChunks;
      for_each<kP>([&](auto i_c) { put(integral_constant<int, st ^ 1>{}, integral_constant<int, c * kP + decltype(i_c)::value>{}); });
      constexpr int kF = (16 * NTW + kChunks - 1) / kChunks;
#pragma unroll
      for (int f = c * kF; f < (c + 1) * kF; ++f)
        if (f < 16 * NTW) sum[f / 16][f % 16] += (double)(st == 0 ? -acc[1][f / 16][f % 16] : acc[0][f / 16][f % 16]);
      __builtin_amdgcn_sched_barrier(0);
    };
    for_each<kChunks>(chunk);
  };
  auto put_all = [&](auto set_c) { for_each<kPuts>([&](auto q_c) { put(set_c, q_c); }); };
  using std::integral_constant;
  const integral_constant<int, 0> c0;
  const integral_constant<int, 1> c1;
  const std::false_type whole;
  const int full = K / kFK;                                      // whole steps
  // (both: a wave without rows multiplies nothing, and after an odd number of steps what acc[0] happened to hold would count as its sums:
  // where that was no number the tile was multiplied again, and its last bits went with what had run before)
#pragma unroll
  for (int j = 0; j < NTW; ++j) acc[0][j] = acc[1][j] = none;
  if (full > 0) {
    load(c0, whole, 0);
    load(c1, whole, full > 1 ? kFK : 0);
    put_all(c0);
    __syncthreads();
    // past the last step the last one is requested and put once more, for nobody
    auto turn = [&](auto st_c, int s) {
      load(st_c, whole, min(s + 2, full - 1) * kFK);
      if (busy) step(st_c);
      else put_all(integral_constant<int, decltype(st_c)::value ^ 1>{});
      __syncthreads();
    };
    for (int s = 0; s < full; s += 2) {
      turn(c0, s);
      if (s + 1 < full) turn(c1, s + 1);
      else {
#pragma unroll
        for (int j = 0; j < NTW; ++j) acc[1][j] = -acc[0][j];
      }
    }
  }
  auto fold = [&]() {
#pragma unroll
    for (int f = 0; f < 16 * NTW; ++f) sum[f / 16][f % 16] -= (double)acc[1][f / 16][f % 16];
  };
  fold();
  if (K % kFK != 0) {                                            // (a negated step: it follows an even number of steps or the last of an odd one)
    load(c1, std::true_type{}, full * kFK);
    put_all(c1);
    load(c0, std::true_type{}, full * kFK);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NTW; ++j) acc[0][j] = none;
#pragma unroll
    for (int j = 0; j < NTW; ++j) acc[1][j] = none;
    if (busy) step(c1);
    fold();
  }
  // An infinity, a NaN, a value that rounds to infinity or one with bits below 2^-133 (from 2^-110 down) has no three bf16 parts: a tile
  // whose sums are not all finite, or that has met such bits, is multiplied again by fp32 MFMAs, whose infinities and NaNs are those of
  // the products.  (The bf16 MFMAs keep subnormal operands, products and sums: small results need nothing of the kind.)  Collecting the bits
  // costs 1 % (the layer of T = 2048 above: 258.7 -> 261.3 us).
  if constexpr (PA + PW > 2) {
    bool finite = true;
#pragma unroll
    for (int f = 0; f < 16 * NTW; ++f) finite = finite && fabs(sum[f / 16][f % 16]) <= 3.402823466e38;
    if (__syncthreads_or(!finite || bits_lost(rests))) {
      float* const af = reinterpret_cast<float*>(As);
      float* const wf = reinterpret_cast<float*>(Ws);
#pragma unroll
      for (int f = 0; f < 16 * NTW; ++f) sum[f / 16][f % 16] = 0.;
      for (int k0 = 0; k0 < K; k0 += kFK) {
        load(c0, std::true_type{}, k0);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < A_PER; ++i) *reinterpret_cast<floatx4*>(af + fswz(ar + kThreads / 8 * i, ac)) = widen4(ra[0][i]);
#pragma unroll
        for (int i = 0; i < W_PER; ++i)
          *reinterpret_cast<floatx4*>(wf + (W_KM ? (tid + kThreads * i) * 4 : fswz(ar + kThreads / 8 * i, ac))) = widen4(rw[0][i]);
        __syncthreads();
        for (int ks = 0; ks < kFK / 8; ++ks) {
          const floatx4 a = *reinterpret_cast<const floatx4*>(af + fswz(wm * 32 + l32, 2 * ks + h));
#pragma unroll
          for (int j = 0; j < NTW; ++j) {
            const int n = (wn * NTW + j) * 32 + l32;
            floatx16 t = none;
#pragma unroll
            for (int q = 0; q < 4; ++q)
              t = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q], wf[W_KM ? (8 * ks + 4 * h + q) * BN + n : fswz(n, 2 * ks + h) + q], t, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 16; ++i) sum[j][i] += (double)t[i];
          }
        }
      }
    }
  }
  if (!busy) return;
#pragma unroll
  for (int j = 0; j < NTW; ++j) {
    const int n = n0 + (wn * NTW + j) * 32 + l32;
    if (n < N) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int m = wm * 32 + acc_row(i, lane);
        if (m < rows) out[(size_t)dst_s[m] * N + n] = (float)(scale_s[m] * sum[j][i]);
      }
    }
  }
}

// Which tiles.  16-row ones (fp32 MFMAs) where experts have few rows, and where 64 x 64 tiles would leave half of the chip idle; 128 x 128
// ones where experts fill them at least by half and there is one for every CU, or for every other CU if they fill them well; else 64 x 64.
// Both products of a forward pass in us (the second and third without collected bits and turned signs, 2 to 4 % more now),
// 16 rows / 64 x 64 / 128 x 128 (and fp32 MFMAs on 64 x 64 tiles, which had these sizes before): H = 768, I = 384, E = 64: 24 rows per
// expert 66 / 73 / 107, 48: 117 / 89 / 113, 93: 181 / 140 / 123, 192: - / 233 / 239 or, on another card, 258 / 206 (311, 348);
// H = 1000, I = 504, E = 64: 16 rows 111 / 110 / 138, 64: 224 / 186 / 164, 256: - / 510 / 421 (627); H = 192, I = 88, E = 16: 96 rows
// 13 / 15 / 24, 187: - / 17 / 25 (19); H = 512, I = 256, E = 9: 56 rows 21 / 24 / 39, 222: - / 34 / 43 (45), 455: - / 52 / 47 (65).
template <typename TA, typename TW, bool W_KM, bool GATHER, bool SCATTER>
hipError_t launch_ggemm_f32(const TA* A, const int32_t* a_index, const TW* W, const int32_t* offsets, const int32_t* out_index,
                            const float* out_scale, int S, int K, int N, int E, float* out, hipStream_t s) {
  auto grid = [&](int BM, int nblk_n) {
    const long long tiles = (long long)(S / BM + E < S ? S / BM + E : S) * nblk_n;
    return dim3((unsigned)(((tiles + 7) & ~7ll) + 8));
  };
  const int nb64 = (N + 63) / 64, nb128 = (N + 127) / 128;
  if constexpr (!W_KM) {
    if ((long long)S <= 30ll * E || (long long)(S / 64 + E / 2) * nb64 <= kCUs / 2) {
      hipLaunchKernelGGL((ggemm_f32_kernel<TA, TW, GATHER, SCATTER>), grid(16, nb64), dim3(256), 0, s, A, a_index, W, offsets, out_index,
                         out_scale, K, N, E, nb64, out);
      return hipGetLastError();
    }
  }
  if ((long long)S >= 60ll * E && (long long)(S / 128 + E / 2) * nb128 >= ((long long)S >= 240ll * E ? kCUs / 2 : kCUs))
    hipLaunchKernelGGL((ggemm_split_kernel<4, 2, 2, TA, TW, W_KM, GATHER, SCATTER>), grid(128, nb128), dim3(512), 0, s, A, a_index, W,
                       offsets, out_index, out_scale, K, N, E, nb128, out);
  else
    hipLaunchKernelGGL((ggemm_split_kernel<2, 2, 1, TA, TW, W_KM, GATHER, SCATTER>), grid(64, nb64), dim3(256), 0, s, A, a_index, W,
                       offsets, out_index, out_scale, K, N, E, nb64, out);
  return hipGetLastError();
}

// dW[e][n][m] = sum over the rows r of expert e of P[srcP(r)][n] Q[srcQ(r)][m]; srcP(r) = index[r] (GATHER_P) or r, likewise
// Q.  Both operands K-major (the contraction runs over rows), in bf16 parts as above, their products in one sum.  Workgroup = WM x WN
// waves, each 32 x 32 NTW of dW.  N, M multiples of 4.  Rows past the expert's end count as zeros.
template <int WM, int WN, int NTW, typename TP, typename TQ, typename TOut, bool GATHER_P, bool GATHER_Q>
__global__ __launch_bounds__(64 * WM * WN, 2) void wgrad_split_kernel(const TP* __restrict__ P, const TQ* __restrict__ Q,
                                                                      const int32_t* __restrict__ index, const int32_t* __restrict__ offsets,
                                                                      int N, int M, int E, int nblk_n, int nblk_m, TOut* __restrict__ dW) {
  constexpr int BP = 32 * WM, BQ = 32 * NTW * WN, kThreads = 64 * WM * WN, PP = Planes<TP>::n, PQ = Planes<TQ>::n;
  constexpr int P_PER = BP * 8 / kThreads, Q_PER = BQ * 8 / kThreads;
  __shared__ __attribute__((aligned(16))) bf16_t Ps[2][PP * BP * kFK];
  __shared__ __attribute__((aligned(16))) bf16_t Qs[2][PQ * BQ * kFK];
  const int per_e = nblk_n * nblk_m;
  const int item = xcd_tile(blockIdx.x, E * per_e);
  if (item >= E * per_e) return;
  const int e = item / per_e, rest = item - e * per_e;
  const int n0 = (rest / nblk_m) * BP, m0 = (rest % nblk_m) * BQ;
  const int lo = offsets[e], hi = offsets[e + 1];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  typedef typename Planes<TP>::raw RawP;
  typedef typename Planes<TQ>::raw RawQ;
  RawP rp[2][P_PER];
  RawQ rq[2][Q_PER];
  // quadruple i of this thread: row (tid + kThreads i) / (B / 4) of the step, columns 4 ((tid + kThreads i) % (B / 4)) on
  int ip[2][P_PER], iq[2][Q_PER];                        // the rows' places in memory, looked up a step before they are read
  auto lookup = [&](auto set_c, int r0) {
    constexpr int set = decltype(set_c)::value;
#pragma unroll
    for (int i = 0; i < P_PER; ++i) {
      const int r = min(r0 + (tid + kThreads * i) / (BP / 4), hi - 1);
      ip[set][i] = GATHER_P ? index[r] : r;
    }
#pragma unroll
    for (int i = 0; i < Q_PER; ++i) {
      const int r = min(r0 + (tid + kThreads * i) / (BQ / 4), hi - 1);
      iq[set][i] = GATHER_Q ? index[r] : r;
    }
  };
  auto load = [&](auto set_c, int r0) {                  // (columns past N or M repeat the last ones and are not stored)
    constexpr int set = decltype(set_c)::value;
#pragma unroll
    for (int i = 0; i < P_PER; ++i) {
      const int g = tid + kThreads * i;
      rp[set][i] = *reinterpret_cast<const RawP*>(P + (size_t)ip[set][i] * N + min(n0 + g % (BP / 4) * 4, N - 4));
      if (r0 + g / (BP / 4) >= hi) rp[set][i] = RawP{};
    }
#pragma unroll
    for (int i = 0; i < Q_PER; ++i) {
      const int g = tid + kThreads * i;
      rq[set][i] = *reinterpret_cast<const RawQ*>(Q + (size_t)iq[set][i] * M + min(m0 + g % (BQ / 4) * 4, M - 4));
      if (r0 + g / (BQ / 4) >= hi) rq[set][i] = RawQ{};
    }
  };
  constexpr int kPuts = P_PER * PP + Q_PER * PQ;
  unsigned rests = 0;
  auto put = [&](auto set_c, auto q_c) {
    constexpr int set = decltype(set_c)::value, q = decltype(q_c)::value;
    if constexpr (q < P_PER * PP) {
      constexpr int i = q / PP, p = q % PP;
      const int g = tid + kThreads * i;
      put_plane<p, set == 1>(Ps[set] + p * (BP * kFK) + kswz<BP>(g / (BP / 4), g % (BP / 4)), rp[set][i], rests);
    } else if constexpr (q < kPuts) {
      constexpr int i = (q - P_PER * PP) / PQ, p = (q - P_PER * PP) % PQ;
      const int g = tid + kThreads * i;
      put_plane<p>(Qs[set] + p * (BQ * kFK) + kswz<BQ>(g / (BQ / 4), g % (BQ / 4)), rq[set][i], rests);
    }
  };
  const int wm = wave % WM, wn = wave / WM, l32 = lane & 31, h = lane >> 5;
  // every other step's negatives in a sum of their own, for the same reason as in ggemm_split_kernel
  floatx16 acc[2][NTW], none;
#pragma unroll
  for (int i = 0; i < 16; ++i) none[i] = 0.f;
#pragma unroll
  for (int j = 0; j < NTW; ++j) acc[0][j] = acc[1][j] = none;
  // as a step of ggemm_split_kernel, but into a running sum: 24 roundings a step where 32 FMAs would make 32
  auto step = [&](auto st_c) {
    constexpr int st = decltype(st_c)::value;
    constexpr int kProducts = PP * PQ == 9 ? 6 : PP * PQ == 3 ? 3 : 1, kChunks = 2 * kProducts;
    using std::integral_constant;
    bf16x8 a[2][PP], b[2][NTW][PQ];
    auto read = [&](int ks) {
#pragma unroll
      for (int p = 0; p < PP; ++p) a[ks][p] = kplane_frag<BP>(Ps[st] + p * (BP * kFK), lane, wm * 32, ks);
#pragma unroll
      for (int j = 0; j < NTW; ++j)
#pragma unroll
        for (int p = 0; p < PQ; ++p) b[ks][j][p] = kplane_frag<BQ>(Qs[st] + p * (BQ * kFK), lane, (wn * NTW + j) * 32, ks);
    };
    read(0);
    for_each<kChunks>([&](auto c_c) {
      constexpr int c = decltype(c_c)::value, ks = c / kProducts, q = c % kProducts;
      if constexpr (c == (kProducts > 2 ? 2 : 0)) read(1);
      constexpr int pp = PP == 3 && PQ == 3 ? (q == 0 ? 2 : q == 2 || q == 3 ? 1 : 0) : PP == 3 ? 2 - q : 0;
      constexpr int pq = PP == 3 && PQ == 3 ? (q == 1 ? 2 : q == 2 || q == 4 ? 1 : 0) : PQ == 3 ? 2 - q : 0;
#pragma unroll
      for (int j = 0; j < NTW; ++j) acc[st][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[ks][pp], b[ks][j][pq], acc[st][j], 0, 0, 0);
      constexpr int kP = (kPuts + kChunks - 1) / kChunks;
      for_each<kP>([&](auto i_c) { put(integral_constant<int, st ^ 1>{}, integral_constant<int, c * kP + decltype(i_c)::value>{}); });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  using std::integral_constant;
  const integral_constant<int, 0> c0;
  const integral_constant<int, 1> c1;
  const int nsteps = (hi - lo + kFK - 1) / kFK;
  if (nsteps > 0) {
    lookup(c0, lo);
    lookup(c1, lo + kFK);
    load(c0, lo);
    load(c1, lo + kFK);
    for_each<kPuts>([&](auto q_c) { put(c0, q_c); });
    lookup(c0, lo + 2 * kFK);
    __syncthreads();
    // rows past the end read the last one and count as zeros: past the last step as well, for nobody
    auto turn = [&](auto st_c, int s) {
      constexpr int st = decltype(st_c)::value;
      load(st_c, lo + (s + 2) * kFK);
      lookup(integral_constant<int, st ^ 1>{}, lo + (s + 3) * kFK);
      step(st_c);
      __syncthreads();
    };
    for (int s = 0; s < nsteps; s += 2) {
      turn(c0, s);
      if (s + 1 < nsteps) turn(c1, s + 1);
    }
  }
#pragma unroll
  for (int j = 0; j < NTW; ++j) acc[0][j] -= acc[1][j];
  if constexpr (PP + PQ > 2) {                           // numbers without three parts, as in ggemm_split_kernel
    bool finite = true;
#pragma unroll
    for (int j = 0; j < NTW; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) finite = finite && fabsf(acc[0][j][i]) <= 3.402823466e38f;
    if (__syncthreads_or(!finite || bits_lost(rests))) {
      float* const pf = reinterpret_cast<float*>(Ps);
      float* const qf = reinterpret_cast<float*>(Qs);
#pragma unroll
      for (int j = 0; j < NTW; ++j) acc[0][j] = none;
      for (int r0 = lo; r0 < hi; r0 += kFK) {
        lookup(c0, r0);
        load(c0, r0);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < P_PER; ++i) *reinterpret_cast<floatx4*>(pf + (tid + kThreads * i) * 4) = widen4(rp[0][i]);
#pragma unroll
        for (int i = 0; i < Q_PER; ++i) *reinterpret_cast<floatx4*>(qf + (tid + kThreads * i) * 4) = widen4(rq[0][i]);
        __syncthreads();
        for (int k = 0; k < kFK; k += 2)
#pragma unroll
          for (int j = 0; j < NTW; ++j)
            acc[0][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(pf[(k + h) * BP + wm * 32 + l32], qf[(k + h) * BQ + (wn * NTW + j) * 32 + l32],
                                                             acc[0][j], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < NTW; ++j) {
    const int m = m0 + (wn * NTW + j) * 32 + l32;
    if (m < M) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int n = n0 + wm * 32 + acc_row(i, lane);
        if (n < N) dW[((size_t)e * N + n) * M + m] = from_float<TOut>(acc[0][j][i]);
      }
    }
  }
}

template <typename TP, typename TQ, typename TOut, bool GATHER_P, bool GATHER_Q>
hipError_t launch_wgrad_f32(const TP* P, const TQ* Q, const int32_t* index, const int32_t* offsets, int N, int M, int E, TOut* dW,
                            hipStream_t s) {
  auto blocks = [](int n, int b) { return (n + b - 1) / b; };
  auto grid = [&](int b) { return dim3((unsigned)((E * blocks(N, b) * blocks(M, b) + 7) & ~7)); };
  if (E * blocks(N, 128) * blocks(M, 128) >= kCUs / 2)
    hipLaunchKernelGGL((wgrad_split_kernel<4, 2, 2, TP, TQ, TOut, GATHER_P, GATHER_Q>), grid(128), dim3(512), 0, s, P, Q, index, offsets,
                       N, M, E, blocks(N, 128), blocks(M, 128), dW);
  else
    hipLaunchKernelGGL((wgrad_split_kernel<2, 2, 1, TP, TQ, TOut, GATHER_P, GATHER_Q>), grid(64), dim3(256), 0, s, P, Q, index, offsets,
                       N, M, E, blocks(N, 64), blocks(M, 64), dW);
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
