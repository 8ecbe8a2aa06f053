// Attention of the 10-layer experimental forward (BiBoAttention.forward, src/modeling/attn/base.py:55-128 without cache):
// QK-norm and RoPE in place on the rows of one q|k|v projection, and causal or banded attention with the XSA correction
// (attn/xsa.py:41-54) in its epilogue, written token-major for the output projection.  bf16 operands, fp32 arithmetic.
#include "stripe.h"

namespace bibo {
namespace {

__device__ __forceinline__ float row16_sum(float v) {      // sum over a DPP row of 16 lanes, the same in every lane
  auto dpp = [](float x, auto ctrl) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, false));
  };
  v += dpp(v, std::integral_constant<int, 0xB1>{});
  v += dpp(v, std::integral_constant<int, 0x4E>{});
  v += dpp(v, std::integral_constant<int, 0x141>{});
  return v + dpp(v, std::integral_constant<int, 0x140>{});
}

// ---- QK-norm (norm.py:19-24 on head rows) and RoPE (attn/rope.py, rotate-half), in place --------------------------
// rows of qkv: [T, ld], the nq query heads first, then the nkv key heads, D elements each; heads [first, nq + nkv).  Sixteen lanes per head row; lane
// c < D / 16 owns elements 8c .. 8c + 7 of the first half and of the second half, i.e. whole rotation pairs.  Memory-bound:
// one read and one write of the columns (in front of attention_kernel from kQueryElems on only the keys': it takes the queries on their way).  qw, kw: [D], or NULL: no norm; cos, sin: rows of D / 2 at stride ld_rope, or NULL.
template <int D>
__global__ __launch_bounds__(256) void qk_norm_rope_kernel(bf16_t* __restrict__ qkv, int ld, int T, int S, int first, int nq, int nkv,
                                                           Vec qw, Vec kw, float eps, Vec cos, Vec sin, int ld_rope) {
  constexpr int kLanes = D / 16;
  const int heads = nq + nkv - first;
  const long long g = ((long long)blockIdx.x * 256 + threadIdx.x) >> 4;
  if (g >= (long long)T * heads) return;                   // whole groups of 16 lanes
  const int t = (int)(g / heads), hd = first + (int)(g - (long long)t * heads);
  const int c = threadIdx.x & 15;
  const bool live = c < kLanes;
  bf16_t* row = qkv + (size_t)t * ld + hd * D;
  float a[8], b[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) a[q] = b[q] = 0.f;
  if (live) {
    const bf16x8 va = *reinterpret_cast<const bf16x8*>(row + c * 8), vb = *reinterpret_cast<const bf16x8*>(row + D / 2 + c * 8);
#pragma unroll
    for (int q = 0; q < 8; ++q) { a[q] = (float)va[q]; b[q] = (float)vb[q]; }
  }
  const Vec w = hd < nq ? qw : kw;
  if (w.p != nullptr) {
    float ss = 0.f;
#pragma unroll
    for (int q = 0; q < 8; ++q) ss = fmaf(a[q], a[q], fmaf(b[q], b[q], ss));
    const float rinv = rsqrtf(row16_sum(ss) / (float)D + eps);
    if (live) {
      float wa[8], wb[8];
      load8(w, c * 8, wa);
      load8(w, D / 2 + c * 8, wb);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        a[q] = wa[q] * (float)(bf16_t)(a[q] * rinv);
        b[q] = wb[q] * (float)(bf16_t)(b[q] * rinv);
      }
    }
  }
  if (!live || (w.p == nullptr && cos.p == nullptr)) return;
  if (cos.p != nullptr) {
    const size_t p = (size_t)(t % S) * ld_rope + c * 8;
    float co[8], si[8];
    load8(cos, p, co);
    load8(sin, p, si);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float x = a[q], y = b[q];
      a[q] = x * co[q] - y * si[q];
      b[q] = y * co[q] + x * si[q];
    }
  }
  bf16x8 oa, ob;
#pragma unroll
  for (int q = 0; q < 8; ++q) { oa[q] = (bf16_t)a[q]; ob[q] = (bf16_t)b[q]; }
  *reinterpret_cast<bf16x8*>(row + c * 8) = oa;
  *reinterpret_cast<bf16x8*>(row + D / 2 + c * 8) = ob;
}

// cos and sin of position * inv_freq, bf16 [S, 2 half], both halves of a row alike (embed.py:63-74): one launch for what is
// nine as tensor operations, of 2 to 5 us each.
__global__ __launch_bounds__(256) void rope_tables_kernel(Vec inv_freq, int S, int half, bf16_t* __restrict__ cos_t,
                                                          bf16_t* __restrict__ sin_t) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long long)S * half) return;
  const int s = (int)(i / half), c = (int)(i - (long long)s * half);
  const float ang = (float)s * inv_freq[c];
  const size_t at = (size_t)s * 2 * half + c;
  cos_t[at] = cos_t[at + half] = (bf16_t)cosf(ang);
  sin_t[at] = sin_t[at + half] = (bf16_t)sinf(ang);
}

// ---- attention -------------------------------------------------------------------------------------------------
// One workgroup = four waves; a wave owns 32 consecutive queries of one head, and 1, 2 or 4 query heads that share a key
// head share the workgroup (hpw), so that a block of 32 keys and values passes through LDS once for all of them.
//   S^T = K Q^T  (v_mfma_f32_32x32x16_bf16, Q fragments in registers): lane = query, registers = keys, so a row's maximum
//     and sum are in-lane but for the other half of the keys in lane ^ 32;
//   O^T = V^T P^T: the probabilities a lane holds (keys 4h .. +4 and 8 + 4h .. +4 of sixteen) are, rounded to bf16, the MFMA
//     operand as they are, with V's operand read in the same key order by transposing LDS reads; O^T has lane = query
//     again, so rescaling and the final division are per-lane scalars.
// FINE (banded layers): a probability goes in as two bf16 parts, its rounding and what that left, so that it keeps 16 bits of
// mantissa; the tensor operations these layers ran before multiplied their probabilities in fp32.  Against float64 both are off by
// what the rounding of the output to bf16 takes, to five digits (1.6433e-3 in the 2-norm at S = 2048, D = 192, window 128; with XSA
// 1.661e-3 here and 2.349e-3 there).  Causal layers' library kernel rounded them to bf16, as the other variant does.
// The running maximum is raised (and O rescaled, D/32 x 16 multiplies) only when a row's maximum passes it by more than 8
// in log2 units: the sums stay exact, the probabilities at most 256.
// K and V blocks arrive by LDS-DMA in three stages, requested two blocks ahead right after the barrier that frees the stage, by transfers that the
// compiler does not see: it waited for all of them in front of the values' reads, that is for the block behind the present one.  A wave's chain
// of a block (12 dependent MFMAs, maximum, 16 exponentials, 12 MFMAs) bounds the causal layers, whose last queries take 64 of them: six key
// fragments are read in front of the first MFMA, and the masks select instead of branching.  Two stages, reads in pairs -> now, us,
// D = 192, 4 and 2 heads, S = 2048: causal 8 x 83.9 -> 74.7, 1 x 65.3 -> 60.4, window 128 8 x 31.8 -> 30.9, 1 x 17.6 -> 15.9; D = 128, 8 and 2
// heads, 4 x 1024 35.9 -> 30.8.  Tried: a block's scores beside the block before's exponentials (registers; reads next to their use: 89.5).
// 16-byte granule g of a K row r sits at g ^ swz, so the 16 rows of a fragment read hit distinct banks; V rows are
// swizzled so that the four rows of a transposing read do.
// Two workgroups per CU (D = 192: 72 KB of LDS, 96 accumulator and 48 query registers per lane): one's softmax runs beside the
// other's MFMAs.  Causal blocks are dealt longest first, then shortest first, so that the two of a CU add up alike.
typedef short attn_v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) attn_v4i16 attn_lds_v4i16;

template <int D> __device__ __forceinline__ int kswz(int row) { return D == 128 ? (row & 15) : ((row >> 1) & 7); }
template <int D> __device__ __forceinline__ int vswz(int row) { return D == 128 ? ((row & 3) << 2) : (((row >> 1) & 1) << 2); }

constexpr int kAttnStages = 3;

// QK-norm and RoPE of the queries, as in qk_norm_rope_kernel; weight, cos, sin may be NULL
struct QueryNorm {
  Vec weight;
  float eps;
  Vec cos, sin;
  int ld_rope;
};

// The fragments of row `pos` of a head: the half-waves h of lane n hold granules 2 s + h.  The same sums in the same order as in
// qk_norm_rope_kernel, whose lane c holds granules c and c + D / 16, hence the same bits.  In place they
// are read and written once more, here they lengthen the chain in front of a wave's first product.  Both launches, us, queries in place / here,
// 4 and 2 heads of 192, causal with norm and window 128 with norm and RoPE: T = 16384: 88.1 / 80.4 and 47.6 / 44.0; 8192: 76.8 / 71.6 and 32.2 /
// 30.3; 4096: 71.6 / 70.2 and 26.8 / 26.5; 2048: 67.0 / 67.8 and 22.7 / 24.4; 128: 15.1 / 18.2.  Hence kQueryElems, the 4096 tokens of these.
// Other heads, as long a call or longer, causal and window 128, 8 x 2048 tokens: 64 wide, 8 and 2: 65.4 / 54.6 and 39.3 / 27.7, 32 and 8: 231 / 185 and
// 122 / 79; 128 wide, 2 and 2: 61.8 / 58.6 and 28.5 / 26.4, 32 and 8: 363 / 326 and 188 / 148.  Of 84 such calls the longest on this side of
// the line is one sequence of 8192 in a window, 192 wide, 2 and 2 heads: 27.5 / 29.4.
// weights(s, first half's 8, second half's 8), tables(s, cos, sin): of granule 2 s + h.
template <int KS, typename Weights, typename Tables>
__device__ __forceinline__ void norm_rope_query(const QueryNorm& nr, bf16x8 (&q)[KS], Weights weights, Tables tables) {
  constexpr int KH = KS / 2, D = 16 * KS;
  float rinv = 0.f;
  if (nr.weight.p != nullptr) {
    float t[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KH; ++s) {
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float a = (float)q[s][e], b = (float)q[s + KH][e];
        ss = fmaf(a, a, fmaf(b, b, ss));
      }
      const Pair p = lanes32(ss);
      t[s] = p.a + p.b;
    }
    rinv = rsqrtf((((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]))) / (float)D + nr.eps);
  }
#pragma unroll
  for (int s = 0; s < KH; ++s) {
    float a[8], b[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) { a[e] = (float)q[s][e]; b[e] = (float)q[s + KH][e]; }
    if (nr.weight.p != nullptr) {
      float wa[8], wb[8];
      weights(s, wa, wb);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        a[e] = wa[e] * (float)(bf16_t)(a[e] * rinv);
        b[e] = wb[e] * (float)(bf16_t)(b[e] * rinv);
      }
    }
    if (nr.cos.p != nullptr) {
      float co[8], si[8];
      tables(s, co, si);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = a[e], y = b[e];
        a[e] = x * co[e] - y * si[e];
        b[e] = y * co[e] + x * si[e];
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) { q[s][e] = (bf16_t)a[e]; q[s + KH][e] = (bf16_t)b[e]; }
  }
}

// A lane of half h keeps elements 4 h .. 4 h + 3 of every granule of its row, but loads and stores whole granules, two of which, 2 j + h, lie in its
// row's two lanes: first halves of (lower lane's, upper lane's) granule <-> half h of granules 2 j and 2 j + 1, in both directions.  Twelve accesses a
// row of 192 instead of 24 of 8 bytes: with XSA, S = 2048, 4 and 2 heads of 192, us: window 128 8 x 30.9 -> 26.8, 1 x 15.9 -> 14.8; causal 8 x
// 74.7 -> 73.7; window 1, which is little but the rows, 23.1 -> 18.5.
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
struct Granules { unsigned a[2], b[2]; };
__device__ __forceinline__ Granules swap_halves(u32x4 v) {
  const auto x = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false), y = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
  return {{(unsigned)x[0], (unsigned)y[0]}, {(unsigned)x[1], (unsigned)y[1]}};
}

// FAR: rows further apart than kAttnNearLd, by 64-bit addresses.
template <int D, bool FINE, bool FAR>
__global__ __launch_bounds__(256, 2) void attention_kernel(const bf16_t* __restrict__ qkv, int ld, int S, int nq, int nkv, int hpw,
                                                           int heads, int nqb, int window, float scale_log2,
                                                           Vec xsa_alpha, QueryNorm nr, bf16_t* __restrict__ out) {
  constexpr int KB = 32, GPR = D / 8, NI = KB * GPR / 256;      // keys per block, granules per row, DMA instructions per operand
  constexpr int DT = D / 32, KS = D / 16;
  static_assert(KB * GPR % 256 == 0, "a block does not divide over the threads");
  __shared__ __attribute__((aligned(16))) bf16_t K[kAttnStages][KB * D];
  __shared__ __attribute__((aligned(16))) bf16_t V[kAttnStages][KB * D];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  // block id -> (query block, group of hpw query heads of one batch); heads = groups over all batches
  const int r = blockIdx.x / heads, grp = blockIdx.x - r * heads;
  const int qb = r < nqb / 2 ? nqb - 1 - r : r - nqb / 2;
  const int gpb = nq / hpw;                                     // groups per batch
  const int b = grp / gpb, gi = grp - b * gpb;
  const int wph = 4 / hpw;                                      // waves per head
  const int head = gi * hpw + wave / wph;
  const int kvh = gi * hpw / (nq / nkv);
  const int QB = 32 * wph;
  const int q0 = qb * QB, q0w = q0 + (wave % wph) * 32;         // the workgroup's and this wave's first query
  const bf16_t* base = qkv + (size_t)b * S * ld;
  const bf16_t* kbase = base + (size_t)(nq + kvh) * D;
  const bf16_t* vbase = base + (size_t)(nq + nkv + kvh) * D;

  bf16x8 q[KS];
  {
    const bf16_t* qrow = base + (size_t)min(q0w + n, S - 1) * ld + head * D + h * 8;
#pragma unroll
    for (int s = 0; s < KS; ++s) q[s] = *reinterpret_cast<const bf16x8*>(qrow + s * 16);
  }
  const unsigned row_bytes = (unsigned)ld * (unsigned)sizeof(bf16_t);
  unsigned koff[NI], voff[NI];                                  // this thread's granules of a block, in bytes from its first row
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int p = i * 256 + tid, row = p / GPR, pos = p - row * GPR;
    koff[i] = row * row_bytes + (pos ^ kswz<D>(row)) * 16;
    voff[i] = row * row_bytes + (pos ^ vswz<D>(row)) * 16;
  }
  // keys [kv0, kv0 + KB) into a stage; rows past the last one lie past the descriptor's end and read as zeros
  auto request = [&](int kv0, auto stage_c) __attribute__((always_inline)) {
    constexpr int st = decltype(stage_c)::value;
    if constexpr (FAR) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int p = i * 256 + tid, row = p / GPR, pos = p - row * GPR;
        const size_t o = (size_t)min(kv0 + row, S - 1) * ld;
        dma16(kbase + o + (pos ^ kswz<D>(row)) * 8, K[st] + (i * 256 + wave * 64) * 8);
        dma16(vbase + o + (pos ^ vswz<D>(row)) * 8, V[st] + (i * 256 + wave * 64) * 8);
      }
      return;
    }
    const unsigned long long left = (unsigned long long)(S - kv0) * row_bytes;
    const unsigned bytes = left < 0xffffffffull ? (unsigned)left : 0xffffffffu;
    const i32x4 kd = make_words(kbase + (size_t)kv0 * ld, bytes), vd = make_words(vbase + (size_t)kv0 * ld, bytes);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      dma16_unseen(kd, koff[i], 0, lds_address(K[st]) + (i * 256 + wave * 64) * 16);
      dma16_unseen(vd, voff[i], 0, lds_address(V[st]) + (i * 256 + wave * 64) * 16);
    }
  };
  const int kv_first = window > 0 ? max(0, (q0 - window + 1)) & ~(KB - 1) : 0;
  const int kv_end = min(q0 + QB, S);                           // keys [kv_first, kv_end)
  using std::integral_constant;
  request(kv_first, integral_constant<int, 0>{});
  if (kv_first + KB < kv_end) request(kv_first + KB, integral_constant<int, 1>{});
  // the tables of this lane's granules, requested with the queries (bf16 ones; load by load behind them it all took 8 us)
  constexpr int KH = KS / 2;
  const int pos = min(q0w + n, S - 1);
  const bool fetched = (nr.weight.p == nullptr || nr.weight.bf16) && (nr.cos.p == nullptr || (nr.cos.bf16 && nr.sin.bf16));
  const size_t at = (size_t)pos * nr.ld_rope + h * 8;
  bf16x8 ct[KH], sn[KH];
  if (fetched && nr.cos.p != nullptr)
#pragma unroll
    for (int s = 0; s < KH; ++s) {
      ct[s] = *reinterpret_cast<const bf16x8*>(static_cast<const bf16_t*>(nr.cos.p) + at + s * 16);
      sn[s] = *reinterpret_cast<const bf16x8*>(static_cast<const bf16_t*>(nr.sin.p) + at + s * 16);
    }
#pragma unroll
  for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(q[s]));   // q has arrived: a wait in the loop, where the compiler cannot know, would be for all transfers
  if (nr.weight.p != nullptr || nr.cos.p != nullptr) {
    auto widen = [](bf16x8 v, float (&to)[8]) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < 8; ++e) to[e] = (float)v[e];
    };
    if (fetched) {
      bf16x8 wt[KS];
      if (nr.weight.p != nullptr)
#pragma unroll
        for (int s = 0; s < KS; ++s) wt[s] = *reinterpret_cast<const bf16x8*>(static_cast<const bf16_t*>(nr.weight.p) + s * 16 + h * 8);
      norm_rope_query<KS>(nr, q, [&](int s, float (&a)[8], float (&b)[8]) __attribute__((always_inline)) { widen(wt[s], a); widen(wt[s + KH], b); },
                          [&](int s, float (&c)[8], float (&d)[8]) __attribute__((always_inline)) { widen(ct[s], c); widen(sn[s], d); });
    } else
      norm_rope_query<KS>(nr, q,
                          [&](int s, float (&a)[8], float (&b)[8]) __attribute__((always_inline)) {
                            load8(nr.weight, s * 16 + h * 8, a);
                            load8(nr.weight, D / 2 + s * 16 + h * 8, b);
                          },
                          [&](int s, float (&c)[8], float (&d)[8]) __attribute__((always_inline)) {
                            load8(nr.cos, at + s * 16, c);
                            load8(nr.sin, at + s * 16, d);
                          });
  }
  floatx16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
  float m = -1.0e30f, l = 0.f;                                  // running maximum (log2 units) and this lane's part of the sum
  // V operand: lane r16 of a 16-lane group points at key 4h + r16 / 4, columns 16 ((lane >> 4) & 1) + 4 (r16 % 4)
  const int r16 = lane & 15;
  const int vkey = 4 * h + (r16 >> 2), vcol = 16 * ((lane >> 4) & 1) + 4 * (r16 & 3);
  const int vsw = vswz<D>(r16 >> 2);                            // the same for every key this lane reads (keys = r16 / 4 mod 4)
  const int ksw = kswz<D>(n);

  auto block = [&](int kv0, const bf16_t* ks, const bf16_t* vs) __attribute__((always_inline)) {
    // nothing of this block is visible to this wave's queries?
    if (kv0 > q0w + 31 || (window > 0 && kv0 + KB - 1 <= q0w - window)) return;
    floatx16 st;
#pragma unroll
    for (int i = 0; i < 16; ++i) st[i] = 0.f;
    // (left to itself the compiler reads two fragments at a time and waits for them)
    constexpr int kAhead = KS < 6 ? KS : 6;
    bf16x8 kf[KS];
    auto kread = [&](int s) __attribute__((always_inline)) { kf[s] = *reinterpret_cast<const bf16x8*>(ks + n * D + (((2 * s + h) ^ ksw) << 3)); };
#pragma unroll
    for (int s = 0; s < kAhead; ++s) kread(s);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s], q[s], st, 0, 0, 0);
      if (s + kAhead < KS) kread(s + kAhead);
      __builtin_amdgcn_sched_barrier(0);
    }
    // register i: key kv0 + 8 (i / 4) + 4 h + i % 4
    if (kv0 + KB - 1 > q0w || (window > 0 && q0w + 31 - kv0 >= window)) {
      const int past = q0w + n - kv0 - 4 * h;                     // key 8 (i / 4) + i % 4 is seen from here on and up to `window` - 1 before
      const unsigned seen = window > 0 ? window : 0x80000000u;
#pragma unroll
      for (int i = 0; i < 16; ++i) st[i] = (unsigned)(past - (8 * (i >> 2) + (i & 3))) < seen ? st[i] : -INFINITY;
    }
    float mx = st[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, st[i]);
    const Pair mxs = lanes32(mx);
    mx = fmaxf(mxs.a, mxs.b) * scale_log2;
    if (__any(mx > m + 8.f)) {
      const float mn = fmaxf(m, mx), al = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= al;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= al;
    }
    bf16x8 p[2], pf[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float e = __builtin_amdgcn_exp2f(fmaf(st[i], scale_log2, -m));
      l += e;
      p[i >> 3][i & 7] = (bf16_t)e;
      if constexpr (FINE) pf[i >> 3][i & 7] = (bf16_t)(e - (float)p[i >> 3][i & 7]);
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const int gcol = dt * 32 + vcol;
        const bf16_t* a = vs + (16 * kk + vkey) * D + (((gcol >> 3) ^ vsw) << 3) + (gcol & 4);
        const attn_v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((attn_lds_v4i16*)a);
        const attn_v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((attn_lds_v4i16*)(a + 8 * D));
        typedef short v8i16 __attribute__((ext_vector_type(8)));
        const v8i16 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, v), p[kk], o[dt], 0, 0, 0);
        if constexpr (FINE) o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, v), pf[kk], o[dt], 0, 0, 0);
      }
  };
  // block kv0 has landed in every wave, nobody reads the stage of the block before it any more, and the block behind it may be on its way
  auto turn = [&](int kv0, auto stage_c) __attribute__((always_inline)) {
    constexpr int st = decltype(stage_c)::value;
    if (kv0 + KB < kv_end) meet_waves<2 * NI>();
    else meet_waves<0>();
    if (kv0 + 2 * KB < kv_end) request(kv0 + 2 * KB, integral_constant<int, (st + 2) % kAttnStages>{});
    block(kv0, K[st], V[st]);
  };
  for (int kv0 = kv_first; kv0 < kv_end; kv0 += kAttnStages * KB) {
    turn(kv0, integral_constant<int, 0>{});
    if (kv0 + KB < kv_end) turn(kv0 + KB, integral_constant<int, 1>{});
    if (kv0 + 2 * KB < kv_end) turn(kv0 + 2 * KB, integral_constant<int, 2>{});
  }
  // y = O / l, then XSA: y -= tanh(alpha) <y, vn> vn with vn = v / |v| of the query's own token
  const int qi = q0w + n;
  const Pair ls = lanes32(l);
  l = ls.a + ls.b;
  const float inv = 1.f / l;
  if (xsa_alpha.p != nullptr) {
    const bf16_t* vrow = vbase + (size_t)min(qi, S - 1) * ld + 8 * h;
    bf16x4 v[DT][4];
    float vv = 0.f, yv = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int c = 0; c < 4; c += 2) {
        const Granules g = swap_halves(*reinterpret_cast<const u32x4*>(vrow + dt * 32 + c * 8));
        v[dt][c] = __builtin_bit_cast(bf16x4, u32x2{g.a[0], g.a[1]});
        v[dt][c + 1] = __builtin_bit_cast(bf16x4, u32x2{g.b[0], g.b[1]});
      }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float f = (float)v[dt][i >> 2][i & 3];
        o[dt][i] *= inv;
        vv = fmaf(f, f, vv);
        yv = fmaf(f, o[dt][i], yv);
      }
    const Pair vvs = lanes32(vv), yvs = lanes32(yv);
    vv = vvs.a + vvs.b;
    yv = yvs.a + yvs.b;
    const float vn = 1.f / fmaxf(sqrtf(vv), 1e-12f);            // F.normalize
    const float coeff = yv * vn * vn * tanhf(xsa_alpha[head]);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[dt][i] = fmaf(-coeff, (float)v[dt][i >> 2][i & 3], o[dt][i]);
  } else {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[dt][i] *= inv;
  }
  bf16_t* orow = out + ((size_t)b * S + min(qi, S - 1)) * nq * D + head * D + 8 * h;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int c = 0; c < 4; c += 2) {
      auto half = [&](int f) __attribute__((always_inline)) {
        return __builtin_bit_cast(u32x2, bf16x4{(bf16_t)o[dt][f], (bf16_t)o[dt][f + 1], (bf16_t)o[dt][f + 2], (bf16_t)o[dt][f + 3]});
      };
      const u32x2 x = half(4 * c), y = half(4 * c + 4);
      const Granules g = swap_halves(u32x4{x[0], x[1], y[0], y[1]});
      if (qi < S) *reinterpret_cast<u32x4*>(orow + dt * 32 + c * 8) = u32x4{g.a[0], g.a[1], g.b[0], g.b[1]};
    }
}

}  // namespace

bool exp_attention_supported(int nq, int nkv, int D) {
  const int g = nkv > 0 ? nq / nkv : 0;
  return (D == 64 || D == 128 || D == 192) && nkv >= 1 && nq % nkv == 0 && (g == 1 || g % 2 == 0);
}

hipError_t launch_qk_norm_rope(void* qkv, int ld, int T, int S, int nq, int nkv, int D, Vec qw, Vec kw, float eps, Vec cos, Vec sin,
                               int ld_rope, bool keys_only, hipStream_t s) {
  const int first = keys_only ? nq : 0;
  const long long groups = (long long)T * (nq + nkv - first);
  if (groups == 0) return hipSuccess;
  const dim3 grid((unsigned)((groups + 15) / 16));
  bf16_t* p = static_cast<bf16_t*>(qkv);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, p, ld, T, S, first, nq, nkv, qw, kw, eps, cos, sin, ld_rope);
  };
  switch (D) {
    case 64: launch(qk_norm_rope_kernel<64>); break;
    case 128: launch(qk_norm_rope_kernel<128>); break;
    case 192: launch(qk_norm_rope_kernel<192>); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_rope_tables(Vec inv_freq, int S, int half, void* cos, void* sin, hipStream_t s) {
  const long long n = (long long)S * half;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(rope_tables_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, inv_freq, S, half,
                     static_cast<bf16_t*>(cos), static_cast<bf16_t*>(sin));
  return hipGetLastError();
}

hipError_t launch_exp_attention(const void* qkv, int ld, int B, int S, int nq, int nkv, int D, int window, float scale,
                                Vec xsa_alpha, Vec qw, float eps, Vec cos, Vec sin, int ld_rope, void* out, hipStream_t s) {
  if (B == 0 || S == 0) return hipSuccess;
  const int g = nq / nkv;
  const int hpw = g % 4 == 0 ? 4 : (g % 2 == 0 ? 2 : 1);
  const int QB = 128 / hpw, nqb = (S + QB - 1) / QB, heads = B * nq / hpw;
  const dim3 grid((unsigned)(heads * nqb));
  const float sl = scale * 1.4426950408889634f;
  const bf16_t* p = static_cast<const bf16_t*>(qkv);
  bf16_t* o = static_cast<bf16_t*>(out);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, p, ld, S, nq, nkv, hpw, heads, nqb, window, sl, xsa_alpha, QueryNorm{qw, eps, cos, sin, ld_rope}, o);
  };
  auto pick = [&](auto d) {
    constexpr int HD = decltype(d)::value;
    if (ld > kAttnNearLd) {
      if (window > 0) launch(attention_kernel<HD, true, true>); else launch(attention_kernel<HD, false, true>);
    } else {
      if (window > 0) launch(attention_kernel<HD, true, false>); else launch(attention_kernel<HD, false, false>);
    }
  };
  switch (D) {
    case 64: pick(std::integral_constant<int, 64>{}); break;
    case 128: pick(std::integral_constant<int, 128>{}); break;
    case 192: pick(std::integral_constant<int, 192>{}); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace bibo
