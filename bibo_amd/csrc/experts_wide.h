// Kernels 3 and 4 in one launch at I = 512, for calls whose permutation a launch of its own writes (launch_fused_nt has the rule): a workgroup
// takes up to 64 permuted rows of one expert through the gate/up projection, Radial NormSiLU and the down projection without the
// activations leaving the CU.  The same tiles, requests and layout of the activations as experts_fused_kernel, with the instructions of both
// products in an order of their own.  What bounds it: the weights of an expert, which every 64 of its rows pull through a CU, and the matrix
// pipes beside them.  H = 1024, E = 64, k = 8, layer, experts_fused_kernel -> this one: 145.6 -> 137.5 us (T = 3001), 264 -> 245 (6000), 582 -> 551
// (16,000); on other cards 263.7 -> 253.1 and 274 -> 257 (6000), 592 -> 568 and 574 -> 541 (16,000), and between 150.0 -> 143.6 and 140.4 -> 139.3 (3001).
//
// Phase 1 (gate/up GEMM, 2 x 4 waves, v_mfma_f32_16x16x32_bf16, operands swapped so that a lane ends up with
// one ROW's values) walks K in steps of 64 elements, so every row an LDS-DMA instruction fetches is a whole
// 128-byte line.  A step is cut into four sub-steps of 256 weight rows: sub-step t holds, for each of the four N waves, its t-th 32-column
// gate tile and the up tile of the same columns.  The 32 KB stages form a ring of three, the x rows of a step have two
// buffers of their own.  A wave keeps the x fragments of a step in registers for all its sub-steps.
// Phase 2 turns the accumulators into bf16 activations and parks them in the stages, whose contents are dead by
// then, as an operand of the second GEMM: slice t holds columns [128t, 128t+128) of all 64 rows; row r keeps
// 16-byte granule c at position c ^ (r & 15).
// Phase 3 has no barriers and no LDS traffic for the weights: the eight waves split a block of 128*CT
// output columns (16*CT each), every wave multiplies ALL 64 resident rows with v_mfma_f32_16x16x32_bf16
// and pulls its own w_down rows straight from global memory into registers, one to two blocks of 128 K elements
// ahead (DownWeights).  Each block of columns is scaled by the routing weight and leaves in slot order through the wave's own part of the
// dead x buffers: a wave's run of 32*CT bytes per row, and no barrier, so that one wave's output runs beside the others' MFMAs.
// M wave wm multiplies 32-row block wm of a tile; a block without rows is not multiplied: the kernel body exists once for one block and
// once for two; every wave still issues its share of the weight requests, which is most of what a tile costs.
// (At I <= 384, with tiles of 128 rows, the same order gave 0 to 4 % on one card and took 0 to 5 % longer on another, and 1 to 2 us longer on
// low tiles on both.)
// Reference: BiBoFusedExperts.forward, src/modeling/ffn/moe.py:81-93.
#pragma once

#include <type_traits>

#include "experts_fused_launch.h"
#include "stripe.h"

namespace bibo {
namespace {

template <int CT>
struct WideShape {
  static constexpr int NT = 4, I = 128 * NT, BM = 64, BK = 64;
  static constexpr int BN2 = 128 * CT;                             // output columns per block: 8 waves x CT x 16
  static constexpr int kRing = 3;                                  // weight stages in LDS
  static constexpr int kXRing = 2;                                 // x buffers
  static constexpr int kActs = 4;                                  // activation fragments in flight in phase 3
  static constexpr int kStageRows = 256;                           // 4 N waves x (gate tile + up tile) x 32 rows
  static constexpr int kStageElems = kStageRows * BK;              // 32 KB = two [64][128] slices of the activations
  static constexpr int kAElems = BM * BK;                          // x rows of one K step
  static constexpr int kOutElems = BM * BN2;
  static constexpr int kXElems = kXRing * kAElems > kOutElems ? kXRing * kAElems : kOutElems;   // serve as either
  static constexpr int kBInstr = kStageRows * (BK / 8) / 512;      // load instructions per thread and weight stage
  static constexpr int kAInstr = BM * (BK / 8) / 512;              // and per x stage
  static_assert(kBInstr == 4 && kAInstr == 1, "stage does not divide over the threads");
  static_assert(NT * BM * 128 <= kRing * kStageElems, "the activations lie in the stages");
};

// a lane's offset that lies past the descriptor's end whatever is in range of it is added: reads zeros
__device__ __forceinline__ unsigned past_end(i32x4 words) { return (unsigned)words[2]; }

// The w_down rows of a wave's 16*CT output columns in blocks of 128 K elements, on their way from memory order to MFMA operand order.  A
// load gives each quad of lanes (a = lane / 16, b = lane / 4 % 4) 64 contiguous bytes, segment k_segment(a) of row 4 b + i in load i: the
// texture unit merges adjacent lanes only, and rows 16 lanes apart, as in the operand layout, move less than half the bytes per second.  Four
// loads are 4 x 4 pieces of 16 bytes in a quad, load by lane; transposed within the quad, lane c holds pieces 0 .. 3 of its segment of row
// 4 b + c: the operands of four MFMAs, register by register, whose K group a is piece m of that segment.  Two steps of v_mov_dpp and
// v_cndmask a register: the VALU has the time, while the ds_bpermute_b32 of experts_fused_kernel take 6 cycles of the LDS each, half again
// what the reads of the activations beside them take.
// Which segment: a 16-byte LDS read is served 16 lanes at a time: lanes 0-3, 12-15, 20-27 together, then 4-11, 16-19, 28-31, and the other half
// alike.  With granule c of activation row r at c ^ r the rows of lanes 0-15 and 16-31 fall on the same banks when their segments differ
// in one bit, and on different ones when they differ in both: 8 cycles a read with segment a, 4 with this one.
__device__ __forceinline__ int k_segment(int a) { return (a & 1) << 1 | ((a ^ a >> 1) & 1); }

template <int I, int CT>
struct DownWeights {
  static constexpr int KB = I / 128;                        // blocks of a column block
  typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
  u32x4_t w[2][CT][4];
  i32x4 words;                                              // this expert's w_down
  unsigned voff;                                            // byte offset of this lane's first piece
  unsigned base;                                            // byte offset of this wave's first row (uniform)
  bool odd1, odd2;                                          // bits of the lane's place in its quad

  __device__ __forceinline__ void init(const bf16_t* wd_e, int H, int first_row, int lane) {
    words = make_words(wd_e, (unsigned)H * I * sizeof(bf16_t));
    voff = (((lane >> 2) & 3) * 4 * I + k_segment(lane >> 4) * 32 + (lane & 3) * 8) * (unsigned)sizeof(bf16_t);
    base = (unsigned)first_row * I * (unsigned)sizeof(bf16_t);
    odd1 = lane & 1;
    odd2 = lane & 2;
  }
  // load i of block kb of the rows `rows_on` behind the first ones; with `none`, no memory is read
  __device__ __forceinline__ void load(int buf, int i, int kb, unsigned rows_on, bool none = false) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)((unsigned long long)(unsigned)words[0] | (unsigned long long)(unsigned)words[1] << 32), 0, words[2], words[3]);
    const unsigned v = none ? past_end(words) : voff, at = none ? 0u : base + (i * I + kb * 128 + rows_on * I) * (unsigned)sizeof(bf16_t);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
      w[buf][ct][i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, v, at + 16 * ct * I * (unsigned)sizeof(bf16_t), 0));
  }
  // 32-bit word d of the four registers of column tile ct
  __device__ __forceinline__ void transpose(int buf, int ct, int d) {
    auto swap1 = [](unsigned v) { return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true); };   // lane ^ 1
    auto swap2 = [](unsigned v) { return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true); };   // lane ^ 2
    const unsigned x0 = w[buf][ct][0][d], x1 = w[buf][ct][1][d], x2 = w[buf][ct][2][d], x3 = w[buf][ct][3][d];
    const unsigned s0 = swap1(x0), s1 = swap1(x1), s2 = swap1(x2), s3 = swap1(x3);      // (outside the choices: every lane trades)
    const unsigned y0 = odd1 ? s1 : x0, y1 = odd1 ? x1 : s0, y2 = odd1 ? s3 : x2, y3 = odd1 ? x3 : s2;
    const unsigned t0 = swap2(y0), t1 = swap2(y1), t2 = swap2(y2), t3 = swap2(y3);
    unsigned r0 = odd2 ? t2 : y0, r1 = odd2 ? t3 : y1, r2 = odd2 ? y2 : t0, r3 = odd2 ? y3 : t1;
    asm volatile("" : "+v"(r0), "+v"(r1), "+v"(r2), "+v"(r3));       // (here, and not where they are used)
    w[buf][ct][0][d] = r0;
    w[buf][ct][1][d] = r1;
    w[buf][ct][2][d] = r2;
    w[buf][ct][3][d] = r3;
  }
  __device__ __forceinline__ bf16x8 operand(int buf, int ct, int m) const { return __builtin_bit_cast(bf16x8, w[buf][ct][m]); }
};

// One block of F::BN2 output columns (from column n0 on) for the first NRT 16-row tiles of a tile whose activations sit in LDS
// (`acts`: [K block][BM][128], granules swizzled), and its way out through `stage` (moe.py:92-93).  Its first K block is in buffer 0,
// transposed already, and the one behind it on its way in buffer 1; `next`: the K blocks of another column block follow.  The pipeline runs
// over (MFMA of the block, row tile): an activation fragment is read three row tiles ahead, the loads of MFMA m's registers two K blocks on
// follow that MFMA's last use of them, and the next K block changes lanes in the second half of this one.
template <int CT, int NRT>
__device__ __forceinline__ void wide_down_block(const bf16_t* acts, DownWeights<WideShape<CT>::I, CT>& dw, bf16x8 (&xa)[WideShape<CT>::kActs], bool next,
                                                int n0, const float* w_s, const int* slot_s, int rows, bf16_t* stage, int H,
                                                bf16_t* __restrict__ yw_) {
  using F = WideShape<CT>;
  constexpr int NX = F::kActs, AH = NX - 1, I = F::I, BM = F::BM, KB = I / 128, kPairs = 4 * NRT, kSlots = kPairs / 2, kSets = CT * 4;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g4 = lane >> 4;
  floatx4 acc[CT][NRT];
  int fo = n * 128 + ((4 * k_segment(g4) ^ n) << 3);        // MFMA m's granule of row n sits at fo ^ 8 m
  // (through an empty asm: a K block's address is made where it is used, instead of one for each kept alive)
  auto frag = [&](int kb, int p) {                           // K block kb, pair p
    return *reinterpret_cast<const bf16x8*>(acts + kb * (BM * 128) + (p % NRT) * 16 * 128 + (fo ^ ((p / NRT) * 8)));
  };
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int buf = kb & 1;
    asm volatile("" : "+v"(fo));
#pragma unroll
    for (int p = 0; p < kPairs; ++p) {
      const int m = p / NRT, rt = p % NRT;
      xa[(kb * kPairs + p + AH) % NX] = p + AH < kPairs ? frag(kb, p + AH) : frag((kb + 1) % KB, p + AH - kPairs);
      if (p >= kPairs - kSlots) {
        const int slot = p - (kPairs - kSlots);
#pragma unroll
        for (int t = slot * kSets / kSlots; t < (slot + 1) * kSets / kSlots; ++t) dw.transpose(buf ^ 1, t >> 2, t & 3);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        acc[ct][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(dw.operand(buf, ct, m), xa[(kb * kPairs + p) % NX],
                                                              kb == 0 && m == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : acc[ct][rt], 0, 0, 0);
      if (rt == NRT - 1) dw.load(buf, m, (kb + 2) % KB, n0 + (kb + 2) / KB * F::BN2, kb + 2 >= KB && !next);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // accumulator: lane holds row 16*rt + n, columns wave*16*CT + 16*ct + 4*g4 + i
  // (The thread index goes through an empty asm so the staging addresses are formed here, per block,
  // instead of being hoisted out of the loop and kept alive across the multiply.)
  int lane_o = lane;
  asm volatile("" : "+v"(lane_o));
  const int no = lane_o & 15, g4o = lane_o >> 4;
  constexpr int kCols = 16 * CT, kPieces = 2 * CT;
  bf16_t* const O = stage + wave * (BM * kCols);
  bf16_t* const yw = yw_ + n0 + wave * kCols;
  size_t row_at[kPieces];
  bool mine[kPieces];
#pragma unroll
  for (int i = 0; i < kPieces; ++i) {
    const int at = lane_o + kWave * i, m = at / kPieces;
    mine[i] = m < NRT * 16 && m < rows;
    row_at[i] = (size_t)slot_s[m] * H + (at - m * kPieces) * 8;
  }
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt) {
    const float ws = w_s[rt * 16 + no];                                              // moe.py:93
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      bf16x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (bf16_t)(ws * acc[ct][rt][i]);
      *reinterpret_cast<bf16x4*>(O + (rt * 16 + no) * kCols + 16 * ct + 4 * g4o) = v;
    }
  }
  asm volatile("" ::: "memory");           // one wave's LDS accesses are served in order
  __builtin_amdgcn_wave_barrier();
  u32x4 out[kPieces];
#pragma unroll
  for (int i = 0; i < kPieces; ++i) out[i] = *reinterpret_cast<const u32x4*>(O + (lane_o + kWave * i) * 8);
#pragma unroll
  for (int i = 0; i < kPieces; ++i)
    if (mine[i]) *reinterpret_cast<u32x4*>(yw + row_at[i]) = out[i];
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}

template <int CT>
__global__ __launch_bounds__(512) void experts_wide_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ wgu,
                                                            const bf16_t* __restrict__ wd,
                                                            const float* __restrict__ theta,
                                                            const float* __restrict__ w,
                                                            const int32_t* __restrict__ offsets,
                                                            const int32_t* __restrict__ perm_slot,
                                                            const int32_t* __restrict__ perm_token, int H, int E,
                                                            int act, unsigned x_bytes, bf16_t* __restrict__ yw) {
  using F = WideShape<CT>;
  constexpr int NT = F::NT, BM = F::BM, I = F::I, BK = F::BK;
  __shared__ __attribute__((aligned(1024))) bf16_t S[F::kRing * F::kStageElems];   // weight stages, then the activations
  __shared__ __attribute__((aligned(16))) bf16_t A[F::kXElems];           // x rows, then output staging
  __shared__ float ssq[4 * BM];
  __shared__ float rinv_s[BM], gain_s[BM], w_s[BM];
  __shared__ int slot_s[BM];

  const TileMap tm = load_tile_map(offsets, E);
  int e, first, rows, tile_e;                           // the same for every lane, in scalar registers
  if (!find_round_tile<BM, 2, 2, 1>(tm, blockIdx.x, e, first, rows, tile_e)) return;
  const int row0 = __builtin_amdgcn_readlane(tm.lo, e) + first;
  // the tiles of an expert walk the weights of a K step from different blocks of columns on (experts_fused_kernel says why)
  const int rot = tile_e % NT;
  const int nblocks = (rows + 31) >> 5;                 // 32-row blocks that hold rows: 1 or 2

  // The rest of the kernel exists once per number of blocks, chosen here, where nothing is alive yet: the copies
  // share no values, so each gets the registers the kernel would get if it were the only one.
  auto body = [&](auto nblocks_c) {
  constexpr int kBlocks = decltype(nblocks_c)::value;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wn = wave & 3, wm = wave >> 2;
  const bool busy = wm < kBlocks;          // the two waves of a SIMD belong to different M waves
  const int mbase = wm * 32;
  // accumulator block j of a wave holds its 32-column block block_of(j)
  auto block_of = [&](int j) { const int b = j + rot; return b >= NT ? b - NT : b; };
  // slice i of the activations, columns [128 i, 128 i + 128) of all BM rows
  auto slice = [&](int i) -> bf16_t* { return S + i * (BM * 128); };

  // ---- phase 1: gate/up projection (moe.py:81-86) ----
  constexpr int RT = 2;                   // a wave's 16-row tiles
  floatx4 acc[RT][2 * NT][2];             // [..][0..NT) gate blocks, [..][NT..2NT) the up blocks of the same columns, two 16-column tiles each
  {
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g4 = lane >> 4;
    // DMA side: thread t of an instruction fills granule t (row t/8, position t%8) of its 64 rows and fetches
    // logical granule (t%8) ^ ((row >> 1) & 7) of that row: granule c of a stage row sits at c ^ ((row >> 1) & 7).
    // Stage row (wn*2 + gu)*32 + r of sub-step t is weight row gu*I + (wn*NT + t)*32 + r: instruction q = wn.
    const int chunk = (tid & 7) ^ ((tid >> 4) & 7);
    const int drow = tid >> 3;
    const unsigned hb = (unsigned)H * sizeof(bf16_t);                            // bytes per weight / hidden-state row
    constexpr unsigned kb = BK * sizeof(bf16_t);
    const int nsteps = H / BK;
    const i32x4 w_rsrc = make_words(wgu + (size_t)e * 2 * I * H, 2u * I * hb), x_rsrc = make_words(x, x_bytes);
    const unsigned b_voff = ((unsigned)((drow >> 5) * I + (drow & 31))) * hb + chunk * 16;
    const unsigned bstep = (unsigned)NT * 32 * hb;
    const unsigned wave_bytes = wave * 1024;
    const unsigned s_lds = lds_address(S) + wave_bytes, a_lds = lds_address(A) + wave_bytes;
    const unsigned a_voff = (unsigned)perm_token[row0 + min(drow, rows - 1)] * hb + chunk * 16;   // gather, moe.py:81 (rows past the end: the last one)
    // the transfers of sub-step (s, t) into stage `st` and of step s into x buffer `xb`; for steps past the last one, whose buffers nobody
    // reads again, they lie past the descriptors' ends and touch no memory (where x is close to 2^32 bytes and the sum of the offsets wraps,
    // they read from its first row): every sub-step issues the same number
    auto request_w = [&](int q, int t, int s, unsigned st) {
      dma16_unseen(w_rsrc, s < nsteps ? b_voff : past_end(w_rsrc), (unsigned)block_of(t) * 32 * hb + (unsigned)s * kb + q * bstep,
                   s_lds + st * (F::kStageElems * (unsigned)sizeof(bf16_t)) + q * 8192);
    };
    auto request_x = [&](int s, unsigned xb) {
      dma16_unseen(x_rsrc, s < nsteps ? a_voff : past_end(x_rsrc), (unsigned)s * kb, a_lds + xb * (F::kAElems * (unsigned)sizeof(bf16_t)));
    };
    // One pipeline over eight groups (k32 step, 16-column tile) a sub-step, RT MFMAs each.  A group's weight fragment is read D groups ahead,
    // across the ends of sub-steps: D groups before a sub-step ends the waves meet (the next stage has landed, every fragment of
    // this one has been read), this stage is requested again for three sub-steps on, a transfer a group, and the next stage's
    // fragments are read.  The x fragments of a step are read while the last sub-step of the step before is multiplied, as the ones they
    // replace fall free.  The order is pinned:
    // left to itself the compiler reads a fragment into the registers of the last one and waits for it on the spot.
    constexpr int kG = 8;
    auto kloop = [&](auto rtc) {
      constexpr int R = decltype(rtc)::value;                   // this wave's 16-row tiles that hold rows
      constexpr int D = 3, NB = D + 1;
      static_assert(kG * NT % NB == 0, "a step's groups end where they began in the ring of fragments");
      constexpr int kOps = F::kBInstr + F::kAInstr;
      const int e0 = (g4 ^ ((n >> 1) & 7)) * 8;                 // granule 4 ks + g4 of a row sits at e0 ^ 32 ks
      const bf16_t* const ap = A + (mbase + n) * BK;
      const bf16_t* const bp = S + (wn * 64 + n) * BK;
      bf16x8 a[2][R > 0 ? R : 1], b[NB];
      auto read_a = [&](int ks, int rt, unsigned xb) { a[ks][rt] = *reinterpret_cast<const bf16x8*>(ap + xb * F::kAElems + (e0 ^ (32 * ks)) + rt * 16 * BK); };
      auto read_b = [&](int q, unsigned st) {                   // group q: k32 step q / 4, tile q % 4 (gate, gate, up, up)
        return *reinterpret_cast<const bf16x8*>(bp + st * F::kStageElems + (e0 ^ (32 * (q >> 2))) + (q & 3) * 16 * BK);
      };
      // operation i of what follows the meeting of a sub-step: four transfers of weights and, behind the first sub-step of a step, of x rows
      auto refill = [&](int i, int t, int s, unsigned st, unsigned xb) {
        if (i < F::kBInstr) request_w(i, (t + 3) % NT, s + (t + 3) / NT, st);
        else if (t == 0 && i < kOps) request_x(s + F::kXRing, xb);
      };
      // prologue, oldest first (weight rows first: they do not wait for the row indices)
#pragma unroll
      for (int q = 0; q < F::kBInstr; ++q) request_w(q, 0, 0, 0);
      request_x(0, 0);
#pragma unroll
      for (int q = 0; q < F::kBInstr; ++q) request_w(q, 1, 0, 1);
      request_x(1, 1);
#pragma unroll
      for (int i = 0; i < D; ++i) refill(i, NT - 1, -1, 2, 2);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int j = 0; j < 2 * NT; ++j) acc[rt][j][0] = acc[rt][j][1] = floatx4{0.f, 0.f, 0.f, 0.f};
      meet_waves<F::kBInstr + F::kAInstr + D>();
      if constexpr (R > 0) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int rt = 0; rt < R; ++rt) read_a(ks, rt, 0);
#pragma unroll
        for (int q = 0; q < D; ++q) b[q] = read_b(q, 0);
      }
      unsigned st = 0, xb = 0;
#pragma clang loop unroll(disable)      // (nor peeled: the copy of the last step spilled accumulators)
      for (int s = 0; s < nsteps; ++s) {
        const unsigned xn = xb + 1 == F::kXRing ? 0 : xb + 1, xp = xb == 0 ? F::kXRing - 1 : xb - 1;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const unsigned next = st + 1 == 3 ? 0 : st + 1, before = st == 0 ? 2 : st - 1;
#pragma unroll
          for (int q = 0; q < kG; ++q) {
            const int ks = q >> 2, j = q & 3, run = t * kG + q;
            if (q == kG - D) {                                  // in flight: what the sub-step before asked for
              if (t == 1) meet_waves<kOps>(); else meet_waves<F::kBInstr>();
            }
            if constexpr (R > 0) {
              b[(run + D) % NB] = q < kG - D ? read_b(q + D, st) : read_b(q + D - kG, next);
#pragma unroll
              for (int rt = 0; rt < R; ++rt) {
                if (t == NT - 1 && q == 4 + rt / 2) read_a(0, rt, xn);    // (the next step's x rows are there, a[0] is free)
                if (t == 0 && q == rt / 2) read_a(1, rt, xb);
              }
              __builtin_amdgcn_sched_barrier(0);
#pragma unroll
              for (int rt = 0; rt < R; ++rt) {
                floatx4& c = acc[rt][(j >> 1) * NT + t][j & 1];
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[run % NB], a[ks][rt], c, 0, 0, 0);
              }
              __builtin_amdgcn_sched_barrier(0);
            }
            // operations of this sub-step's refill behind its meeting, of the one before's in front of it
            if (q >= kG - D) refill(q - (kG - D), t, s, st, xb);
            else if (t > 0) refill(q + D, t - 1, s, before, xb);
            else refill(q + D, NT - 1, s - 1, before, xp);
            __builtin_amdgcn_sched_barrier(0);
          }
          st = next;
        }
        xb = xn;
      }
    };
    using std::integral_constant;
    if (busy) kloop(integral_constant<int, RT>{});
    else kloop(integral_constant<int, 0>{});
  }
  wait_loads_and_sync();                   // every transfer has landed and every wave is done with the stages
  // (through an empty asm, so that nothing made of it is kept alive across phase 1)
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63, n = lane & 15, g4 = lane >> 4;

  // ---- phase 2: Radial NormSiLU (moe.py:87-92), activations to LDS ----
  DownWeights<I, CT> dw;
  // The accumulators are transposed (lane = row mbase + 16*rt + n, register i = column 4*g4 + i of its 16-column tile),
  // so a row's sum of gate^2 is a sum over this lane's registers, the three lanes with the row's other columns and the four N
  // waves; and every lane owns runs of four consecutive columns, which leave as one 8-byte LDS write.
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    float part[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      part[j] = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) part[j] = fmaf(acc[rt][j][i >> 2][i & 3], acc[rt][j][i >> 2][i & 3], part[j]);
    }
    float sq = 0.f;
#pragma unroll
    for (int b = 0; b < NT; ++b) {             // in column order, whichever block the tile began with
      float v = part[0];
#pragma unroll
      for (int j = 1; j < NT; ++j) v = block_of(j) == b ? part[j] : v;
      sq += v;
    }
    Pair p = lanes16(sq);
    sq = p.a + p.b;
    p = lanes32(sq);
    sq = p.a + p.b;
    if (g4 == 0) ssq[wn * BM + mbase + rt * 16 + n] = sq;
  }
  __syncthreads();
  if (tid < BM) {
    const float p = radial_exponent(theta, e, act);                                   // moe.py:89
    const float ms = ((ssq[tid] + ssq[BM + tid]) + ssq[2 * BM + tid]) + ssq[3 * BM + tid];
    radial_row_scalars(ms, I, p, act, rinv_s[tid], gain_s[tid]);                      // 1/r and r^p, moe.py:88-89
    const int slot = perm_slot[row0 + min(tid, rows - 1)];
    slot_s[tid] = slot;
    w_s[tid] = w[slot];
  }
  __syncthreads();
  // phase 3 streams w_down through registers; its first two K blocks are requested here, in the second half of the activation: the
  // accumulators of the first are dead by then and make room, and the loads fly during the rest of the activation arithmetic
  dw.init(wd + (size_t)e * H * I, H, wave * (16 * CT), lane);
  {
    // slice t holds activation columns [128t, 128t + 128) of all 64 rows, [64][128], granules swizzled
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) dw.load(rt, i, rt, 0);
      if (!busy) continue;                    // a block without rows: nobody reads its activations
      const int m = mbase + rt * 16 + n;
      const float rinv = rinv_s[m];
      const float nrl = -1.44269504f * rinv, rg = rinv * gain_s[m];            // per-row constants folded once
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int tile32 = wn * NT + block_of(j);      // 32-column block of the activation row: slice tile32 / 4, granules (tile32 % 4) * 4 + ..
        bf16_t* hrow = slice(tile32 >> 2) + m * 128 + 4 * (g4 & 1);
#pragma unroll
        for (int c = 0; c < 2; ++c) {        // columns tile32*32 + 16*c + 4*g4 + 0..3: half of a granule
          bf16x4 hv;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float g = acc[rt][j][c][r];
            const float sg = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(g * nrl));   // sigmoid(g/r)
            hv[r] = (bf16_t)(g * rg * sg * acc[rt][NT + j][c][r]);                     // SiLU(g/r) r^p up
          }
          const int gr = (tile32 & 3) * 4 + 2 * c + (g4 >> 1);
          *reinterpret_cast<bf16x4*>(hrow + (gr ^ (m & 15)) * 8) = hv;
        }
      }
    }
  }
  __syncthreads();                         // the activation tile is complete

  // ---- phase 3: down projection, routing weight, scatter to slot order (moe.py:92-93) ----
  constexpr int NRT = 2 * kBlocks;
#pragma unroll
  for (int t = 0; t < 4 * CT; ++t) dw.transpose(0, t >> 2, t & 3);
  bf16x8 xa[F::kActs];
#pragma unroll
  for (int p = 0; p < F::kActs - 1; ++p)
    xa[p] = *reinterpret_cast<const bf16x8*>(S + ((p % NRT) * 16 + n) * 128 + (((4 * k_segment(g4) ^ n) ^ (p / NRT)) << 3));
  for (int n0 = 0; n0 < H; n0 += F::BN2) wide_down_block<CT, NRT>(S, dw, xa, n0 + F::BN2 < H, n0, w_s, slot_s, rows, A, H, yw);
  };   // body
  if (nblocks == 2) body(std::integral_constant<int, 2>{});
  else body(std::integral_constant<int, 1>{});
}

template <int CT>
void launch_wide_t(const bf16_t* x, const bf16_t* wgu, const bf16_t* wd, const float* theta, const float* w, const int32_t* offsets,
                   const int32_t* perm_slot, const int32_t* perm_token, int S, int H, int E, int act, unsigned x_bytes, void* yw,
                   hipStream_t s) {
  hipLaunchKernelGGL(experts_wide_kernel<CT>, dim3(round_tiles_most(S, E, WideShape<CT>::BM)), dim3(512), 0, s, x, wgu, wd, theta, w, offsets,
                     perm_slot, perm_token, H, E, act, x_bytes, static_cast<bf16_t*>(yw));
}

}  // namespace
}  // namespace bibo
