// Kernels 3 and 4 in one launch: a workgroup takes up to 128 permuted rows of one expert through the gate/up
// projection, Radial NormSiLU and the down projection without the activations leaving the CU.
//
// Phase 1 (gate/up GEMM, 2 x 4 waves, v_mfma_f32_32x32x16_bf16, operands swapped so that a lane ends up with
// one ROW's values) walks K in steps of 64 elements, so every row an LDS-DMA instruction fetches is a whole
// 128-byte line: the L2 -> LDS path moves almost twice the bytes per second for whole lines than for the
// half lines of a 32-element step.  All 2I weight rows of a step would not fit LDS more than once, so a step
// is cut into I/128 sub-steps of 256 rows: sub-step t holds, for each of the four N waves, its t-th 32-column
// gate tile and the up tile of the same columns (16 MFMAs per wave).  The 32 KB stages form a ring of three (two
// where I < 384 meets blocks of 384 output columns, whose staging buffers leave no room): the rows of sub-step
// n + ring - 1 are requested while sub-step n is multiplied, and a wave waits only until the loads older than the
// latest sub-step's have landed (loads complete in order), so the L2 -> LDS path always has a stage or two in flight
// instead of draining at every barrier.  The x rows of step s+1 arrive during step s in a double buffer of their own
// (I = 384), or those of step s+2 in a ring of three (I < 384).
// Phase 2 turns the accumulators into bf16 activations and parks them in the stages, whose contents are dead by
// then, as an operand of the second GEMM: stage t holds columns [128t, 128t+128) of all 128 rows; row r keeps
// 16-byte granule c at position c ^ (r & 15), which spreads the 16 lanes of a fragment read over all banks
// although the row stride is 256 bytes.
// Phase 3 has no barriers and no LDS traffic for the weights: the eight waves split a block of 128*CT
// output columns (16*CT each), every wave multiplies ALL 128 resident rows with v_mfma_f32_16x16x32_bf16
// and pulls its own w_down rows straight from global memory into registers, up to three 128-byte K
// blocks ahead (the four lanes of a weight row fetch 64 contiguous bytes per instruction).  Keeping the
// in-flight bytes in registers instead of LDS is what lets a CU cover the memory latency here: the
// activations already fill most of the LDS.
// Each block of columns is scaled by the routing weight, staged through LDS 32 rows at a time (in the two x
// buffers, which are idle by then) and scattered to slot order as 256-byte row segments.
// A tile may hold fewer than 128 rows: find_round_tile chooses the heights of a call's tiles by the rounds of the chip they come to, and
// an expert's last tile may have less.  32-row blocks without rows are not multiplied: the kernel body exists once per number of blocks
// (1 to 4), with the MFMAs, activations, down projection row tiles and output rounds of the missing blocks left out, and of up to two blocks
// each M wave takes one; every wave still issues its share of the weight requests, which is most of what a tile costs.
// Reference: BiBoFusedExperts.forward, src/modeling/ffn/moe.py:81-93.
#pragma once

#include <climits>
#include <type_traits>

#include "experts_fused_launch.h"
#include "experts_wide.h"
#include "stripe.h"

namespace bibo {
namespace {

template <int NT, int CT, int MT_ = 2>
struct FusedShape {
  static constexpr int MT = MT_, BM = 64 * MT, BK = 64;
  static constexpr int I = 128 * NT;
  static constexpr int BN2 = 128 * CT;                             // output columns per block: 8 waves x CT x 16
  // I = 384: the three stages are the three sub-steps of a K step and the x rows alternate between two buffers.
  // I < 384 with at most 256 output columns per block (kDeep): three stages all the same, walked round by the running
  // sub-step, and a third x buffer, so that x rows are requested two K steps ahead.  Otherwise two stages.
  // I = 512 (NT = 4) takes 64-row tiles (MT = 1): a row's 1024 accumulator columns leave registers for no more.  Its four
  // sub-steps per K step walk the ring by the running sub-step too.
  static constexpr bool kDeep = (NT < 3 && CT < 3) || NT == 4;
  static constexpr int kRing = (NT == 3 || kDeep) ? 3 : 2;         // weight stages in LDS
  static constexpr int kDist = kRing - 1;                          // sub-steps between a stage's request and its use
  static constexpr int kStageRows = 256;                           // 4 N waves x (gate tile + up tile) x 32 rows
  static constexpr int kStageElems = kStageRows * BK;              // 32 KB = one [128][128] slice of the activations
  static constexpr int kAElems = BM * BK;                          // x rows of one K step
  static constexpr int kOutRows = 32;                              // rows of a column block staged at a time
  static constexpr int kOutElems = kOutRows * BN2;
  static constexpr int kXElems = kAElems > kOutElems ? kAElems : kOutElems;   // a buffer that serves as either
  static constexpr int kBInstr = kStageRows * (BK / 8) / 512;      // load instructions per thread and weight stage
  static constexpr int kAInstr = BM * (BK / 8) / 512;              // and per x stage
  static_assert(kBInstr == 4 && kAInstr == MT && BM * (BK / 8) % 512 == 0, "stage does not divide over the threads");
  static_assert(MT == 2 ? NT <= 3 : NT <= 4, "accumulators and activations of a tile");
};

// What one thread needs to request a weight stage and the x rows of a K step.
template <typename F>
struct SubLoader {
  __amdgpu_buffer_rsrc_t w_rsrc, x_rsrc;   // this expert's w_gate_up block; the hidden states
  unsigned b_voff;         // byte offset of this thread's row and granule inside an instruction's 64 rows
  unsigned b_soff;         // byte offset of the stage's first tile row, K offset included (uniform)
  unsigned bstep;          // bytes between the rows of consecutive instructions (uniform)
  bf16_t* b_dst;           // LDS stage
  unsigned a_voff[F::kAInstr];   // byte offsets of this thread's token rows and granule
  unsigned a_soff;         // K offset in bytes (uniform)
  bf16_t* a_dst;           // LDS x stage
  int wave_elems;          // this wave's place in an instruction's LDS block, in elements (uniform: a scalar register,
                           // so that the LDS base of every transfer is formed by scalar instructions alone)
};

// The load instructions of one sub-step: the weight stage kDist sub-steps ahead and, in the first sub-step of a K
// step (WITH_A), the next step's x rows.  Shaped like StripeLoader so that stripe_step can spread them between its
// MFMAs.
template <typename F, bool WITH_A>
struct SubIssuer {
  const SubLoader<F>& d;
  static constexpr int kInstr = F::kBInstr + (WITH_A ? F::kAInstr : 0);
  template <int Q>
  __device__ __forceinline__ void issue(int, bf16_t*) const {
    if constexpr (Q < F::kBInstr) dma16_buf(d.w_rsrc, d.b_voff, d.b_soff + Q * d.bstep, d.b_dst + Q * 512 * 8 + d.wave_elems);
    else if constexpr (WITH_A && Q < F::kBInstr + F::kAInstr)
      dma16_buf(d.x_rsrc, d.a_voff[Q - F::kBInstr], d.a_soff, d.a_dst + (Q - F::kBInstr) * 512 * 8 + d.wave_elems);
  }
};

// One 128-byte K block of a wave's 16*CT w_down rows as it comes from memory: lane l holds 16-byte piece l % 4 of
// the first (s = 0) or second (s = 1) 64 bytes of row l / 4 of column tile ct.  The four lanes of a row are
// ADJACENT, so the texture unit merges them into one 64-byte request; lanes that are 16 apart, as in the MFMA
// operand layout, are not merged and move less than half the bytes per second.
template <int CT>
struct WBlock {
  bf16x8 w[CT][2];
};

template <int CT>
__device__ __forceinline__ void load_wblock(WBlock<CT>& b, const bf16_t* __restrict__ wp, size_t tile_stride, int kb) {
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const bf16_t* p = wp + ct * tile_stride + kb * 64;
    b.w[ct][0] = *reinterpret_cast<const bf16x8*>(p);
    b.w[ct][1] = *reinterpret_cast<const bf16x8*>(p + 32);
  }
}

// Memory order -> MFMA operand order: lane r + 16 g takes the register of lane 4 r + g (row r, piece g).  sel is
// 4 * (source lane); the exchange uses the LDS crossbar and no LDS memory.
__device__ __forceinline__ bf16x8 to_operand_lanes(bf16x8 v, int sel) {
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  i32x4 u = __builtin_bit_cast(i32x4, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) u[i] = __builtin_amdgcn_ds_bpermute(sel, u[i]);
  return __builtin_bit_cast(bf16x8, u);
}

// One block of F::BN2 output columns (from column n0 on) for the first NRT 16-row tiles of a tile whose activations sit in LDS
// (`slice(i)`: columns [128 i, 128 i + 128) of all rows), and its way out through the staging buffers O0 and O1 (moe.py:92-93).
// wb: the first D K blocks of this wave's w_down rows, already requested; with `more`, the next column block's are on return.
// f32_rows: the rows leave in fp32, 16-byte stores from the accumulators, 64 bytes of a row by four of them.
template <typename F, int CT, int KB, int D, int NB, int NRT, typename Slice>
__device__ __forceinline__ void down_block(Slice slice, WBlock<CT> (&wb)[NB], const bf16_t*& wp, size_t tile_stride, bool more, int n0,
                                           const float* w_s, const int* slot_s, int rows, bf16_t* O0, bf16_t* O1, int H,
                                           void* __restrict__ yw_, bool f32_rows) {
  bf16_t* const yw = static_cast<bf16_t*>(yw_);
  constexpr int I = F::I;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int r16 = lane & 15, g4 = lane >> 4;
  const int sel = 4 * (4 * r16 + g4);
  floatx4 acc2[CT][NRT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) acc2[ct][rt] = floatx4{0.f, 0.f, 0.f, 0.f};
  // Activation fragments are read a row tile ahead of the MFMAs that consume them (across K block
  // boundaries too).
  auto frag = [&](int kb, int rt, int s) {
    // K elements 64 kb + 32 s + 8 g4 .. + 8 of row 16 rt + r16: slice kb / 2, granule (kb % 2) * 8 + 4 s + g4
    const int gq = ((((kb & 1) * 8 + g4) ^ r16) * 8) ^ (s * 32);
    return *reinterpret_cast<const bf16x8*>(slice(kb >> 1) + (rt * 16 + r16) * 128 + gq);
  };
  // The multiply walks half K blocks (32 elements, one MFMA deep): while half hs is multiplied with all NRT
  // row tiles, the weights of half hs + 1 change lanes and the activation fragment of the next row tile is read.
  bf16x8 wc[2][CT], xa[2];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) wc[0][ct] = to_operand_lanes(wb[0].w[ct][0], sel);
  xa[0] = frag(0, 0, 0);
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    if (kb + D < KB) load_wblock<CT>(wb[(kb + D) % NB], wp, tile_stride, kb + D);
    __builtin_amdgcn_sched_barrier(0);     // keep the loads D blocks ahead of their use
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int hs = 2 * kb + s;
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) {
        const int g = hs * NRT + rt;         // running (half K block, row tile) index
        if (g + 1 < KB * 2 * NRT) xa[(g + 1) & 1] = frag(((g + 1) / NRT) >> 1, (g + 1) % NRT, ((g + 1) / NRT) & 1);
        // the CT lane exchanges of the next half are spread over the row tiles (the last tile takes what is left)
#pragma unroll
        for (int cx = 0; cx < CT; ++cx)
          if ((cx == rt || (rt == NRT - 1 && cx > rt)) && hs + 1 < 2 * KB)
            wc[(hs + 1) & 1][cx] = to_operand_lanes(wb[((hs + 1) >> 1) % NB].w[cx][(hs + 1) & 1], sel);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
          acc2[ct][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[hs & 1][ct], xa[g & 1], acc2[ct][rt], 0, 0, 0);
      }
    }
  }
  wp += (size_t)F::BN2 * I;                                  // next block of columns: in flight during the epilogue
  if (more) {
#pragma unroll
    for (int d = 0; d < D; ++d) load_wblock<CT>(wb[d], wp, tile_stride, d);
  }
  __builtin_amdgcn_sched_barrier(0);
  // accumulator: lane holds row 16*rt + r16, columns wave*16*CT + 16*ct + 4*g4 + i.  The block leaves 32 rows at
  // a time through the two x buffers in turn; between two barriers a wave stages the next 32 rows into one
  // buffer and copies the previous 32 out of the other.  Staged row r keeps granule c at position c ^ (r & 15): the 8-byte writes of a half wave
  // then cover all banks.  Copy-out: 16 consecutive threads move 256 contiguous bytes of one row.
  // (The thread index goes through an empty asm so the staging addresses are formed here, per block,
  // instead of being hoisted out of the loop and kept alive across the multiply.)
  int tid_o = tid;
  asm volatile("" : "+v"(tid_o));
  const int r16o = tid_o & 15, g4o = (tid_o >> 4) & 3;
  const int ro = tid_o >> 4, pco = tid_o & 15;             // copy-out: staged row, first granule position
  auto stage_rows = [&](int hf) {          // rows 32 hf .. + 32 of the block into buffer hf % 2
    bf16_t* const O = (hf & 1) ? O1 : O0;
#pragma unroll
    for (int rq = 0; rq < F::kOutRows / 16; ++rq) {
      const int rt = hf * (F::kOutRows / 16) + rq;
      const float ws = w_s[rt * 16 + r16o];                                            // moe.py:93
      bf16_t* orow = O + (rq * 16 + r16o) * F::BN2 + (g4o & 1) * 4;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const int c = wave * (2 * CT) + ct * 2 + (g4o >> 1);
        bf16x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (bf16_t)(ws * acc2[ct][rt][i]);
        *reinterpret_cast<bf16x4*>(orow + (c ^ r16o) * 8) = v;
      }
    }
  };
  auto copy_out = [&](int hf) {
    const bf16_t* const O = (hf & 1) ? O1 : O0;
    const int m = hf * F::kOutRows + ro;
    if (m < rows) {
      bf16_t* dst = yw + (size_t)slot_s[m] * H + n0;
      const bf16_t* src = O + ro * F::BN2;
#pragma unroll
      for (int q = 0; q < CT; ++q) {                         // 16 CT granules per row, 16 threads per row
        const int pc = pco + 16 * q;
        *reinterpret_cast<u32x4*>(dst + (pc ^ (ro & 15)) * 8) = *reinterpret_cast<const u32x4*>(src + pc * 8);
      }
    }
  };
  constexpr int NR = NRT * 16 / F::kOutRows;
  if (f32_rows) {
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
      const int m = rt * 16 + r16o;
      if (m >= rows) continue;
      const float ws = w_s[m];
      float* const dst = static_cast<float*>(yw_) + (size_t)slot_s[m] * H + n0 + wave * (16 * CT) + 4 * g4o;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) *reinterpret_cast<floatx4*>(dst + 16 * ct) = ws * acc2[ct][rt];
    }
    return;
  }
  stage_rows(0);
#pragma unroll
  for (int hf = 0; hf < NR; ++hf) {
    __syncthreads();                       // rows of round hf are staged; round hf - 1 has left its buffer
    if (hf + 1 < NR) stage_rows(hf + 1);
    copy_out(hf);
  }
}

// MODE 0: the forward pass.  MODE 1: the backward pass's recomputation - the kernel stops after phase 1 and writes the
// pre-activations themselves, rounded to bf16, to `preact` [S, 2I] in permuted row order (gate columns, then up
// columns), staged through the LDS stages into whole row segments.  MODE 2: the training forward - the forward pass that
// also leaves those pre-activations for its backward, in the same way (8-byte stores straight from the accumulator
// registers during phase 2 were slower: 140 against 133 us at T = 8192).  MODE 3: as MODE 1, but the fp32 sums as they are, for
// down_act_kernel (`preact` points to floats): 16-byte stores from the accumulators, a row's 128 bytes in four of them.
// SCAN (slots a thread looks at): no permutation has run.  A workgroup adds up the router's histograms for the tile map and looks through
// all selections for its tile's rows, a wave 64 slots in a row at a time, in slot order as the permutation has them.  Reading offsets and
// rows of a permutation takes two memory latencies too, and the launch in front of it is saved: 0.4 to 1.5 us more here (0.11 a slot of a
// thread) against 3.0 to 5.9 of permuting and the gap between two launches.  Kernels of a layer, permutation -> this, us: H = 512,
// I = 256, k = 6: 30.8 -> 27.5 (T = 256), 33.0 -> 29.1 (800), 38.3 -> 37.0 (2000); H = 768, I = 384: 49.9 -> 47.4, 57.3 -> 54.7,
// 61.1 -> 60.7; nine experts, k = 2: 31.8 -> 26.5, 30.2 -> 26.6, 32.1 -> 28.4.  Beyond one round of tiles a CU would look twice: level at
// 16,000 slots of H = 1024, I = 512.
static_assert(kScanSlots / 128 + kMaxE <= kCUs && kScanSlots / 2 / 64 + kMaxE <= kCUs, "tiles of a call that finds its rows itself fit a round");
template <int NT, int CT, int MODE = 0, int MTP = 2, int SCAN = 0, bool F32_ROWS = false>
__global__ __launch_bounds__(512) void experts_fused_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ wgu,
                                                            const bf16_t* __restrict__ wd,
                                                            const float* __restrict__ theta,
                                                            const float* __restrict__ w,
                                                            const int32_t* __restrict__ offsets,
                                                            const int32_t* __restrict__ perm_slot,
                                                            const int32_t* __restrict__ perm_token, int H, int E,
                                                            int act, unsigned x_bytes, void* __restrict__ yw,
                                                            bf16_t* __restrict__ preact, int column_blocks, ScanArgs scan) {
  using FT = FusedShape<NT, CT, MTP>;
  constexpr int BM = FT::BM, I = FT::I, BK = FT::BK;
  // Every buffer that is read while LDS-DMA fills another is a variable of its own: the compiler orders a DMA
  // transfer against later LDS reads of the same variable with a full wait for the transfer.
  __shared__ __attribute__((aligned(16))) bf16_t S0[FT::kStageElems];  // weight stages, then the activations
  __shared__ __attribute__((aligned(16))) bf16_t S1[FT::kStageElems];
  __shared__ __attribute__((aligned(16))) bf16_t S2[FT::kRing == 3 ? FT::kStageElems : 8];
  __shared__ __attribute__((aligned(16))) bf16_t A0[FT::kXElems];      // x rows of even K steps; then output staging,
  __shared__ __attribute__((aligned(16))) bf16_t A1[FT::kXElems];      // x rows of odd K steps;  alternating per 32 rows
  __shared__ __attribute__((aligned(16))) bf16_t A2[FT::kDeep ? FT::kAElems : 8];   // kDeep: x rows of every third K step
  __shared__ float ssq[4 * BM];
  __shared__ float rinv_s[BM], gain_s[BM], w_s[BM];
  __shared__ int slot_s[BM];

  // MODE 1 and 3 may cut a tile's columns over several workgroups (the others need whole rows): workgroup cb of a tile then
  // owns gate columns [cb I, cb I + I) of a row of row_i = column_blocks I and the up columns behind the same gate columns.
  const int ncb = MODE == 1 || MODE == 3 ? column_blocks : 1, row_i = I * ncb;
  __shared__ int found[SCAN ? 8 * kWave : 1];
  int picked[SCAN ? SCAN : 1];                       // selections of this wave's slots, 64 in a row a time
  const int scan_per = SCAN ? (scan.S + 511) >> 9 : 0;
  int scan_first = 0;
  TileMap tm;
  if constexpr (SCAN > 0) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    scan_first = wave * scan_per * kWave;
#pragma unroll
    for (int q = 0; q < SCAN; ++q) picked[q] = scan.idx[min(scan_first + q * kWave + lane, scan.S - 1)];
    int n = 0;
    for (int c0 = 0; c0 < scan.nhist; c0 += 64) {
      int v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = scan.hist[min(c0 + wave + 8 * u, scan.nhist - 1) * kMaxE + lane];
#pragma unroll
      for (int u = 0; u < 8; ++u) n += c0 + wave + 8 * u < scan.nhist ? v[u] : 0;
    }
#pragma unroll
    for (int q = 0; q < SCAN; ++q)
      if (q >= scan_per || scan_first + q * kWave + lane >= scan.S) picked[q] = -1;
    found[wave * kWave + lane] = n;
    __syncthreads();
    n = 0;
#pragma unroll
    for (int v = 0; v < 8; ++v) n += found[v * kWave + lane];
    tm.n = lane < E ? n : 0;
    tm.lo = wave_inclusive_scan(tm.n) - tm.n;
  } else {
    tm = load_tile_map(offsets, E);
  }
  if constexpr (SCAN > 0 && MODE >= 2) {
    if (blockIdx.x == 0 && threadIdx.x < (unsigned)E) {   // (also where every slot went to an expert that has no weights)
      scan.offsets[threadIdx.x] = tm.lo;
      if (threadIdx.x == (unsigned)E - 1) scan.offsets[E] = tm.lo + tm.n;
      if (scan.counts != nullptr) scan.counts[threadIdx.x] = tm.n;
    }
  }
  int e, first, rows, tile_e, cb = 0;                   // the same for every lane, in scalar registers; first: the tile's first row in its expert
  if (MODE == 3 || ncb > 1) {
    count_tiles(tm, BM);
    const int flat = xcd_tile(blockIdx.x, tm.total * ncb);
    if (flat >= tm.total * ncb) return;
    const int tile = flat / ncb;
    cb = flat - tile * ncb;
    find_tile(tm, tile, e, first, rows, tile_e);
    first = tile_e * BM;
  } else if (!find_round_tile<BM, (NT == 2 ? 2 : 3), (SCAN > 0 ? 0 : NT == 1 ? 1 : INT_MAX), (NT == 2 ? 2 : 3)>(tm, blockIdx.x, e, first, rows, tile_e)) {
    return;
  }
  const int row0 = __builtin_amdgcn_readlane(tm.lo, e) + first;
  // The tiles of an expert walk the weights of a K step from different blocks of columns on: of the tiles that run side by side on an XCD,
  // one pays HBM's latency for a line and the others find it in L2.  A CU keeps about 40 KB of misses in flight, 47 GB/s from HBM and 90
  // from L2.  (Not from different K offsets on: a row's sums would then depend on its place in the tile.)  Layer, weights from HBM, all tiles
  // in the same order -> this: H = 768, I = 384, k = 6: 67 -> 63 us at T = 2049, 130 -> 126 at 6000; H = 1024, I = 512, k = 8: 160 -> 145 at
  // 2049, 292 -> 287 at 6000, 370 -> 355 at 8192.  At I = 256 it is within 2 us either way; so is walking w_down's blocks like this, but at
  // I = 512 (145 -> 155 us at T = 2049).
  const int rot = NT >= 3 ? tile_e % NT : 0;
  if constexpr (SCAN > 0) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int count = 0;
#pragma unroll
    for (int q = 0; q < SCAN; ++q) count += __popcll(__ballot(picked[q] == e));
    __syncthreads();                                     // the histograms' sums have been read
    if (lane == 0) found[wave] = count;
    if (tid < BM) slot_s[tid] = 0;
    __syncthreads();
    int r0 = -first;
#pragma unroll
    for (int v = 0; v < 7; ++v) r0 += v < wave ? found[v] : 0;
#pragma unroll
    for (int q = 0; q < SCAN; ++q) {
      const unsigned long long mine = __ballot(picked[q] == e);
      const int r = r0 + __builtin_amdgcn_mbcnt_hi((unsigned)(mine >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mine, 0));
      if (picked[q] == e && r >= 0 && r < rows) slot_s[r] = scan_first + q * kWave + lane;
      r0 += __popcll(mine);
    }
    __syncthreads();
    if constexpr (MODE >= 2) {
      if (cb == 0 && tid < rows) {
        const int slot = slot_s[tid];
        scan.perm_slot[row0 + tid] = slot;
        if (scan.perm_token != nullptr) scan.perm_token[row0 + tid] = slot / scan.k;
      }
    }
  }
  const int nblocks = (rows + 31) >> 5;                 // 32-row blocks that hold rows: 1 .. 2 MTP

  // The rest of the kernel exists once per number of blocks, chosen here, where nothing is alive yet: the copies
  // share no values, so each gets the registers the kernel would get if it were the only one.
  auto body = [&](auto nblocks_c) {
  constexpr int kBlocks = decltype(nblocks_c)::value;
  constexpr int MT = kBlocks <= 2 ? 1 : MTP;
  using F = FusedShape<NT, CT, MT>;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wn = wave & 3, wm = wave >> 2;
  // M wave wm owns block wm of up to two, else blocks 2 wm and 2 wm + 1; blocks without rows are not multiplied.  The two waves of a SIMD
  // belong to different M waves, so what a SIMD's MFMA pipe has to do goes with the tile's blocks either way.
  const int my_blocks = __builtin_amdgcn_readfirstlane(wm == 0 ? (kBlocks < MT ? kBlocks : MT) : (kBlocks > MT ? kBlocks - MT : 0));
  const int n = lane & 31;
  const int mbase = wm * MT * 32;
  auto stage = [&](auto ic) -> bf16_t* {
    constexpr int i = decltype(ic)::value;
    if constexpr (i == 0) return S0; else if constexpr (i == 1) return S1; else return S2;
  };
  // accumulator tile j of a wave holds its column tile block_of(j)
  auto block_of = [&](int j) { const int b = j + rot; return b >= NT ? b - NT : b; };
  // slice i of the activations, columns [128 i, 128 i + 128) of all BM rows: a whole stage (BM = 128) or half of one
  auto slice = [&](int i) -> bf16_t* {
    if constexpr (MTP == 2) return i == 0 ? S0 : (i == 1 ? S1 : S2);
    else return (i < 2 ? S0 : S1) + (i & 1) * (BM * 128);
  };

  // ---- phase 1: gate/up projection (moe.py:81-86) ----
  floatx16 acc[MT][2 * NT];               // [..][0..NT) gate tiles, [..][NT..2NT) the up tiles of the same columns
  {
    // DMA side: thread t of an instruction fills granule t (row t/8, position t%8) of its 64 rows and fetches
    // logical granule (t%8) ^ ((row >> 1) & 7) of that row: granule c of a stage row sits at c ^ ((row >> 1) & 7).
    // Stage row (wn*2 + gu)*32 + r of sub-step t is weight row gu*I + (wn*NT + t)*32 + r: instruction q = wn.
    const int chunk = (tid & 7) ^ ((tid >> 4) & 7);
    const int drow = tid >> 3;
    const unsigned hb = (unsigned)H * sizeof(bf16_t);                            // bytes per weight / hidden-state row
    const int nsteps = H / BK;
    SubLoader<F> ld;
    ld.w_rsrc = make_rsrc(wgu + (size_t)e * 2 * row_i * H, 2u * row_i * hb);
    ld.x_rsrc = make_rsrc(x, x_bytes);
    ld.b_voff = ((unsigned)((drow >> 5) * row_i + cb * I + (drow & 31))) * hb + chunk * 16;
    ld.bstep = (unsigned)NT * 32 * hb;
    ld.wave_elems = __builtin_amdgcn_readfirstlane(wave) * 64 * 8;
#pragma unroll
    for (int a = 0; a < F::kAInstr; ++a) {
      const int m = min(a * 64 + drow, rows - 1);                                // rows past the end re-read the last valid row
      const int token = SCAN ? slot_s[m] / scan.k : perm_token[row0 + m];
      ld.a_voff[a] = (unsigned)token * hb + chunk * 16;                          // gather, moe.py:81
    }
    const int pos0 = ((lane >> 5) ^ ((n >> 1) & 7)) * 8;    // fragment side: lane (n, h) reads logical granule 2*ss + h of rows congruent to n mod 32
    auto frag_row = [&](int j) { return (wn * 2 + j) * 32; };
    using std::integral_constant;
    auto zero_acc = [&]() {                      // (after the prologue's requests, which do not wait for it)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < 2 * NT; ++j)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[mt][j][i] = 0.f;
    };
    if constexpr (F::kDeep) {
      // Sub-step g = s NT + t reads stage g % 3 and x buffer s % 3, and requests the weight rows of sub-step g + 2
      // and, at t = 0, the x rows of step s + 2 (K steps clamped to the last one: requests past the end fetch valid
      // rows into buffers nobody reads again).  The K loop is unrolled by three steps (ph = s % 3), so every buffer is
      // chosen at compile time.  What a sub-step may leave in flight are the loads of the sub-step before it.
      auto abuf = [&](auto ic) -> bf16_t* {
        constexpr int i = decltype(ic)::value;
        if constexpr (i == 0) return A0; else if constexpr (i == 1) return A1; else return A2;
      };
      constexpr unsigned kb = BK * sizeof(bf16_t);
      // prologue, oldest first: sub-step 0, x rows of steps 0 and 1, sub-step 1
#pragma unroll
      for (int q = 0; q < F::kBInstr; ++q)
        dma16_buf(ld.w_rsrc, ld.b_voff, (unsigned)block_of(0) * 32 * hb + q * ld.bstep, S0 + q * 512 * 8 + ld.wave_elems);
#pragma unroll
      for (int a = 0; a < F::kAInstr; ++a) dma16_buf(ld.x_rsrc, ld.a_voff[a], 0, A0 + a * 512 * 8 + ld.wave_elems);
#pragma unroll
      for (int a = 0; a < F::kAInstr; ++a) dma16_buf(ld.x_rsrc, ld.a_voff[a], kb, A1 + a * 512 * 8 + ld.wave_elems);
#pragma unroll
      for (int q = 0; q < F::kBInstr; ++q)
        dma16_buf(ld.w_rsrc, ld.b_voff, (NT == 1 ? kb : (unsigned)block_of(1) * 32 * hb) + q * ld.bstep, S1 + q * 512 * 8 + ld.wave_elems);
      zero_acc();
      auto substep = [&](auto mc, auto phc, auto tc, int s) {
        constexpr int nmt = decltype(mc)::value;
        constexpr int ph = decltype(phc)::value, t = decltype(tc)::value;
        constexpr int cur = (ph * NT + t) % 3, target = (ph * NT + t + 2) % 3;
        constexpr int tn = (t + 2) % NT, ds = (t + 2) / NT;
        constexpr bool after_t0 = NT == 1 || t == 1;                   // the sub-step before also requested x rows
        sync_keep_loads<F::kBInstr + (after_t0 ? F::kAInstr : 0)>();
        const bf16_t* a0 = abuf(integral_constant<int, ph>{}) + (mbase + n) * BK + pos0;
        const bf16_t* b0 = stage(integral_constant<int, cur>{}) + n * BK;
        ld.b_soff = (unsigned)block_of(tn) * 32 * hb + (unsigned)min(s + ds, nsteps - 1) * kb;
        ld.b_dst = stage(integral_constant<int, target>{});
        ld.a_soff = (unsigned)min(s + 2, nsteps - 1) * kb;
        ld.a_dst = abuf(integral_constant<int, (ph + 2) % 3>{});
        const SubIssuer<F, t == 0> issuer{ld};
        if constexpr (nmt > 0)
          stripe_step<nmt, 2, BK, true, 2 * NT, t, NT>(acc, a0, 32 * BK, b0, pos0, frag_row, issuer, true, 0, nullptr);
        else
          issue_some<0, SubIssuer<F, t == 0>::kInstr>(issuer, 0, nullptr);
      };
      auto kstep = [&](auto mc, auto phc, int s) {
        substep(mc, phc, integral_constant<int, 0>{}, s);
        if constexpr (NT > 1) substep(mc, phc, integral_constant<int, 1>{}, s);
        if constexpr (NT > 2) substep(mc, phc, integral_constant<int, 2>{}, s);
        if constexpr (NT > 3) substep(mc, phc, integral_constant<int, 3>{}, s);
      };
      auto kloop = [&](auto mc) {
        for (int s = 0; s < nsteps; s += 3) {
          kstep(mc, integral_constant<int, 0>{}, s);
          if (s + 1 < nsteps) kstep(mc, integral_constant<int, 1>{}, s + 1);
          if (s + 2 < nsteps) kstep(mc, integral_constant<int, 2>{}, s + 2);
        }
      };
      if (MT == 2 && my_blocks == 2) kloop(integral_constant<int, MT>{});
      else if (my_blocks == 1) kloop(integral_constant<int, 1>{});
      else kloop(integral_constant<int, 0>{});
    } else {
    // what sub-step (s, t) requests: the weight rows of sub-step (s, t) + kDist (its K step clamped to the last
    // one: requests past the end fetch valid rows into a stage nobody reads again), and at t = 0 the x rows of
    // step s + 1.  Every sub-step issues the same number of loads, so the wait counts below are constants.
    auto request = [&](auto tc, auto pc, int s) {
      constexpr int t = decltype(tc)::value, par = decltype(pc)::value;
      constexpr int tn = (t + F::kDist) % NT, ds = (t + F::kDist) / NT;
      constexpr int target = NT == 1 ? (par + ds) % 2 : tn;
      ld.b_soff = (unsigned)block_of(tn) * 32 * hb + (unsigned)min(s + ds, nsteps - 1) * (unsigned)(BK * sizeof(bf16_t));
      ld.b_dst = stage(std::integral_constant<int, target>{});
      ld.a_soff = (unsigned)min(s + 1, nsteps - 1) * (unsigned)(BK * sizeof(bf16_t));
      ld.a_dst = par ? A0 : A1;
    };
    // prologue: the first kDist sub-steps' weight rows and the x rows of step 0 (weight rows first: they do not wait
    // for the row indices)
#pragma unroll
    for (int q = 0; q < F::kBInstr; ++q)
      dma16_buf(ld.w_rsrc, ld.b_voff, (unsigned)block_of(0) * 32 * hb + q * ld.bstep, S0 + q * 512 * 8 + ld.wave_elems);
#pragma unroll
    for (int a = 0; a < F::kAInstr; ++a) dma16_buf(ld.x_rsrc, ld.a_voff[a], 0, A0 + a * 512 * 8 + ld.wave_elems);
    if constexpr (F::kDist == 2) {
#pragma unroll
      for (int q = 0; q < F::kBInstr; ++q)
        dma16_buf(ld.w_rsrc, ld.b_voff, (unsigned)block_of(1) * 32 * hb + q * ld.bstep, S1 + q * 512 * 8 + ld.wave_elems);   // sub-step (0, 1)
    }
    zero_acc();
    auto substep = [&](auto mc, auto tc, auto pc, int s) {
      constexpr int nmt = decltype(mc)::value;           // M tiles of this wave that hold rows
      constexpr int t = decltype(tc)::value, par = decltype(pc)::value;
      constexpr int cur = NT == 1 ? par : t;
      // loads still allowed in flight: those of the sub-steps after the one whose stage is read now
      if constexpr (F::kDist == 1) sync_keep_loads<0>();
      else if constexpr (t == 1) sync_keep_loads<F::kBInstr + F::kAInstr>();     // the sub-step before (t = 0) also requested x rows
      else sync_keep_loads<F::kBInstr>();
      const bf16_t* a0 = (par ? A1 : A0) + (mbase + n) * BK + pos0;
      const bf16_t* b0 = stage(std::integral_constant<int, cur>{}) + n * BK;
      request(tc, pc, s);
      const SubIssuer<F, t == 0> issuer{ld};
      if constexpr (nmt > 0)
        stripe_step<nmt, 2, BK, true, 2 * NT, t, NT>(acc, a0, 32 * BK, b0, pos0, frag_row, issuer, true, 0, nullptr);
      else
        issue_some<0, SubIssuer<F, t == 0>::kInstr>(issuer, 0, nullptr);   // its share of the requests all the same
    };
    // one copy of the K loop per number of M tiles with rows, chosen once: a choice inside the loop would meet at
    // every sub-step with all 192 accumulator registers alive
    auto kloop = [&](auto mc) {
      for (int s = 0; s < nsteps; s += 2) {                                       // H / BK is even
        substep(mc, integral_constant<int, 0>{}, integral_constant<int, 0>{}, s);
        if constexpr (NT > 1) substep(mc, integral_constant<int, 1>{}, integral_constant<int, 0>{}, s);
        if constexpr (NT > 2) substep(mc, integral_constant<int, 2>{}, integral_constant<int, 0>{}, s);
        substep(mc, integral_constant<int, 0>{}, integral_constant<int, 1>{}, s + 1);
        if constexpr (NT > 1) substep(mc, integral_constant<int, 1>{}, integral_constant<int, 1>{}, s + 1);
        if constexpr (NT > 2) substep(mc, integral_constant<int, 2>{}, integral_constant<int, 1>{}, s + 1);
      }
    };
    if (MT == 2 && my_blocks == 2) kloop(integral_constant<int, MT>{});
    else if (my_blocks == 1) kloop(integral_constant<int, 1>{});
    else kloop(integral_constant<int, 0>{});
      }
  }
  wait_loads_and_sync();                   // every transfer has landed and every wave is done with the stages

  if constexpr (MODE == 3) {
    float* pre = reinterpret_cast<float*>(preact);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int m = mbase + mt * 32 + n;
      if (mt >= my_blocks || m >= rows) continue;
      float* prow = pre + (size_t)(row0 + m) * (2 * row_i) + cb * I + 4 * (lane >> 5);
#pragma unroll
      for (int j = 0; j < 2 * NT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int half = j / NT, col = (wn * NT + block_of(j % NT)) * 32 + 8 * q;
          *reinterpret_cast<floatx4*>(prow + half * row_i + col) =
              floatx4{acc[mt][j][4 * q], acc[mt][j][4 * q + 1], acc[mt][j][4 * q + 2], acc[mt][j][4 * q + 3]};
        }
    }
    return;
  }
  if constexpr (MODE != 0) {
    // gate half, then up half: accumulators -> the stages in the activation layout (stage t = columns [128 t, 128 t + 128)
    // of the half, granule c of row m at c ^ (m & 15)) -> whole 256-byte row segments to memory
    const int hh = lane >> 5;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        if (mt >= my_blocks) continue;
        const int m = mbase + mt * 32 + n;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const int tile32 = wn * NT + block_of(j);
          bf16_t* hrow = slice(tile32 >> 2) + m * 128 + 4 * hh;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            bf16x4 hv;
#pragma unroll
            for (int r = 0; r < 4; ++r) hv[r] = (bf16_t)acc[mt][half * NT + j][4 * q + r];
            const int c = (tile32 & 3) * 4 + q;
            *reinterpret_cast<bf16x4*>(hrow + (c ^ (m & 15)) * 8) = hv;
          }
        }
      }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const bf16_t* from = slice(t);
        for (int g = tid; g < BM * 16; g += 512) {
          const int m = g >> 4, pos = g & 15;
          if (m < rows)
            *reinterpret_cast<u32x4*>(preact + (size_t)(row0 + m) * (2 * row_i) + half * row_i + cb * I + t * 128 + ((pos ^ (m & 15)) * 8)) =
                *reinterpret_cast<const u32x4*>(from + m * 128 + pos * 8);
        }
      }
      __syncthreads();                     // the stages are free for the other half
    }
    if constexpr (MODE == 1) return;
  }

  // ---- phase 2: Radial NormSiLU (moe.py:87-92), activations to LDS ----
  // The accumulators are transposed (lane = row mbase + 32*mt + n, register i = column acc_row(i, lane) of
  // its 32-column tile), so a row's sum of gate^2 is a sum over this lane's registers, the lane with the
  // other half of the columns (lane ^ 32) and the four N waves; and every lane owns runs of four
  // consecutive columns, which leave as one 8-byte LDS write.
  const int hh = lane >> 5;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    float part[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      part[j] = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) part[j] = fmaf(acc[mt][j][i], acc[mt][j][i], part[j]);
    }
    float sq = 0.f;
#pragma unroll
    for (int b = 0; b < NT; ++b) {            // in column order, whichever block the tile began with
      float v = part[0];
#pragma unroll
      for (int j = 1; j < NT; ++j) v = block_of(j) == b ? part[j] : v;
      sq += v;
    }
    const Pair halves = lanes32(sq);
    sq = halves.a + halves.b;
    if (hh == 0) ssq[wn * BM + mbase + mt * 32 + n] = sq;
  }
  __syncthreads();
  if (tid < BM) {
    const float p = radial_exponent(theta, e, act);                                   // moe.py:89
    const float ms = ((ssq[tid] + ssq[BM + tid]) + ssq[2 * BM + tid]) + ssq[3 * BM + tid];
    radial_row_scalars(ms, I, p, act, rinv_s[tid], gain_s[tid]);                      // 1/r and r^p, moe.py:88-89
    const int slot = SCAN ? slot_s[min(tid, rows - 1)] : perm_slot[row0 + min(tid, rows - 1)];
    if constexpr (SCAN == 0) slot_s[tid] = slot;
    w_s[tid] = w[slot];
  }
  __syncthreads();
  // phase 3 streams w_down through registers; its first K blocks are requested here, between the two M tiles of
  // the activation: the accumulators of the first tile are dead by then and make room, and the loads fly during
  // the rest of the activation arithmetic
  constexpr int KB = I / 64;                 // 128-byte K blocks
  const size_t tile_stride = (size_t)16 * I;
  const bf16_t* wp = wd + ((size_t)e * H + wave * (16 * CT) + (lane >> 2)) * I + (lane & 3) * 8;
  constexpr int D = KB > 3 ? 3 : KB - 1;      // K blocks requested ahead of the one being multiplied
  constexpr int NB = D + 1;
  WBlock<CT> wb[NB];
  {
    // stage t holds activation columns [128t, 128t + 128) of all 128 rows, [128][128], granules swizzled
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if (mt == MT - 1) {
#pragma unroll
        for (int d = 0; d < D; ++d) load_wblock<CT>(wb[d], wp, tile_stride, d);
      }
      if (mt >= my_blocks) continue;          // a block without rows: nobody reads its activations
      const int m = mbase + mt * 32 + n;
      const float rinv = rinv_s[m];
      const float nrl = -1.44269504f * rinv, rg = rinv * gain_s[m];            // per-row constants folded once
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int tile32 = wn * NT + block_of(j);      // 32-column tile of the activation row: slice tile32 / 4, granules (tile32 % 4) * 4 + q
        bf16_t* hrow = slice(tile32 >> 2) + m * 128 + 4 * hh;
#pragma unroll
        for (int q = 0; q < 4; ++q) {        // columns tile32*32 + 8*q + 4*hh + 0..3: half of a granule
          bf16x4 hv;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float g = acc[mt][j][4 * q + r];
            const float sg = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(g * nrl));   // sigmoid(g/r)
            hv[r] = (bf16_t)(g * rg * sg * acc[mt][NT + j][4 * q + r]);                // SiLU(g/r) r^p up
          }
          const int c = (tile32 & 3) * 4 + q;
          *reinterpret_cast<bf16x4*>(hrow + (c ^ (m & 15)) * 8) = hv;
        }
      }
    }
  }
  __syncthreads();                         // the activation tile is complete

  // ---- phase 3: down projection, routing weight, scatter to slot order (moe.py:92-93) ----
  const int nblk = H / F::BN2;
  for (int nb = 0; nb < nblk; ++nb)
    down_block<F, CT, KB, D, NB, 2 * kBlocks>(slice, wb, wp, tile_stride, nb + 1 < nblk, nb * F::BN2, w_s, slot_s, rows, A0, A1, H, yw,
                                                  F32_ROWS);
  };   // body
  if (MTP == 2 && nblocks == 4) body(std::integral_constant<int, 2 * MTP>{});
  else if (MTP == 2 && nblocks == 3) body(std::integral_constant<int, 2 * MTP - 1>{});
  else if (nblocks == 2) body(std::integral_constant<int, 2>{});
  else body(std::integral_constant<int, 1>{});
}


// The second half of the fused kernel on its own, for calls with fewer tiles than CUs: the activations of a tile from the fp32
// pre-activations [S, 2I] that the first half left (phase 2), and ONE block of output columns (phase 3), so that an expert's
// w_down passes through H / BN2 CUs at once.  Every one of them computes the tile's activations again, one wave per row, while
// its first weights are on their way.  With `preact`, the workgroups of column block 0 also leave the pre-activations rounded to
// bf16, for a backward pass.
template <int NT, int CT, int MTP>
__global__ __launch_bounds__(512) void down_act_kernel(const float* __restrict__ gu, const bf16_t* __restrict__ wd,
                                                       const float* __restrict__ theta, const float* __restrict__ w,
                                                       const int32_t* __restrict__ offsets, const int32_t* __restrict__ perm_slot,
                                                       int H, int E, int act, void* __restrict__ yw, int f32_rows,
                                                       bf16_t* __restrict__ preact) {
  using F = FusedShape<NT, CT, MTP>;
  constexpr int BM = F::BM, I = F::I;
  __shared__ __attribute__((aligned(16))) bf16_t acts[NT * BM * 128];
  __shared__ __attribute__((aligned(16))) bf16_t O0[F::kOutElems];
  __shared__ __attribute__((aligned(16))) bf16_t O1[F::kOutElems];
  __shared__ float w_s[BM];
  __shared__ int slot_s[BM];
  const int nblk = H / F::BN2;
  const TileMap tm = make_tile_map(offsets, E, BM);
  const int flat = xcd_tile(blockIdx.x, tm.total * nblk);
  if (flat >= tm.total * nblk) return;
  const int tile = flat / nblk, nb = flat - tile * nblk;
  int e, row0, rows;
  find_tile(tm, tile, e, row0, rows);
  e = __builtin_amdgcn_readfirstlane(e);
  row0 = __builtin_amdgcn_readfirstlane(row0);
  rows = __builtin_amdgcn_readfirstlane(rows);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  constexpr int KB = I / 64;                 // every K block of the weights is requested up front
  const size_t tile_stride = (size_t)16 * I;
  const bf16_t* wp = wd + ((size_t)e * H + nb * F::BN2 + wave * (16 * CT) + (lane >> 2)) * I + (lane & 3) * 8;
  WBlock<CT> wb[KB];
  // a wave's rows are wave, wave + 8, ...; the first kRowsAhead of them are requested ahead of the weights, which a CU would
  // otherwise serve first
  constexpr int kRowsAhead = NT == 4 ? 6 : 8;            // (what the registers hold beside I = 512 worth of weights)
  const bool live = lane * 8 < I;
  floatx4 g[kRowsAhead][2], u[kRowsAhead][2];
  auto request = [&](int m0) {
#pragma unroll
    for (int i = 0; i < kRowsAhead; ++i) {
      const float* src = gu + (size_t)(row0 + min(m0 + 8 * i, rows - 1)) * 2 * I + lane * 8;
      if (live && m0 + 8 * i < rows) {
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          g[i][v] = *reinterpret_cast<const floatx4*>(src + 4 * v);
          u[i][v] = *reinterpret_cast<const floatx4*>(src + I + 4 * v);
        }
      }
    }
  };
  request(wave);
  if (tid < BM) {
    const int slot = perm_slot[row0 + min(tid, rows - 1)];
    slot_s[tid] = slot;
    w_s[tid] = w[slot];
  }
  const float p = radial_exponent(theta, e, act);                                   // moe.py:89
#pragma unroll
  for (int d = 0; d < KB; ++d) load_wblock<CT>(wb[d], wp, tile_stride, d);
  for (int m0 = wave; m0 < rows; m0 += 8 * kRowsAhead) {
    if (m0 > wave) request(m0);
#pragma unroll
    for (int i = 0; i < kRowsAhead; ++i) {
      const int m = m0 + 8 * i;
      if (m >= rows) break;
      float ss = 0.f;
      if (live) {
#pragma unroll
        for (int q = 0; q < 8; ++q) ss = fmaf(g[i][q >> 2][q & 3], g[i][q >> 2][q & 3], ss);
      }
      ss = wave_sum(ss);
      float rinv, gain;
      radial_row_scalars(ss, I, p, act, rinv, gain);                                // 1/r and r^p, moe.py:88-89
      const float nrl = -1.44269504f * rinv, rg = rinv * gain;
      if (live) {
        bf16x8 h;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const float gq = g[i][q >> 2][q & 3];
          const float sg = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(gq * nrl));
          h[q] = (bf16_t)(gq * rg * sg * u[i][q >> 2][q & 3]);                      // SiLU(g/r) r^p up
        }
        if constexpr (NT < 4) {              // (a state-keeping forward has I <= 384)
          if (preact != nullptr && nb == 0) {
            bf16x8 gb, ub;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
              gb[q] = (bf16_t)g[i][q >> 2][q & 3];
              ub[q] = (bf16_t)u[i][q >> 2][q & 3];
            }
            bf16_t* dst = preact + (size_t)(row0 + m) * 2 * I + lane * 8;
            *reinterpret_cast<bf16x8*>(dst) = gb;
            *reinterpret_cast<bf16x8*>(dst + I) = ub;
          }
        }
        *reinterpret_cast<bf16x8*>(acts + (lane >> 4) * (BM * 128) + m * 128 + (((lane & 15) ^ (m & 15)) << 3)) = h;
      }
    }
  }
  __syncthreads();
  auto slice = [&](int i) -> const bf16_t* { return acts + i * (BM * 128); };
  auto body = [&](auto nblocks_c) {
    down_block<F, CT, KB, KB, KB, 2 * decltype(nblocks_c)::value>(slice, wb, wp, tile_stride, false, nb * F::BN2, w_s, slot_s, rows, O0,
                                                                 O1, H, yw, f32_rows != 0);
  };
  const int nblocks = (rows + 31) >> 5;
  if (MTP == 2 && nblocks == 4) body(std::integral_constant<int, 2 * MTP>{});
  else if (MTP == 2 && nblocks == 3) body(std::integral_constant<int, 2 * MTP - 1>{});
  else if (nblocks == 2) body(std::integral_constant<int, 2>{});
  else body(std::integral_constant<int, 1>{});
}

// slots a thread of a SCAN kernel looks at, 512 threads; MOST: slots of the largest call that finds its rows itself
template <int MOST, typename Launch>
void scan_variant(int S, Launch launch) {
  static_assert(MOST <= 32 * 512, "slots of a scan");
  if constexpr (MOST > 16 * 512) {
    if (S > 16 * 512) { launch(std::integral_constant<int, 32>()); return; }
  }
  if constexpr (MOST > 8 * 512) {
    if (S > 8 * 512) { launch(std::integral_constant<int, 16>()); return; }
  }
  launch(std::integral_constant<int, 8>());
}

template <int NT, int CT, int MT>
void launch_fused_t(const bf16_t* x, const bf16_t* wgu, const bf16_t* wd, const float* theta, const float* w,
                    const int32_t* offsets, const int32_t* perm_slot, const int32_t* perm_token, int S, int H, int E,
                    int act, unsigned x_bytes, void* yw, bool f32_rows, bf16_t* preact, const ScanArgs& scan, hipStream_t s) {
  const int grid = round_tiles_most(S, E, 64 * MT);
  auto launch = [&](auto mode, auto f32, auto per) {
    constexpr int MODE = decltype(mode)::value, SCAN = decltype(per)::value;
    hipLaunchKernelGGL((experts_fused_kernel<NT, CT, MODE, MT, SCAN, decltype(f32)::value>), dim3(grid), dim3(512), 0, s, x, wgu, wd, theta,
                       w, offsets, perm_slot, perm_token, H, E, act, x_bytes, yw, preact, 1, scan);
  };
  const std::false_type bf16_rows;
  const bool find = scan.idx != nullptr;
  const std::integral_constant<int, 0> permuted;
  if constexpr (NT < 4) {                    // (a state-keeping forward has I <= 384)
    if (preact != nullptr) {
      const std::integral_constant<int, 2> train;
      if (find) scan_variant<kScanSlots>(S, [&](auto per) { launch(train, bf16_rows, per); });
      else launch(train, bf16_rows, permuted);
      return;
    }
  }
  const std::integral_constant<int, 0> forward;
  if (f32_rows) {                            // (kernels of their own: as a branch of the usual ones it cost those 0.3 to 0.5 % at I = 512)
    static_assert(kStreamMaxSlots <= 8 * 512, "calls that may stream fit the shortest scan");
    if (find) launch(forward, std::true_type(), std::integral_constant<int, 8>());
    else launch(forward, std::true_type(), permuted);
  } else if (find) {
    scan_variant<NT == 4 ? kScanSlots / 2 : kScanSlots>(S, [&](auto per) { launch(forward, bf16_rows, per); });
  } else {
    launch(forward, bf16_rows, permuted);
  }
}

}  // namespace

template <int NT>
void launch_down_act_nt(const float* gu, const bf16_t* wd, const float* theta, const float* w, const int32_t* offsets,
                        const int32_t* perm_slot, int S, int H, int E, int act, void* yw, bool f32_rows, bf16_t* preact,
                        hipStream_t s) {
  auto launch = [&](auto mt, auto ct) {
    constexpr int MT = decltype(mt)::value, CT = decltype(ct)::value;
    const int tiles = S / (64 * MT) + E < S ? S / (64 * MT) + E : S;
    const int grid = ((tiles * (H / (128 * CT)) + 7) & ~7) + 8;
    hipLaunchKernelGGL((down_act_kernel<NT, CT, MT>), dim3(grid), dim3(512), 0, s, gu, wd, theta, w, offsets, perm_slot, H, E, act, yw,
                       (int)f32_rows, preact);
  };
  // 64-row tiles while they and their column blocks leave no workgroup waiting for a CU: shorter, and more of them pull weights
  using std::integral_constant;
  const bool two = H % 256 == 0;
  const bool tall = (S / 64 + E / 2) * (H / (two ? 256 : 128)) > 256;
  if constexpr (NT < 4) {
    if (tall) {
      if (two) launch(integral_constant<int, 2>{}, integral_constant<int, 2>{}); else launch(integral_constant<int, 2>{}, integral_constant<int, 1>{});
      return;
    }
  }
  if (two) launch(integral_constant<int, 1>{}, integral_constant<int, 2>{}); else launch(integral_constant<int, 1>{}, integral_constant<int, 1>{});
}

// I = 512 has a kernel of its own behind the calls that find their rows themselves.  H = 1024, E = 64, k = 8, layer, this kernel -> that one, the
// same weights again and again, in turn on one card: 74.2 -> 72.1 us (T = 1025), 77.2 -> 74.6 (1500), 130.7 -> 122.3 (2047), 145.6 -> 137.5 (3001),
// 264 -> 245 (6000), 582 -> 551 (16,000); H = 768, E = 32, k = 4: 107.6 -> 102.3 (4100); H = 640, E = 16, k = 2: 57.1 -> 53.9 (4200); H = 512, E = 8,
// k = 1: 48.9 -> 48.9 (9000).  Cards differ, as the clock their power leaves does: T = 3001 on others 150.0 -> 143.6, 149.5 -> 144.6, 140.4 -> 139.3.
template <int NT>
void launch_fused_nt(const bf16_t* x, const bf16_t* wgu, const bf16_t* wd, const float* theta, const float* w,
                     const int32_t* offsets, const int32_t* perm_slot, const int32_t* perm_token, int S, int H, int E,
                     int act, unsigned x_bytes, void* yw, bool f32_rows, bf16_t* preact, const ScanArgs& scan, hipStream_t s) {
  constexpr int MT = NT == 4 ? 1 : 2;
  auto launch = [&](auto ct) {
    if constexpr (NT == 4) {
      if (S > kScanSlots / 2) {
        static_assert(kStreamMaxSlots <= kScanSlots / 2, "fp32 rows go with the few rows of a streaming call");
        launch_wide_t<decltype(ct)::value>(x, wgu, wd, theta, w, offsets, perm_slot, perm_token, S, H, E, act, x_bytes, yw, s);
        return;
      }
    }
    launch_fused_t<NT, decltype(ct)::value, MT>(x, wgu, wd, theta, w, offsets, perm_slot, perm_token, S, H, E, act, x_bytes, yw, f32_rows,
                                               preact, scan, s);
  };
  // (blocks of 256 columns leave room for the third x buffer of the deeper ring where I is not 384)
  if constexpr (NT != 4) {
    if (H % 384 == 0 && (NT == 3 || H % 256 != 0)) {
      launch(std::integral_constant<int, 3>{});
      return;
    }
  }
  if (H % 256 == 0) launch(std::integral_constant<int, 2>{});
  else launch(std::integral_constant<int, 1>{});
}

template <int NT, int MODE>
void launch_raw_nt(const bf16_t* x, const bf16_t* wgu, const int32_t* offsets, const int32_t* perm_token, int S, int H, int E,
                   unsigned x_bytes, bf16_t* gu, int column_blocks, hipStream_t s, const ScanArgs& scan) {
  constexpr int MT = NT == 4 ? 1 : 2;
  const int tiles = S / (64 * MT) + E < S ? S / (64 * MT) + E : S;
  const int grid = MODE == 3 || column_blocks > 1 ? ((tiles * column_blocks + 7) & ~7) + 8 : round_tiles_most(S, E, 64 * MT);
  if constexpr (MODE == 3) {
    if (scan.idx != nullptr) {
      scan_variant<kSplitSlots>(S, [&](auto per) {
        hipLaunchKernelGGL((experts_fused_kernel<NT, 1, MODE, MT, decltype(per)::value>), dim3(grid), dim3(512), 0, s, x, wgu, nullptr,
                           nullptr, nullptr, nullptr, nullptr, nullptr, H, E, 0, x_bytes, nullptr, gu, column_blocks, scan);
      });
      return;
    }
  }
  hipLaunchKernelGGL((experts_fused_kernel<NT, 1, MODE, MT>), dim3(grid), dim3(512), 0, s, x, wgu, nullptr, nullptr, nullptr,
                     offsets, nullptr, perm_token, H, E, 0, x_bytes, nullptr, gu, column_blocks, scan);
}

}  // namespace bibo
