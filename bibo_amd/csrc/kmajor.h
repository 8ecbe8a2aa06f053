// Grouped GEMMs whose operands are contiguous ACROSS the contraction instead of along it ("K-major": element (k, n)
// at k * ld + n), for the backward pass on gfx950.  The two weight tensors are stored [E, 2I, H] and [E, H, I]; the
// forward pass contracts along their last dimension, the input gradients contract along the middle one, and the
// weight gradients contract along the ROWS of row-major activations.  Instead of transposed copies in memory, a
// K-major operand goes to LDS as it lies (LDS-DMA, 64 k rows x 128 n per sub-tile) and the MFMA fragments are read
// with ds_read_b64_tr_b16, which hands a lane four consecutive k of one n:
//   within a group of 16 lanes, lane r addresses 8 bytes (4 elements) M[r][0..3], and lane j receives
//   M[j / 4 + 4 i][j % 4] for i = 0..3.  With lane r pointing at (k0 + r / 4, n0 + 4 (r % 4)) the group covers a
//   4 (k) x 16 (n) block and lane j ends up with (k0 .. k0 + 3, n0 + j).
// Two such reads give the 8 consecutive k of an MFMA operand lane.
#pragma once

#include "stripe.h"

namespace bibo {
namespace {

typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;

constexpr int kKS = 32;                 // k rows per LDS stage
constexpr int kRing = 4;                // stages in LDS: one being multiplied, two on their way, one being requested
constexpr int kSubW = 128;              // n elements per sub-tile row (256 bytes: whole 128-byte lines per DMA row)
constexpr int kWaveElems = 4 * kSubW + 8;      // what one wave of an LDS-DMA instruction fills, 1 KB, and 16 bytes of nothing
constexpr int kSubElems = kKS / 4 * kWaveElems;    // a sub-tile: one LDS-DMA instruction of the 512 threads
constexpr int kATile = 128 * kKS;       // row-major operand tile, 128 rows: 8 KB as well

// LDS layout of a K-major sub-tile [32 k][128 n]: 16-byte granule G of row k sits at position G ^ ((k & 3) << 2).
// The four k rows that 16 lanes of a transposed read touch then lie in four different 64-byte quarters of the 256-byte bank
// period.  The 16 lanes beside them read eight rows on, which the gap behind every four rows moves to the other half of the quarters: no
// bank conflicts (4.0 cycles a read without the gaps, 2.4 with them).  Thread t of the fill writes row t / 16, position t % 16, and therefore
// fetches granule (t % 16) ^ (((t / 16) & 3) << 2) of that row.
__device__ __forceinline__ int kfill_granule(int tid) { return (tid & 15) ^ (((tid >> 4) & 3) << 2); }

// Fill one sub-tile: `row` = this thread's row (tid / 16) of the stage, already offset to the sub-tile's first
// column and to this thread's granule.
__device__ __forceinline__ void kfill_subtile(const bf16_t* row, bf16_t* sub) {
  dma16(row, sub + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * kWaveElems);
}

// Per-lane element offset, inside a sub-tile, of the first transposed read of the 16 (n) x 32 (k) fragment whose first column is
// nbase (a multiple of 16): the four k behind those it hands a lane are kWaveElems elements on.
__device__ __forceinline__ int kfrag_offset(int lane, int nbase) {
  const int r = lane & 15, krow = 8 * (lane >> 4) + (r >> 2);
  const int n = nbase + 4 * (r & 3);
  const int pos = (n >> 3) ^ ((r >> 2) << 2);                  // (k & 3) == r / 4 for both reads of the fragment
  return (krow >> 2) * kWaveElems + (krow & 3) * kSubW + pos * 8 + (n & 4);
}

// The fragment of a stage: lane (n = lane % 16, g = lane / 16) gets k = 8 g .. + 8 of column nbase + n.
__device__ __forceinline__ bf16x8 kfrag_read(const bf16_t* sub, int off) {
  const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(sub + off));
  const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(sub + off + kWaveElems));
  typedef short v8i16 __attribute__((ext_vector_type(8)));
  const v8i16 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return __builtin_bit_cast(bf16x8, v);
}

// 16 x 16 x 32 and not 32 x 32 x 16: the chip's clock gives way to the power of its matrix pipes, and on operands that are not zeros a loop of
// nothing but the one runs at 1.97 GHz (2.0 PFLOP/s), of the other at 1.75 (1.78).  ROW_LANES: operands swapped, a lane ends up with columns of ONE row of A; else with rows of one row of B.
template <bool ROW_LANES>
__device__ __forceinline__ floatx4 mfma_pair(bf16x8 a, bf16x8 b, floatx4 c) {
  return ROW_LANES ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, c, 0, 0, 0) : __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// The multiplication of a wave's RT x CT tiles of 16 x 16 as one software pipeline over the row tiles of ALL stages (a stage is one MFMA
// deep): a row fragment is read two row tiles ahead of its MFMAs, the column fragments are held for the whole stage, and in its last row
// tile the next stage's take their places one by one behind their last MFMAs.  Two row tiles before a stage ends every row fragment of
// it has been read and its column fragments are held, so that is where the waves meet (`meet`: the next stage has landed, the one just
// read may be filled again), and 2 CT MFMAs run while the next stage's first fragments are on their way.  The order is pinned: left to
// itself the compiler reads a fragment into the registers of the last one and waits for it on the spot.  The loop over a ring's stages has
// no other way in or out of its middle, because where two ways meet the compiler waits for every transfer before the next LDS read.
// T = 8192, H = 768, I = 384, E = 64, k = 6, best times: dh' 41.0 -> 35.0 us (pinned order 40.0, with these MFMAs 37.0), backward_gemms_kernel
// 195 -> 163.  In traces of training passes on several cards they average 39 to 41 and 181 to 199, cold first pass included.
template <int RT, int CT, bool ROW_LANES>
struct StagePipe {
  static constexpr int NA = RT % 3 == 2 ? 3 : 4;           // row fragments in flight; divides the row tiles of a ring
  bf16x8 af[NA], bfr[CT];

  template <typename ReadA, typename ReadB>
  __device__ __forceinline__ void begin(ReadA read_a, ReadB read_b) {
#pragma unroll
    for (int j = 0; j < CT; ++j) bfr[j] = read_b(j);
    af[0] = read_a(0);
    af[1] = read_a(1);
    __builtin_amdgcn_sched_barrier(0);
  }
  // Transfer q of a refill is issued q row tiles behind the meeting that allows it, the last ones together where a stage has fewer.
  static constexpr int slot(int q) { return q < RT ? q : RT - 1; }
  // FIRST: running number of the stage's first row tile, mod NA.  refill(q): transfer q into the buffer of this stage;
  // refill_before(q): of the stage before.
  template <int FIRST, int OPS, typename Meet, typename ReadA, typename NextA, typename NextB, typename Refill, typename Before>
  __device__ __forceinline__ void stage(floatx4 (&acc)[RT][CT], Meet meet, ReadA read_a, NextA next_a, NextB next_b, Refill refill,
                                        Before refill_before) {
#pragma unroll
    for (int p = 0; p < RT; ++p) {
      if (p == RT - 2) {
        meet();
        __builtin_amdgcn_sched_barrier(0);
      }
      af[(FIRST + p + 2) % NA] = p < RT - 2 ? read_a(p + 2) : next_a(p + 2 - RT);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        acc[p][j] = mfma_pair<ROW_LANES>(af[(FIRST + p) % NA], bfr[j], acc[p][j]);
        if (p == RT - 1) {
          __builtin_amdgcn_sched_barrier(0);
          bfr[j] = next_b(j);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (j == 0) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int q = 0; q < OPS; ++q) {
            if (slot(q) != (p + 2) % RT) continue;
            if (p >= RT - 2) refill(q); else refill_before(q);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
};

// Row-major operand tile [128 rows][32 k]: granule c of row r at c ^ row_swizzle(r).  A 16-byte LDS read is served 16 lanes at a time: lanes
// 0-3, 12-15, 20-27 together, then 4-11, 16-19, 28-31, and the other half alike; lane (row n, granule g) of a 16-row fragment meets no
// other on a bank (4.3 cycles a read; 8.0 with (r >> 2) & 3).
__device__ __forceinline__ int row_swizzle(int r) {
  const int q = (r >> 2) & 3;
  return ((q ^ q >> 1) & 1) << 1 | q >> 1;                       // 0, 2, 3, 1
}
// Thread t of the fill writes row t / 4, position t % 4.  `row` = that row's K extent, already
// offset to the stage's first k and to this thread's granule (afill_granule).
__device__ __forceinline__ int afill_granule(int tid) { return (tid & 3) ^ row_swizzle(tid >> 2); }
__device__ __forceinline__ void afill(const bf16_t* row, bf16_t* tile) {
  dma16(row, tile + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * 64 * 8);
}

// The stages form a ring, each a __shared__ variable of its own (the compiler orders an LDS-DMA transfer against later reads of the same
// variable with a full wait).  Where the waves meet in stage i (StagePipe), the transfers of stage i + 1 have landed, those of the R - 2
// stages behind it may stay in flight (loads complete in order), and stage i + R is requested into the buffer that stage i has just been
// read from.  Every stage issues the same number of transfers (a request past the last stage repeats the last one), so the wait count is a
// constant.

// The stages of a ring, a row operand's and a column operand's each, as a kernel declares them; the fourth ones only for rings of four.
struct Ring {
  bf16_t *a0, *a1, *a2, *a3, *b0, *b1, *b2, *b3;
  template <int I> __device__ __forceinline__ bf16_t* a() const { return I == 0 ? a0 : I == 1 ? a1 : I == 2 ? a2 : a3; }
  template <int I> __device__ __forceinline__ bf16_t* b() const { return I == 0 ? b0 : I == 1 ? b1 : I == 2 ? b2 : b3; }
};

// ---- input gradients: out[dst(r), n] = sum_k A[src(r), k] W[e][k, n] for the rows r of expert e ----------------
// A row-major (K contiguous), W K-major as stored: [K, N] per expert.  src(r) = a_index[r] (GATHER) or r; dst(r) =
// out_index[r] (SCATTER) or r.  Workgroup = 64 MT rows x 128 NTW columns, 2 x 4 waves, 16x16x32 MFMA, operands swapped
// so that a lane owns one output row.  K is a multiple of 128.  MT = 2: 128-row tiles, ring of four stages.  MT = 4:
// 256-row tiles for experts with many rows - an expert's weights then pass through LDS once per 256 rows instead of
// once per 128; 192 accumulator registers and 40 KB stages, ring of three.  With the transfers or the LDS reads left out the tall tiles are
// 10 % faster, with neither (MFMAs alone) 14 %: they are bound by the matrix pipes at the clock these leave.
template <int MT, int NTW, bool GATHER, bool SCATTER>
__device__ __forceinline__ void dgrad_block(const Ring& ring, int* dst_s, int block, const bf16_t* __restrict__ A,
                                            const int32_t* __restrict__ a_index, const bf16_t* __restrict__ W,
                                            const int32_t* __restrict__ offsets, const int32_t* __restrict__ out_index, int K, int N, int E,
                                            int nblk_n, bf16_t* __restrict__ out) {
  static_assert(MT == 2 || MT == 4, "128- or 256-row tiles");
  constexpr int BM = 64 * MT, BN = kSubW * NTW;
  constexpr int R = MT == 4 ? 3 : kRing;                 // stages that fit LDS
  constexpr int kAOps = MT / 2;                          // 128-row blocks of the row operand
  constexpr int kOps = kAOps + NTW;                      // transfers per thread and stage

  const TileMap tm = make_tile_map(offsets, E, BM);
  const int total = tm.total * nblk_n;
  const int flat = xcd_tile(block, total);
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
  // fill side
  const bf16_t* arow[kAOps];
#pragma unroll
  for (int hb = 0; hb < kAOps; ++hb) {
    const int ar = row0 + min(hb * 128 + (tid >> 2), rows - 1);    // rows past the end re-read the last one
    arow[hb] = A + (size_t)(GATHER ? a_index[ar] : ar) * K + afill_granule(tid) * 8;
  }
  const int n0 = nb * BN;
  const bf16_t* wrow = W + (size_t)e * K * N + (size_t)(tid >> 4) * N + n0 + kfill_granule(tid) * 8;
  const int nstages = K / kKS;
  auto abuf = [&](auto bc) -> bf16_t* { return ring.template a<decltype(bc)::value>(); };
  auto bbuf = [&](auto bc) -> bf16_t* { return ring.template b<decltype(bc)::value>(); };
  // transfer q of a stage into buffer bc
  auto fill = [&](auto bc, int stage, int q) {
    const int k0 = min(stage, nstages - 1) * kKS;
    if (q < kAOps) afill(arow[q] + k0, abuf(bc) + q * kATile);
    else kfill_subtile(wrow + (size_t)k0 * N + (q - kAOps) * kSubW, bbuf(bc) + (q - kAOps) * kSubElems);
  };
  using std::integral_constant;
  auto fill_all = [&](auto bc, int stage) {
#pragma unroll
    for (int q = 0; q < kOps; ++q) fill(bc, stage, q);
  };
  fill_all(integral_constant<int, 0>{}, 0);
  fill_all(integral_constant<int, 1>{}, 1);
  if constexpr (R == 4) fill_all(integral_constant<int, 2>{}, 2);
  constexpr int kFirst = 2;                               // transfers that stage 0 does not issue for the one before it
#pragma unroll
  for (int q = 0; q < kFirst; ++q) fill(integral_constant<int, R - 1>{}, R - 1, q);

  constexpr int RT = 2 * MT, CT = 2 * NTW;                // a wave's tiles of 16 x 16
  floatx4 acc[RT][CT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[rt][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  // fragment side.  A: lane (n, g) reads granule g of row mbase + 16 rt + n.  W: wave wn's tile j is columns (wn CT + j) 16 of the block =
  // sub-tile (wn CT + j) / 8, column ((wn CT + j) % 8) 16 inside it.
  const int n = lane & 15, g4 = lane >> 4;
  const int mbase = wm * MT * 32;
  const int aoff = (mbase + n) * kKS + (g4 ^ row_swizzle(n)) * 8;
  int boff[CT / 2];                                        // of the even tiles: an odd one is 16 elements on
#pragma unroll
  for (int t = 0; t < CT / 2; ++t) {
    const int t16 = wn * CT + 2 * t;
    boff[t] = (t16 >> 3) * kSubElems + kfrag_offset(lane, (t16 & 7) * 16);
  }
  auto read_a = [&](auto bc, int rt) { return *reinterpret_cast<const bf16x8*>(abuf(bc) + aoff + rt * 16 * kKS); };
  auto read_b = [&](auto bc, int j) { return kfrag_read(bbuf(bc) + (j & 1) * 16, boff[j >> 1]); };
  using Pipe = StagePipe<RT, CT, true>;
  Pipe pipe;
  sync_keep_loads<(R - 2) * kOps + kFirst>();
  {
    const integral_constant<int, 0> b0;
    pipe.begin([&](int rt) { return read_a(b0, rt); }, [&](int j) { return read_b(b0, j); });
  }
  auto step = [&](auto bc, int stage) {
    constexpr int b = decltype(bc)::value;
    const integral_constant<int, (b + 1) % R> nc;
    const integral_constant<int, (b + R - 1) % R> pc;
    pipe.template stage<b * RT % Pipe::NA, kOps>(
        acc, [&]() { sync_keep_loads<(R - 2) * kOps>(); }, [&](int rt) { return read_a(bc, rt); }, [&](int rt) { return read_a(nc, rt); },
        [&](int j) { return read_b(nc, j); }, [&](int q) { fill(bc, stage + R, q); }, [&](int q) { fill(pc, stage + R - 1, q); });
  };
  int i = 0;
  for (; i + R <= nstages; i += R) {
    step(integral_constant<int, 0>{}, i);
    step(integral_constant<int, 1>{}, i + 1);
    step(integral_constant<int, 2>{}, i + 2);
    if constexpr (R == 4) step(integral_constant<int, 3>{}, i + 3);
  }
  if (i < nstages) step(integral_constant<int, 0>{}, i);
  if (i + 1 < nstages) step(integral_constant<int, 1>{}, i + 1);
  if constexpr (R == 4) if (i + 2 < nstages) step(integral_constant<int, 2>{}, i + 2);
  wait_loads_and_sync();                 // the repeated requests of the last steps have landed; every wave is done reading

  // Epilogue (accumulators transposed: lane = row, four consecutive columns per register quad): 32 rows at a time
  // through a wave-private LDS tile, out as 16-byte row segments.
  constexpr int kOutCols = NTW * 32;
  constexpr int kOutStride = kOutCols + 8;          // +16 bytes staggers the rows over the banks
  static_assert(3 * 32 * kOutStride <= NTW * kSubElems, "output staging does not fit a weight stage");
  bf16_t* otile = ring.b0;               // three waves per stage buffer
  if (wave >= 6) otile = ring.b2; else if (wave >= 3) otile = ring.b1;
  otile += (wave % 3) * (32 * kOutStride);
  constexpr int kGranPerRow = kOutCols / 8;
  const int colbase = n0 + wn * kOutCols;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        bf16x4 hv;
#pragma unroll
        for (int r = 0; r < 4; ++r) hv[r] = (bf16_t)acc[2 * mt + q][j][r];
        *reinterpret_cast<bf16x4*>(otile + (16 * q + n) * kOutStride + j * 16 + 4 * g4) = hv;
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

// The compiler lays LDS variables out by alignment: the row operand's stages come first, so that their addresses fit the 16-bit offset of a
// read and need no registers of their own.
constexpr int kLowLds = 64;

// Elements of a stage's row and column operand.
constexpr int ring_a(int MT) { return MT / 2 * (kSubElems > kATile ? kSubElems : kATile); }
constexpr int ring_b(int NTW) { return NTW * kSubElems; }

template <int MT, int NTW, bool GATHER, bool SCATTER>
__global__ __launch_bounds__(512) void dgrad_kmajor_kernel(const bf16_t* __restrict__ A, const int32_t* __restrict__ a_index,
                                                           const bf16_t* __restrict__ W, const int32_t* __restrict__ offsets,
                                                           const int32_t* __restrict__ out_index, int K, int N, int E, int nblk_n,
                                                           bf16_t* __restrict__ out) {
  constexpr bool four = MT == 2;
  __shared__ __attribute__((aligned(kLowLds))) bf16_t a0[ring_a(MT)];
  __shared__ __attribute__((aligned(kLowLds))) bf16_t a1[ring_a(MT)];
  __shared__ __attribute__((aligned(kLowLds))) bf16_t a2[ring_a(MT)];
  __shared__ __attribute__((aligned(kLowLds))) bf16_t a3[four ? ring_a(MT) : 8];
  __shared__ __attribute__((aligned(16))) bf16_t b0[ring_b(NTW)];
  __shared__ __attribute__((aligned(16))) bf16_t b1[ring_b(NTW)];
  __shared__ __attribute__((aligned(16))) bf16_t b2[ring_b(NTW)];
  __shared__ __attribute__((aligned(16))) bf16_t b3[four ? ring_b(NTW) : 8];
  __shared__ int dst_s[64 * MT];
  dgrad_block<MT, NTW, GATHER, SCATTER>(Ring{a0, a1, a2, a3, b0, b1, b2, b3}, dst_s, blockIdx.x, A, a_index, W, offsets, out_index, K, N, E,
                                        nblk_n, out);
}

// ---- weight gradients: dW[e][n][m] = sum over the rows r of expert e of P[srcP(r)][n] Q[srcQ(r)][m] ------------
// Both operands row-major activations, contracted over their rows: K-major both.  srcP(r) = index[r] (GATHER_P) or r,
// likewise Q.  A K stage is 32 rows; rows past the expert's end read `zrow` (zeros, at least 128 elements) on the P
// side and the expert's last row on the Q side (memory that is certainly finite, whatever the rows behind the
// expert's hold).  One workgroup per (expert, 64 MT rows of dW, 128 NTW columns of dW); MT = 4 (256 rows) halves what
// a workgroup streams of Q per row of dW, at 192 accumulator registers and a ring of three 40 KB stages.
// An expert with more than `chunk` rows is cut into chunks of that many rows, each a workgroup of its own per tile of
// dW, so that a few experts holding most of the rows do not leave a few workgroups with most of the work; such an
// expert's chunks write fp32 partial tiles to `part` (one [N, M] slot per chunk, slots numbered over all experts'
// chunks) and wgrad_reduce_block adds them in chunk order.  Experts of one chunk write dW directly, in bf16 or, with `f32`
// (gradients of fp32 master weights), as they are: a conversion pass afterwards cost 61 us at T = 8192.  The chunks are
// listed once per backward pass by wgrad_plan (below), so that a workgroup finds its chunk with one load.
struct WgradPlan {
  int total;         // chunks over all experts
  int n_cut;         // experts cut into more than one chunk
  int pad[2];
  // followed by int4 chunk[total] = {expert, first row, end row, chunks of that expert},
  // from entry `slots` on int4 cut[n_cut] = {expert, its first chunk, its chunks, 0},
  // and from entry `slots + E` on int4 expert[E] = {first chunk, chunks, 0, 0}
};

// One wave: lane = expert, over ALL routed experts (the +/-Identity ones have rows for the router's weight gradient).
// `slots` = the capacity of the chunk list (backward_chunk_slots).
__device__ __forceinline__ void wgrad_plan(const int32_t* __restrict__ offsets, int E, int chunk, int slots, int* __restrict__ plan) {
  const int lane = lane_id();
  int lo = 0, hi = 0;
  if (lane < E) { lo = offsets[lane]; hi = offsets[lane + 1]; }
  const int mine = lane < E ? max(1, (hi - lo + chunk - 1) / chunk) : 0;   // an idle expert keeps one (empty) chunk: its zero gradient
  const int incl = wave_inclusive_scan(mine);
  const int first = incl - mine;
  const unsigned long long cut = __ballot(mine > 1);
  if (lane == kWave - 1) { plan[0] = incl; plan[1] = __popcll(cut); }
  typedef int int4v __attribute__((ext_vector_type(4)));
  int4v* list = reinterpret_cast<int4v*>(plan + 4);
  for (int c = 0; c < mine; ++c) list[first + c] = int4v{lane, lo + c * chunk, min(lo + (c + 1) * chunk, hi), mine};
  if (mine > 1) list[slots + __popcll(cut & ((1ull << lane) - 1))] = int4v{lane, first, mine, 0};
  if (lane < E) list[slots + E + lane] = int4v{first, mine, 0, 0};
}

// the neighbour's value: lanes 2 i and 2 i + 1 trade
__device__ __forceinline__ float quad_swap(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
}

// SMALL: an operand's rows lie within kNoRow bytes of its first one, so that a transfer's address is a descriptor and one 32-bit offset, and a row
// past the end is an offset past the descriptor's, which reads zeros.  (With 64-bit addresses the tall tiles spill, and a spilled
// register's reload waits for every transfer before it.)
constexpr unsigned kNoRow = 0xffffff00u;
template <int MT, int NTW, bool GATHER_P, bool GATHER_Q, bool SMALL>
__device__ __forceinline__ void wgrad_block(const Ring& ring, int block, const bf16_t* __restrict__ P, const bf16_t* __restrict__ Q,
                                            const int32_t* __restrict__ index, const bf16_t* __restrict__ zrow, int N, int M, int E,
                                            const int* __restrict__ plan, float* __restrict__ part, void* __restrict__ dW, int f32) {
  static_assert(MT == 2 || MT == 4, "128 or 256 rows of dW per workgroup");
  constexpr int BM = 64 * MT, BN = kSubW * NTW;
  constexpr int R = MT == 4 ? 3 : kRing;                 // stages that fit LDS (MT = 4: 40 KB each)
  constexpr int kPOps = MT / 2;                          // 128-column sub-tiles of P
  constexpr int kOps = kPOps + NTW;
  // Workgroup ids congruent mod 8 run on one XCD: they walk a contiguous range of (expert, m block, n block) triples,
  // so the workgroups that read the same rows of Q (and of P) share that XCD's L2.
  const int nblk_n = N / BM, nblk_m = M / BN;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int total_chunks = __builtin_amdgcn_readfirstlane(plan[0]);
  // With experts cut into chunks the work per chunk is uneven (a cut expert's chunks are several times a small
  // expert's rows) and contiguous ranges of chunks per XCD would leave some XCDs with most of it: round robin then.
  const bool uneven = __builtin_amdgcn_readfirstlane(plan[1]) > 0;
  const int item = uneven ? block : xcd_tile(block, total_chunks * nblk_n * nblk_m);
  if (item >= total_chunks * nblk_n * nblk_m) return;
  const int cg = item / (nblk_n * nblk_m), rest = item - cg * (nblk_n * nblk_m);      // chunk, numbered over all experts
  const int* entry = plan + 4 + 4 * cg;
  const int e = __builtin_amdgcn_readfirstlane(entry[0]);
  if (e >= E) return;                    // E = experts with weights; the chunks behind them belong to +/-Identity experts
  const int lo = __builtin_amdgcn_readfirstlane(entry[1]), hi = __builtin_amdgcn_readfirstlane(entry[2]);
  const int e_chunks = __builtin_amdgcn_readfirstlane(entry[3]);
  const int n0 = (rest % nblk_n) * BM, m0 = (rest / nblk_n) * BN;
  const int wn = wave & 3, wm = wave >> 2;
  constexpr int RT = 2 * MT, CT = 2 * NTW;                // a wave's tiles of 16 x 16
  floatx4 acc[RT][CT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[rt][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  auto pbuf = [&](auto bc) -> bf16_t* { return ring.template a<decltype(bc)::value>(); };
  auto qbuf = [&](auto bc) -> bf16_t* { return ring.template b<decltype(bc)::value>(); };
  const int nstages = (hi - lo + kKS - 1) / kKS;
  const int gofs = kfill_granule(tid) * 8;
  // This thread's row of stage `stage` (row tid / 16 of the stage's 32), counted from lo
  const int count = hi - lo;
  auto stage_row = [&](int stage) { return min(stage, nstages - 1) * kKS + (tid >> 4); };
  auto lookup = [&](int stage) { return (GATHER_P || GATHER_Q) ? index[lo + min(stage_row(stage), count - 1)] : 0; };
  // transfer q of a stage into buffer bc, the row index ix looked up before
  const int wave_elems = __builtin_amdgcn_readfirstlane(tid >> 6) * kWaveElems;
  const unsigned gbytes = gofs * sizeof(bf16_t);
  const __amdgpu_buffer_rsrc_t p_rsrc = make_rsrc(uniform(P + (GATHER_P ? 0 : (size_t)lo * N) + n0), SMALL ? kNoRow : 0);
  const __amdgpu_buffer_rsrc_t q_rsrc = make_rsrc(uniform(Q + (GATHER_Q ? 0 : (size_t)lo * M) + m0), SMALL ? kNoRow : 0);
  unsigned pv = 0, qv = 0;
  auto fill = [&](auto bc, int stage, int ix, int q) {
    if constexpr (SMALL) {
      if (q == 0) {
        const int r = stage_row(stage);
        pv = r < count ? (unsigned)(GATHER_P ? ix : r) * (unsigned)(N * (int)sizeof(bf16_t)) + gbytes : kNoRow;
        qv = r < count ? (unsigned)(GATHER_Q ? ix : r) * (unsigned)(M * (int)sizeof(bf16_t)) + gbytes : kNoRow;
      }
      const int sub = q < kPOps ? q : q - kPOps;
      bf16_t* const dst = (q < kPOps ? pbuf(bc) : qbuf(bc)) + sub * kSubElems + wave_elems;
      dma16_buf(q < kPOps ? p_rsrc : q_rsrc, q < kPOps ? pv : qv, sub * kSubW * (unsigned)sizeof(bf16_t), dst);
    } else {
      const int r = lo + stage_row(stage);
      const bool live = r < hi;
      const int rc = live ? r : hi - 1;
      if (q < kPOps) {
        const bf16_t* prow = live ? P + (size_t)(GATHER_P ? ix : rc) * N + n0 : zrow;
        kfill_subtile(prow + q * kSubW + gofs, pbuf(bc) + q * kSubElems);
      } else {
        const bf16_t* qrow = Q + (size_t)(GATHER_Q ? ix : rc) * M + m0;
        kfill_subtile(qrow + (q - kPOps) * kSubW + gofs, qbuf(bc) + (q - kPOps) * kSubElems);
      }
    }
  };
  int poff[RT / 2], qoff[CT / 2];                          // of the even tiles: an odd one is 16 elements on
#pragma unroll
  for (int t = 0; t < RT / 2; ++t) {
    const int t16 = wm * RT + 2 * t;
    poff[t] = (t16 >> 3) * kSubElems + kfrag_offset(lane, (t16 & 7) * 16);
  }
#pragma unroll
  for (int t = 0; t < CT / 2; ++t) {
    const int t16 = wn * CT + 2 * t;
    qoff[t] = (t16 >> 3) * kSubElems + kfrag_offset(lane, (t16 & 7) * 16);
  }
  using std::integral_constant;
  if (nstages > 0) {                                               // an idle expert's gradient is zero
    // The row index of a gathered operand is loaded R stages before the transfers that use it: the index of stage s sits in ix[s % R], and
    // where stage s + R is requested with it the one of stage s + 2 R is loaded.  No wait counts these loads: the compiler drops the ones
    // that nothing behind them uses, as in the last stages, and moves others, and a wait that counts a load it has dropped lets the last
    // transfer of the stage that is read next stay in flight.  Counted by transfers alone, which are all issued at their places, a wait
    // is for R - 2 operations more than it need be where the loads are there: no difference in time (T = 8192, H = 768, I = 384, E = 64, k = 6:
    // 154 to 170 us either way).
    constexpr int kVm = kOps + ((GATHER_P || GATHER_Q) ? 1 : 0);           // operations of a stage
    int ix[R];
    using Pipe = StagePipe<RT, CT, false>;
#pragma unroll
    for (int i = 0; i < R; ++i) ix[i] = lookup(i);
    auto request = [&](auto bc, int stage, int q) {       // operation q of a stage: its transfers, then the lookup
      constexpr int b = decltype(bc)::value;
      if (q < kOps) fill(bc, stage, ix[b], q);
      else ix[b] = lookup(stage + R);
      __builtin_amdgcn_sched_barrier(0);                   // (stage by stage, as the waits assume)
    };
    auto request_all = [&](auto bc, int stage) {
#pragma unroll
      for (int q = 0; q < kVm; ++q) request(bc, stage, q);
    };
    request_all(integral_constant<int, 0>{}, 0);
    request_all(integral_constant<int, 1>{}, 1);
    if constexpr (R == 4) request_all(integral_constant<int, 2>{}, 2);
#pragma unroll
    for (int q = 0; q < 2; ++q) request(integral_constant<int, R - 1>{}, R - 1, q);
    auto read_p = [&](auto bc, int rt) { return kfrag_read(pbuf(bc) + (rt & 1) * 16, poff[rt >> 1]); };
    auto read_q = [&](auto bc, int j) { return kfrag_read(qbuf(bc) + (j & 1) * 16, qoff[j >> 1]); };
    Pipe pipe;
    sync_keep_loads<(R - 2) * kOps + 2>();
    {
      const integral_constant<int, 0> b0;
      pipe.begin([&](int rt) { return read_p(b0, rt); }, [&](int j) { return read_q(b0, j); });
    }
    auto step = [&](auto bc, int stage) {
      constexpr int b = decltype(bc)::value;
      const integral_constant<int, (b + 1) % R> nc;
      const integral_constant<int, (b + R - 1) % R> pc;
      pipe.template stage<b * RT % Pipe::NA, kVm>(
          acc, [&]() { sync_keep_loads<(R - 2) * kOps>(); }, [&](int rt) { return read_p(bc, rt); }, [&](int rt) { return read_p(nc, rt); },
          [&](int j) { return read_q(nc, j); }, [&](int q) { request(bc, stage + R, q); }, [&](int q) { request(pc, stage + R - 1, q); });
    };
    int i = 0;
    for (; i + R <= nstages; i += R) {
      step(integral_constant<int, 0>{}, i);
      step(integral_constant<int, 1>{}, i + 1);
      step(integral_constant<int, 2>{}, i + 2);
      if constexpr (R == 4) step(integral_constant<int, 3>{}, i + 3);
    }
    if (i < nstages) step(integral_constant<int, 0>{}, i);
    if (i + 1 < nstages) step(integral_constant<int, 1>{}, i + 1);
    if constexpr (R == 4) if (i + 2 < nstages) step(integral_constant<int, 2>{}, i + 2);
    __builtin_amdgcn_s_waitcnt(0);       // the repeated requests of the last steps land before the workgroup ends
  }
  // lane = column m0 + (wn CT + j) 16 + lane % 16, register r = row n0 + (wm RT + rt) 16 + 4 (lane / 16) + r: 16 lanes of a store leave 64
  // contiguous bytes of a row in fp32, and in bf16 (lane pairs trade the odd row of one for the even row of the other, two columns a lane)
  // 32.  With a lane per row, 16 bytes of each in a store, the launch took 207 us instead of 195 at T = 8192, H = 768, I = 384, E = 64, k = 6.
  const int n = lane & 15, g4 = lane >> 4;
  // Offsets count from the tile's first element: an expert's matrix may hold 2^32 bytes and more.
  const unsigned row = wm * MT * 32 + 4 * g4, col = wn * NTW * 32 + n;
  const size_t tile = (size_t)n0 * M + m0;
  if (e_chunks == 1 && !f32) {
    const __amdgpu_buffer_rsrc_t dst = make_rsrc(uniform(static_cast<bf16_t*>(dW) + (size_t)e * N * M + tile), kNoRow);
    const bool odd = n & 1;
    const unsigned voff = ((row + odd) * M + (col & ~1u)) * sizeof(bf16_t);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int i = 0; i < 4; i += 2)
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          const float lo = acc[rt][j][i], hi2 = acc[rt][j][i + 1];
          const float got = quad_swap(odd ? lo : hi2);
          typedef bf16_t bf16x2 __attribute__((ext_vector_type(2)));
          const bf16x2 v = {(bf16_t)(odd ? got : lo), (bf16_t)(odd ? hi2 : got)};
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), dst, voff,
                                                ((rt * 16 + i) * M + j * 16) * (unsigned)sizeof(bf16_t), 0);
        }
  } else {
    float* const base = e_chunks == 1 ? static_cast<float*>(dW) + (size_t)e * N * M : part + (size_t)cg * N * M;
    const __amdgpu_buffer_rsrc_t dst = make_rsrc(uniform(base + tile), kNoRow);
    const unsigned voff = (row * M + col) * sizeof(float);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          const float v = acc[rt][j][i];         // (a bit_cast of the element itself reads element 0)
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), dst, voff, ((rt * 16 + i) * M + j * 16) * (unsigned)sizeof(float),
                                                0);
        }
  }
}

// ---- the three products behind act_bwd_kernel in one launch --------------------------------------------------------
// dx of every slot = [dg, du] W_gate_up (blocks [0, n_dx)), dW_gate_up = [dg, du]^T x (the next n_gu), dW_down = d^T (w h) (the rest).
// They need nothing from one another, and a workgroup fills a CU in each: as launches of their own each ended with a round in which most
// CUs had none, and a small call spent three launches on three handfuls of workgroups.  Longest workgroups first.  NH, NI: what 128-column
// sub-tiles H and I divide into.  TALL: 256-row tiles in all three, dW_down's only where they divide H (tall_d); else in none.  The three
// launches -> this one: T = 8192, H = 768, I = 384, E = 64, k = 6: 259 -> 233 us; T = 2500: 118 -> 90; T = 1111, H = 512, I = 256, E = 9,
// k = 2: 36 -> 14; T = 16000, H = 1024, I = 512, E = 64, k = 8: 750 -> 731.
struct BackwardGemms {
  const bf16_t *x, *d_out, *dgu, *hidden, *wgu, *zrow;
  const int32_t *offsets, *perm_slot, *perm_token;
  const int* plan;
  bf16_t* dxs;
  void *dwgu, *dwd;
  float *part_gu, *part_d;
  int H, I, E, f32, n_dx, n_gu;
  bool tall_d;
};

template <int NH, int NI, bool TALL>
__global__ __launch_bounds__(512) void backward_gemms_kernel(BackwardGemms g) {
  constexpr int MT = TALL ? 4 : 2, NB = NH > NI ? NH : NI;
  __shared__ __attribute__((aligned(kLowLds))) bf16_t a0[ring_a(MT)];
  __shared__ __attribute__((aligned(kLowLds))) bf16_t a1[ring_a(MT)];
  __shared__ __attribute__((aligned(kLowLds))) bf16_t a2[ring_a(MT)];
  __shared__ __attribute__((aligned(kLowLds))) bf16_t a3[ring_a(2)];
  __shared__ __attribute__((aligned(16))) bf16_t b0[ring_b(NB)];
  __shared__ __attribute__((aligned(16))) bf16_t b1[ring_b(NB)];
  __shared__ __attribute__((aligned(16))) bf16_t b2[ring_b(NB)];
  __shared__ __attribute__((aligned(16))) bf16_t b3[ring_b(NB)];
  __shared__ int dst_s[64 * MT];
  const Ring ring{a0, a1, a2, a3, b0, b1, b2, b3};
  const int block = blockIdx.x;
  auto down = [&](auto mt) {
    wgrad_block<decltype(mt)::value, NI, true, false, TALL>(ring, block - g.n_dx - g.n_gu, g.d_out, g.hidden, g.perm_token, g.zrow, g.H, g.I, g.E,
                                                            g.plan, g.part_d, g.dwd, g.f32);
  };
  if (block < g.n_dx)
    dgrad_block<MT, NH, false, true>(ring, dst_s, block, g.dgu, nullptr, g.wgu, g.offsets, g.perm_slot, 2 * g.I, g.H, g.E, g.H / (kSubW * NH),
                                     g.dxs);
  else if (block < g.n_dx + g.n_gu)
    wgrad_block<MT, NH, false, true, TALL>(ring, block - g.n_dx, g.dgu, g.x, g.perm_token, g.zrow, 2 * g.I, g.H, g.E, g.plan, g.part_gu, g.dwgu,
                                           g.f32);
  else if (!TALL || g.tall_d)
    down(std::integral_constant<int, MT>{});
  else
    down(std::integral_constant<int, 2>{});
}

// For the experts that were cut into chunks (none, when the tokens are spread evenly): dW[e] = the sum of expert e's
// partial tiles, in chunk order, for both weight tensors (partials of the first in `part_a`, [.., NMa] each, of the
// second in `part_b`).  Workgroup `block` of 256 threads, a thread per four elements.  E = experts with weights.
__device__ __forceinline__ void wgrad_reduce_block(int block, const float* __restrict__ part_a, const float* __restrict__ part_b,
                                                   const int* __restrict__ plan, int slots, int NMa, int NMb, int E,
                                                   void* __restrict__ dWa, void* __restrict__ dWb, int f32) {
  const int n_cut = plan[1];
  if (n_cut == 0) return;
  const size_t i = ((size_t)block * 256 + threadIdx.x) * 4;
  const int* cut = plan + 4 + 4 * slots;
  auto reduce = [&](const float* part, int NM, void* dW, int e, int first, int n) {
    if (i >= (size_t)NM) return;
    floatx4 acc = *reinterpret_cast<const floatx4*>(part + (size_t)first * NM + i);
    for (int c = 1; c < n; ++c) {
      const floatx4 v = *reinterpret_cast<const floatx4*>(part + (size_t)(first + c) * NM + i);
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] += v[r];
    }
    if (f32) {
      *reinterpret_cast<floatx4*>(static_cast<float*>(dW) + (size_t)e * NM + i) = acc;
      return;
    }
    bf16x4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = (bf16_t)acc[r];
    *reinterpret_cast<bf16x4*>(static_cast<bf16_t*>(dW) + (size_t)e * NM + i) = o;
  };
  for (int q = 0; q < n_cut; ++q) {
    const int e = cut[4 * q], first = cut[4 * q + 1], n = cut[4 * q + 2];
    if (e >= E) continue;
    reduce(part_a, NMa, dWa, e, first, n);
    reduce(part_b, NMb, dWb, e, first, n);
  }
}

}  // namespace
}  // namespace bibo
