// Host side of the fused kernel (experts_fused.h): which width, and whether a tile's columns are cut over several workgroups.
#include "experts_fused_launch.h"

namespace bibo {

// Phase 1 of the fused kernel alone: gu[row] = [x W_gate^T, x W_up^T] in bf16 for every permuted row (what the backward
// pass recomputes, moe.py:84).  Same shapes as launch_experts_fused.
// `split`: one workgroup per 128 gate (and up) columns of a tile, for calls with fewer tiles than CUs.
hipError_t launch_gateup_raw(const void* x, const void* wgu, const int32_t* offsets, const int32_t* perm_token, int T, int H,
                             int E, int k, int I, void* gu, bool split, bool f32, hipStream_t s, const ScanArgs& scan) {
  const int S = T * k;
  if (S == 0) return hipSuccess;
  if ((unsigned long long)T * H * sizeof(bf16_t) >= (1ull << 32)) return hipErrorInvalidValue;
  const unsigned xb = (unsigned)((size_t)T * H * sizeof(bf16_t));
  const bf16_t* xp = static_cast<const bf16_t*>(x);
  const bf16_t* gp = static_cast<const bf16_t*>(wgu);
  bf16_t* out = static_cast<bf16_t*>(gu);
  if ((f32 && !split) || (scan.idx != nullptr && (!f32 || S > kSplitSlots))) return hipErrorInvalidValue;
  if (f32) {
    launch_raw_nt<1, 3>(xp, gp, offsets, perm_token, S, H, E, xb, out, I / 128, s, scan);
    return hipGetLastError();
  }
  if (split) {
    launch_raw_nt<1, 1>(xp, gp, offsets, perm_token, S, H, E, xb, out, I / 128, s, scan);
    return hipGetLastError();
  }
  switch (I) {
    case 128: launch_raw_nt<1, 1>(xp, gp, offsets, perm_token, S, H, E, xb, out, 1, s, scan); break;
    case 256: launch_raw_nt<2, 1>(xp, gp, offsets, perm_token, S, H, E, xb, out, 1, s, scan); break;
    case 384: launch_raw_nt<3, 1>(xp, gp, offsets, perm_token, S, H, E, xb, out, 1, s, scan); break;
    case 512: launch_raw_nt<4, 1>(xp, gp, offsets, perm_token, S, H, E, xb, out, 1, s, scan); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// Whether a tile's columns are cut over several workgroups.  The fused kernel keeps a row's tile on one CU, which pulls all of the expert's
// weights then, at HBM's latency where no other tile of the expert runs beside it.  Cut (launch_gateup_raw, launch_down_act), each CU pulls a
// part of them, the pre-activations make a round trip and every column block computes the activations again.  So the limit, in routed slots,
// goes with the weights of an expert, H x I; with the experts, because many of them share what the chip's L2s deliver; and with few experts
// as the square of H x I, because their tiles are short streams then that the second launch outweighs (the divisors: where the two meet
// up to 1.5 MB of weights an expert, and above them a line below which it pays off at every size measured).  At I = 512 the second half's tiles
// of 64 rows come to two rounds from about 3600 slots on.  A layer replayed from a graph, cold weights, bf16, uncut -> cut, us:
//   E = 64, k = 6: H = 768, I = 384: 58 -> 49 at 1800 slots, 58 -> 53 at 3120; H = 1024, I = 256: 53 -> 48 at 1800, 53 -> 50 at 2640;
//     H = 768, I = 256: 45 -> 42 at 1440, 45 -> 44 at 2100; H = 512, I = 384: 43 -> 39 at 1200, 43 -> 43 at 1920; H = 512, I = 256: 34 -> 32 at
//     780, 35 -> 35 at 1350
//   E = 64, k = 8, H = 1024, I = 512, sum of the kernels: 90 -> 68 at 2048, 89 -> 72 at 2800, 84 -> 86 at 3600
//   E = 32, k = 4: H = 768, I = 384: 54 -> 40 at 800, 50 -> 46 at 2000; H = 1024, I = 256: 48 -> 42 at 1200, 48 -> 46 at 1960; H = 768, I = 256:
//     32 -> 29 at 600, 32 -> 34 at 1200; H = 512, I = 384: 31 -> 31 at 800, 31 -> 32 at 1120
//   E = 16, k = 3: H = 768, I = 384: 38 -> 33 at 600, 38 -> 38 at 1350, 38 -> 39 at 1710; H = 1024, I = 256: 36 -> 34 at 600, 37 -> 38 at 1200; H = 768, I = 256:
//     31 -> 29 at 384, 31 -> 31 at 576, 32 -> 33 at 750; H = 512, I = 384: 30 -> 29 at 390, 30 -> 31 at 570
//   E = 48, k = 4, H = 512, I = 256: 26 -> 27 at 712
//   E = 9, k = 2: H = 768, I = 384: 37 -> 33 at 400, 38 -> 36 at 600, 38 -> 38 at 880; H = 512, I = 512: 34 -> 35 at 600
// and with larger weights, which it pays off for longer: E = 9, k = 2: H = 640, I = 512: 42 -> 37 at 1180; H = 768, I = 512: 47 -> 41 at 1700;
//   H = 896, I = 512: 51 -> 46 at 2100, 51 -> 50 at 2300; H = 1024, I = 384: 45 -> 43 at 1700; H = 1024, I = 512: 54 -> 46 at 2300;
//   E = 16, k = 3: H = 640, I = 512: 43 -> 38 at 1950; H = 1024, I = 384: 46 -> 48 at 2160, 48 -> 47 at 2370; H = 1024, I = 512: 62 -> 53 at 3120
// Pre-activations in bf16 were 1 to 5 us faster and half again as far from the exact result (3.5e-3 against 2.3e-3).
bool split_columns(int S, int E, int H, int I) {
  const long long hi = (long long)H * I / 1024;
  return I >= 256 && S <= kSplitSlots && S <= hi * (46 + E) / 10 && S <= hi * hi * E / (hi <= 256 ? 1100 : 763);
}

// gu [S, 2I] fp32 -> routing-weighted rows in slot order (bf16 or, with f32_rows, fp32), and with `preact` their bf16 copy (down_act_kernel; I <= 384); shapes as
// launch_gateup_raw takes them, I = 256 to 512
hipError_t launch_down_act(const void* gu, const void* wd, const float* theta, const float* w, const int32_t* offsets,
                           const int32_t* perm_slot, int S, int H, int E, int I, int act, void* yw, bool f32_rows, void* preact,
                           hipStream_t s) {
  if (S == 0) return hipSuccess;
  if (I == 512 && preact != nullptr) return hipErrorInvalidValue;
  const float* gp = static_cast<const float*>(gu);
  bf16_t* pp = static_cast<bf16_t*>(preact);
  const bf16_t* dp = static_cast<const bf16_t*>(wd);
  switch (I) {
    case 256: launch_down_act_nt<2>(gp, dp, theta, w, offsets, perm_slot, S, H, E, act, yw, f32_rows, pp, s); break;
    case 384: launch_down_act_nt<3>(gp, dp, theta, w, offsets, perm_slot, S, H, E, act, yw, f32_rows, pp, s); break;
    case 512: launch_down_act_nt<4>(gp, dp, theta, w, offsets, perm_slot, S, H, E, act, yw, f32_rows, pp, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

bool fused_supported(int H, int I, int dtype) {
  // the activation tile plus two weight stages have to fit 160 KB of LDS: I <= 384
  return dtype == BIBO_DTYPE_BF16 && H >= 128 && (H % 128) == 0 && (I == 128 || I == 256 || I == 384);
}

// I = 512 on 64-row tiles: what `auto` runs for the shape, under the name of the two-kernel family the stage calls run
bool fused_wide_supported(int H, int I, int dtype) { return dtype == BIBO_DTYPE_BF16 && H >= 128 && H % 128 == 0 && I == 512; }

hipError_t launch_experts_fused(const void* x, const void* wgu, const void* wd, const float* theta, const float* w,
                                const int32_t* offsets, const int32_t* perm_slot, const int32_t* perm_token, int T,
                                int H, int E, int k, int I, int act, void* yw, bool f32_rows, void* preact, hipStream_t s,
                                const ScanArgs& scan) {
  const int S = T * k;
  if (S == 0) return hipSuccess;
  if ((unsigned long long)T * H * sizeof(bf16_t) >= (1ull << 32)) return hipErrorInvalidValue;   // 32-bit byte offsets into x
  if (I == 512 && preact != nullptr) return hipErrorInvalidValue;
  if (f32_rows && (preact != nullptr || S > kStreamMaxSlots)) return hipErrorInvalidValue;   // compiled for calls that may stream
  const unsigned xb = (unsigned)((size_t)T * H * sizeof(bf16_t));
  const bf16_t* xp = static_cast<const bf16_t*>(x);
  const bf16_t* gp = static_cast<const bf16_t*>(wgu);
  const bf16_t* dp = static_cast<const bf16_t*>(wd);
  bf16_t* pp = static_cast<bf16_t*>(preact);
  switch (I) {
    case 128: launch_fused_nt<1>(xp, gp, dp, theta, w, offsets, perm_slot, perm_token, S, H, E, act, xb, yw, f32_rows, pp, scan, s); break;
    case 256: launch_fused_nt<2>(xp, gp, dp, theta, w, offsets, perm_slot, perm_token, S, H, E, act, xb, yw, f32_rows, pp, scan, s); break;
    case 384: launch_fused_nt<3>(xp, gp, dp, theta, w, offsets, perm_slot, perm_token, S, H, E, act, xb, yw, f32_rows, pp, scan, s); break;
    case 512: launch_fused_nt<4>(xp, gp, dp, theta, w, offsets, perm_slot, perm_token, S, H, E, act, xb, yw, f32_rows, pp, scan, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace bibo
