// Launches of the fused kernel, of its first phase and of its second half by expert width I = 128 NT.  Each width is compiled in a file of
// its own (experts_fused_128.hip to experts_fused_512.hip): together they are a hundred variants of one large kernel.
#pragma once

#include "common.h"

namespace bibo {

constexpr int kSplitSlots = 3600;       // routed slots up to which a tile's columns may be cut (split_columns)

// MODE 1: pre-activations in bf16; MODE 3: in fp32 (experts_fused_kernel)
template <int NT>
void launch_fused_nt(const bf16_t* x, const bf16_t* wgu, const bf16_t* wd, const float* theta, const float* w,
                     const int32_t* offsets, const int32_t* perm_slot, const int32_t* perm_token, int S, int H, int E,
                     int act, unsigned x_bytes, void* yw, bool f32_rows, bf16_t* preact, const ScanArgs& scan, hipStream_t s);
template <int NT, int MODE>
void launch_raw_nt(const bf16_t* x, const bf16_t* wgu, const int32_t* offsets, const int32_t* perm_token, int S, int H, int E,
                   unsigned x_bytes, bf16_t* gu, int column_blocks, hipStream_t s, const ScanArgs& scan);
template <int NT>
void launch_down_act_nt(const float* gu, const bf16_t* wd, const float* theta, const float* w, const int32_t* offsets,
                        const int32_t* perm_slot, int S, int H, int E, int act, void* yw, bool f32_rows, bf16_t* preact,
                        hipStream_t s);

}  // namespace bibo
