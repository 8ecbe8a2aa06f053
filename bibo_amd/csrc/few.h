// Device code of the few-token kernels (experts_few.hip) that the router kernel with a gate/up pass behind it (router.hip) shares.
#pragma once
#include "tile_f32.h"

namespace bibo {
namespace {

__device__ __forceinline__ void load8(float (&v)[8], const float* p) {
  const floatx4 a = *reinterpret_cast<const floatx4*>(p), b = *reinterpret_cast<const floatx4*>(p + 4);
#pragma unroll
  for (int q = 0; q < 4; ++q) { v[q] = a[q]; v[4 + q] = b[q]; }
}

// eight weights as they come from memory
template <typename T> struct Raw8;
template <> struct Raw8<bf16_t> {
  bf16x8 v;
  __device__ __forceinline__ void load(const bf16_t* p) { v = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(p)); }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = (bf16_t)0.f;
  }
  __device__ __forceinline__ float get(int q) const { return (float)v[q]; }
};
template <> struct Raw8<float> {
  floatx4 a, b;
  __device__ __forceinline__ void load(const float* p) {
    a = __builtin_nontemporal_load(reinterpret_cast<const floatx4*>(p));
    b = __builtin_nontemporal_load(reinterpret_cast<const floatx4*>(p + 4));
  }
  __device__ __forceinline__ void zero() { a = b = floatx4{0.f, 0.f, 0.f, 0.f}; }
  __device__ __forceinline__ float get(int q) const { return q < 4 ? a[q] : b[q - 4]; }
};

__device__ __forceinline__ float sum16(float v) {          // over the 16 lanes of a DPP row, the same in every lane
  auto dpp = [](float x, auto ctrl) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, false));
  };
  v += dpp(v, std::integral_constant<int, 0xB1>{});
  v += dpp(v, std::integral_constant<int, 0x4E>{});
  v += dpp(v, std::integral_constant<int, 0x141>{});
  return v + dpp(v, std::integral_constant<int, 0x140>{});
}

// the end of a dot product: the lanes' four partial sums each.  Sixty-four chains and a tree, as where a wave's lanes share a row
// (experts_generic.hip): one chain per lane was 1.3 times as far from exact in fp32 at H = 768
__device__ __forceinline__ float sum64(const float (&part)[4]) { return sum16((part[0] + part[1]) + (part[2] + part[3])); }

constexpr int kGateRows = 32;           // weight rows per workgroup of the gate/up kernel: two per 16 lanes

// rows row0 and row0 + 16 of an expert's gate/up weights [I2, H] times a token's row; 16 lanes a weight row, lane c of them.  NG =
// ceil(H / 128): 8-element granules of a row per lane.
template <typename T, int NG>
__device__ __forceinline__ void gateup_rows(const Raw8<T> (&xv)[NG], const T* __restrict__ we, int row0, int c, int H, int I2,
                                            float* __restrict__ gu) {
  Raw8<T> wv[2][NG];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const T* wr = we + (size_t)min(row0 + 16 * r, I2 - 1) * H;
#pragma unroll
    for (int u = 0; u < NG; ++u) {
      const int g = (u * 16 + c) * 8;
      if (g < H) wv[r][u].load(wr + g); else wv[r][u].zero();
    }
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NG; ++u)
#pragma unroll
      for (int q = 0; q < 8; ++q) part[q & 3] = fmaf(wv[r][u].get(q), xv[u].get(q), part[q & 3]);
    const float acc = sum64(part);
    if (c == 0 && row0 + 16 * r < I2) gu[row0 + 16 * r] = acc;
  }
}

}  // namespace
}  // namespace bibo
