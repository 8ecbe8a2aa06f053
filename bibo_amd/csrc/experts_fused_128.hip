// The launches of experts_fused_launch.h at I = 128.
#include "experts_fused.h"

namespace bibo {

template void launch_fused_nt<1>(const bf16_t*, const bf16_t*, const bf16_t*, const float*, const float*, const int32_t*, const int32_t*,
                                 const int32_t*, int, int, int, int, unsigned, void*, bool, bf16_t*, const ScanArgs&, hipStream_t);
template void launch_raw_nt<1, 1>(const bf16_t*, const bf16_t*, const int32_t*, const int32_t*, int, int, int, unsigned, bf16_t*, int,
                                  hipStream_t, const ScanArgs&);
template void launch_raw_nt<1, 3>(const bf16_t*, const bf16_t*, const int32_t*, const int32_t*, int, int, int, unsigned, bf16_t*, int,
                                  hipStream_t, const ScanArgs&);

}  // namespace bibo
