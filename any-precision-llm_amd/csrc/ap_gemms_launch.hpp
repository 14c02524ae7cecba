// Host-side launch interface of the staged K-split fused GEMM kernels (one translation unit per bit-width:
// ap_gemms_inst.hip with -DAP_BITS=b).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ap {

constexpr int kGemmsRows = 16;     // weight rows of a workgroup
constexpr int kGemmsWaves = 4;     // waves of a workgroup, each on every fourth step of 512 elements
constexpr int kGemmsMaxM = 32;
constexpr int kGemmsMaxGroup = 4;  // linears one launch can serve (they share x, K, M and w_bits)

// The linears of a launch.  Blocks of 16 weight rows are numbered through the members: member g owns blocks
// block0[g] .. block0[g + 1).  Output rows of member g are ldo[g] elements apart.
struct GemmsMembers {
    const uint32_t *qweight[kGemmsMaxGroup];
    const uint16_t *lut[kGemmsMaxGroup];
    uint16_t *out[kGemmsMaxGroup];
    int N[kGemmsMaxGroup];
    int block0[kGemmsMaxGroup + 1];
    int count;
    long long ldo[kGemmsMaxGroup];
    const uint16_t *bias;  // of member 0, the only one then; null: none
};

// Launches gemms_kbit_kernel<BITS, .> for 1 <= M <= 32 activation rows on `stream`.
template <int BITS>
void launch_gemms(const uint16_t *x, const GemmsMembers &members, int M, int K, hipStream_t stream);

extern template void launch_gemms<3>(const uint16_t *, const GemmsMembers &, int, int, hipStream_t);
extern template void launch_gemms<4>(const uint16_t *, const GemmsMembers &, int, int, hipStream_t);
extern template void launch_gemms<5>(const uint16_t *, const GemmsMembers &, int, int, hipStream_t);
extern template void launch_gemms<6>(const uint16_t *, const GemmsMembers &, int, int, hipStream_t);
extern template void launch_gemms<7>(const uint16_t *, const GemmsMembers &, int, int, hipStream_t);
extern template void launch_gemms<8>(const uint16_t *, const GemmsMembers &, int, int, hipStream_t);

}  // namespace ap
