// Host-side launch interface of the block-tile fused GEMM kernels (one translation unit per bit-width:
// ap_gemmb_inst.hip with -DAP_BITS=b).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ap {

constexpr int kGemmbRows = 32;  // weight rows of a wave

struct GemmbGeometry {
    int mb;      // blocks of 32 activation rows per workgroup tile
    int wn;      // waves side by side over the weight rows: a workgroup owns 32 wn of them
    int wk;      // groups of wn waves, each on its share of K
    int grid_n;  // tiles of 32 wn weight rows over all members
    int grid_m;  // ceil(M / (32 mb))
    double us;   // what the launch is estimated to take
};

constexpr int kGemmbMaxGroup = 4;  // linears one launch can serve (they share x, K, M and w_bits)

// The linears of a launch.  Tiles of 32 wn weight rows are numbered through the members: member g owns tiles
// tile0[g] .. tile0[g + 1) (grid_n = tile0[count]).  Output rows of member g are ldo[g] elements apart.
struct GemmbMembers {
    const uint32_t *qweight[kGemmbMaxGroup];
    const uint16_t *lut[kGemmbMaxGroup];
    uint16_t *out[kGemmbMaxGroup];
    int N[kGemmbMaxGroup];
    int tile0[kGemmbMaxGroup + 1];
    int count;
    long long ldo[kGemmbMaxGroup];
    const uint16_t *bias;  // of member 0, the only one then; null: none
};

// Launches gemmb_kbit_kernel<BITS, geo.mb, geo.wn, geo.wk> on `stream`; false if there is no such kernel.
template <int BITS>
bool launch_gemmb(const GemmbGeometry &geo, const uint16_t *x, const GemmbMembers &members, int M, int K, hipStream_t stream);

extern template bool launch_gemmb<3>(const GemmbGeometry &, const uint16_t *, const GemmbMembers &, int, int, hipStream_t);
extern template bool launch_gemmb<4>(const GemmbGeometry &, const uint16_t *, const GemmbMembers &, int, int, hipStream_t);
extern template bool launch_gemmb<5>(const GemmbGeometry &, const uint16_t *, const GemmbMembers &, int, int, hipStream_t);
extern template bool launch_gemmb<6>(const GemmbGeometry &, const uint16_t *, const GemmbMembers &, int, int, hipStream_t);
extern template bool launch_gemmb<7>(const GemmbGeometry &, const uint16_t *, const GemmbMembers &, int, int, hipStream_t);
extern template bool launch_gemmb<8>(const GemmbGeometry &, const uint16_t *, const GemmbMembers &, int, int, hipStream_t);

}  // namespace ap
