// Staged K-split fused GEMM kernels of one bit-width (compile with -DAP_BITS=3..8) and their launch dispatch.
#include "ap_gemms.hpp"
#include "ap_gemms_launch.hpp"

#ifndef AP_BITS
#error "compile with -DAP_BITS=<3..8>"
#endif

namespace ap {

template <int BITS>
void launch_gemms(const uint16_t *x, const GemmsMembers &members, int M, int K, hipStream_t stream) {
    const half_t *xh = reinterpret_cast<const half_t *>(x);
    const dim3 block(kWave, kGemmsWaves), grid((unsigned)members.block0[members.count]);
    if (M <= 4) gemms_kbit_kernel<BITS, 4><<<grid, block, 0, stream>>>(xh, members, M, K);
    else if (M <= 8) gemms_kbit_kernel<BITS, 8><<<grid, block, 0, stream>>>(xh, members, M, K);
    else if (M <= 16) gemms_kbit_kernel<BITS, 16><<<grid, block, 0, stream>>>(xh, members, M, K);
    else gemms_kbit_kernel<BITS, 32><<<grid, block, 0, stream>>>(xh, members, M, K);
}

template void launch_gemms<AP_BITS>(const uint16_t *, const GemmsMembers &, int, int, hipStream_t);

}  // namespace ap
