// Block-tile fused GEMM kernels of one bit-width (compile with -DAP_BITS=3..8) and their launch dispatch.
#include "ap_gemmb.hpp"
#include "ap_gemmb_launch.hpp"

#ifndef AP_BITS
#error "compile with -DAP_BITS=<3..8>"
#endif

namespace ap {

template <int BITS>
bool launch_gemmb(const GemmbGeometry &geo, const uint16_t *x, const GemmbMembers &members, int M, int K, hipStream_t stream) {
    const half_t *xh = reinterpret_cast<const half_t *>(x);
    const uint32_t tiles_pad = (uint32_t)((geo.grid_n + 7) / 8 * 8);
    const dim3 block(kWave, geo.wn * geo.wk), grid(tiles_pad * (unsigned)geo.grid_m);
    const uint32_t tile_div = geo.grid_m <= 8 ? 8u * (uint32_t)geo.grid_m : tiles_pad, tile_magic = reciprocal_floor(tile_div);
#define AP_GO(MB_, WN_, WK_)                                                                                                     \
    if (geo.mb == MB_ && geo.wn == WN_ && geo.wk == WK_) {                                                                       \
        if constexpr (GemmbLds<BITS, MB_, WN_, WK_>::kFits) {                                                                     \
            gemmb_kbit_kernel<BITS, MB_, WN_, WK_><<<grid, block, 0, stream>>>(xh, members, M, K, geo.grid_m, tile_div, tile_magic); \
            return true;                                                                                                         \
        }                                                                                                                        \
    }
    AP_GO(8, 4, 1)
    AP_GO(3, 4, 2)
    AP_GO(3, 2, 4)
    AP_GO(4, 4, 2)
    AP_GO(4, 2, 4)
    AP_GO(2, 4, 2)
    AP_GO(2, 2, 4)
    AP_GO(2, 1, 8)
    AP_GO(1, 2, 4)
#undef AP_GO
    return false;
}

template bool launch_gemmb<AP_BITS>(const GemmbGeometry &, const uint16_t *, const GemmbMembers &, int, int, hipStream_t);

}  // namespace ap
