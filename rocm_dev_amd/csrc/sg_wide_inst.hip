// Instantiates the wide-tile kernel (sg_wide_kernel.h) and exposes the launcher the dispatcher in sg_api.hip calls.
#include <type_traits>

#include "sg_wide_kernel.h"
#include "sg_host.h"

namespace sg {

template <int RGW, int MH, int WN, int DW, int DX, bool TAIL>
static int launch_one(const StreamArgs& a, unsigned grid, hipStream_t stream) {
    constexpr size_t ring = ((size_t)DW * 16 * RGW * WN + (size_t)DX * 32 * MH) * 128;
    constexpr size_t out = (size_t)WN * 2 * 16 * MH * (32 * RGW + 16);    // the epilogue's copy of the tile
    constexpr size_t lds = ring > out ? ring : out;
    static_assert(lds <= 160 * 1024, "LDS");
    auto kernel = wide_gemm_kernel<RGW, MH, WN, DW, DX, TAIL>;
    static LdsGranted granted;
    if (int rc = request_dynamic_lds(reinterpret_cast<const void*>(kernel), lds, granted)) return rc;
    kernel<<<dim3(grid), dim3(WN * 128), lds, stream>>>(a);
    return report_hip("wide_gemm_kernel launch", hipGetLastError()) == hipSuccess ? SG_SUCCESS : SG_LAUNCH_FAILED;
}

int launch_wide(int rgw, int mh, const StreamArgs& a, unsigned grid, hipStream_t stream) {
    const bool tail = (a.k & 127) != 0;
#define SG_WIDE(RGW_, MH_, DW_, DX_)                                                                                  \
    if (rgw == RGW_ && mh == MH_)                                                                                     \
        return tail ? launch_one<RGW_, MH_, 2, DW_, DX_, true>(a, grid, stream) : launch_one<RGW_, MH_, 2, DW_, DX_, false>(a, grid, stream);
    SG_WIDE(4, 8, 4, 3) SG_WIDE(5, 8, 3, 3) SG_WIDE(6, 8, 4, 2) SG_WIDE(7, 8, 3, 2) SG_WIDE(8, 8, 3, 2)   // 128 .. 256 x 256
    SG_WIDE(4, 4, 4, 4) SG_WIDE(8, 4, 4, 2)                                                               // 128, 256 x 128
#undef SG_WIDE
    return SG_INVALID_CONFIG;
}

}  // namespace sg
