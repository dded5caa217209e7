// Instantiates the mid-batch kernel for rows off their lines (sg_line_kernel.h) and exposes the launcher the dispatcher in
// sg_api.hip calls.
#include "sg_line_kernel.h"
#include "sg_host.h"

namespace sg {

template <int RGW, int MH, int WN, int DEPTH>
static int launch_one(const StreamArgs& a, unsigned grid, hipStream_t stream) {
    constexpr size_t lds = (size_t)DEPTH * (16 * RGW * WN + 32 * MH) * 128;
    static_assert(lds <= 160 * 1024, "LDS");
    auto kernel = line_gemm_kernel<RGW, MH, WN, DEPTH>;
    static LdsGranted granted;
    if (int rc = request_dynamic_lds(reinterpret_cast<const void*>(kernel), lds, granted)) return rc;
    kernel<<<dim3(grid), dim3(WN * 128), lds, stream>>>(a);
    return report_hip("line_gemm_kernel launch", hipGetLastError()) == hipSuccess ? SG_SUCCESS : SG_LAUNCH_FAILED;
}

int launch_line(int rgw, int mh, int wn, const StreamArgs& a, unsigned grid, hipStream_t stream) {
#define SG_LINE(RGW_, MH_, WN_, DEPTH_) \
    if (rgw == RGW_ && mh == MH_ && wn == WN_) return launch_one<RGW_, MH_, WN_, DEPTH_>(a, grid, stream);
    SG_LINE(2, 2, 2, 9)                                            // 64 x 64 on four waves
    SG_LINE(2, 2, 4, 6) SG_LINE(2, 4, 4, 5) SG_LINE(2, 6, 4, 4)    // 128 x 64, 128 x 128, 128 x 192 on eight
    SG_LINE(3, 4, 4, 4)                                            // 192 x 128
#undef SG_LINE
    return SG_INVALID_CONFIG;
}

}  // namespace sg
