// Instantiates the skinny kernels for rows off their lines (sg_skinny_line_kernel.h) and exposes the launchers the dispatcher
// in sg_api.hip calls.
#include "sg_skinny_line_kernel.h"
#include "sg_host.h"

namespace sg {

template <int MT, int RG, int XU, int DEPTH>
static int launch_tile(const StreamArgs& a, unsigned grid, unsigned threads, size_t lds, hipStream_t stream) {
    if (threads > 512) return SG_INVALID_CONFIG;
    auto kernel = skinny_line_kernel<MT, RG, XU, DEPTH>;
    static LdsGranted granted;
    if (int rc = request_dynamic_lds(reinterpret_cast<const void*>(kernel), lds, granted)) return rc;
    kernel<<<dim3(grid), dim3(threads), lds, stream>>>(a);
    return report_hip("skinny_line_kernel launch", hipGetLastError()) == hipSuccess ? SG_SUCCESS : SG_LAUNCH_FAILED;
}
template <int MT, int XU, int DEPTH>
static int launch_resident(const StreamArgs& a, unsigned grid, unsigned threads, size_t lds, hipStream_t stream) {
    if (threads > 512) return SG_INVALID_CONFIG;
    auto kernel = skinny_line_resident_kernel<MT, XU, DEPTH>;
    static LdsGranted granted;
    if (int rc = request_dynamic_lds(reinterpret_cast<const void*>(kernel), lds, granted)) return rc;
    kernel<<<dim3(grid), dim3(threads), lds, stream>>>(a);
    return report_hip("skinny_line_resident_kernel launch", hipGetLastError()) == hipSuccess ? SG_SUCCESS : SG_LAUNCH_FAILED;
}

int launch_skinny_line(int mt, int rg, int xu, int depth, bool resident, const StreamArgs& a, unsigned grid, unsigned threads, size_t lds,
                       hipStream_t stream) {
#define SG_RES(MT_, XU_, DEPTH_) \
    if (resident && mt == MT_ && rg == 1 && xu == XU_ && depth == DEPTH_) return launch_resident<MT_, XU_, DEPTH_>(a, grid, threads, lds, stream);
#define SG_TILE(MT_, RG_, XU_, DEPTH_) \
    if (!resident && mt == MT_ && rg == RG_ && xu == XU_ && depth == DEPTH_) return launch_tile<MT_, RG_, XU_, DEPTH_>(a, grid, threads, lds, stream);
    // what skinny_line_config (sg_api.hip) chooses from
    SG_RES(1, 1, 3) SG_RES(1, 1, 4) SG_RES(1, 2, 3) SG_RES(1, 2, 4) SG_RES(1, 4, 3) SG_RES(1, 4, 4) SG_RES(2, 8, 3) SG_RES(2, 8, 4)
    SG_TILE(1, 1, 1, 4) SG_TILE(1, 1, 2, 4) SG_TILE(1, 1, 4, 4)
    SG_TILE(1, 2, 1, 3) SG_TILE(1, 2, 1, 4) SG_TILE(1, 2, 2, 3) SG_TILE(1, 2, 2, 4) SG_TILE(1, 2, 4, 3) SG_TILE(1, 2, 4, 4)
    SG_TILE(1, 4, 4, 3)
    SG_TILE(2, 1, 8, 4) SG_TILE(2, 2, 8, 4) SG_TILE(2, 4, 8, 3)
#undef SG_TILE
#undef SG_RES
    return SG_INVALID_CONFIG;
}

}  // namespace sg
