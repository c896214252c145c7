// The dense UE8M0 tiles that dense_schedule (gemm.hip) picks for more than 64
// rows where 128x128 or 256x256 tiles would leave CUs idle or split K over
// them; kernels in gemm_kernel.h.  Built with the VGPR-form MFMA option, as
// gemm.hip, in its own translation unit so the two compile side by side.
#include "gemm_kernel.h"

namespace kbn {

template <bool kRowW>
static int launch_mid(const GemmArgs& a, const Schedule& sc, hipStream_t st, const char* what) {
    if (sc.bm == 128 && sc.bn == 64 && sc.stages == 4)
        return launch_gemm<128, 64, 4, true, false, 4, 0, kRowW>(a, sc, st, what);
    if (sc.bm == 64 && sc.bn == 256 && sc.stages == 3)
        return launch_gemm<64, 256, 3, true, false, 4, 0, kRowW>(a, sc, st, what);
    if (sc.bm == 128 && sc.bn == 256 && sc.stages == 3 && sc.waves == 8)
        return launch_gemm<128, 256, 3, true, false, 8, 0, kRowW>(a, sc, st, what);
    if (sc.bm == 256 && sc.bn == 128 && sc.stages == 3)
        return launch_gemm<256, 128, 3, true, false, 4, 0, kRowW>(a, sc, st, what);
    set_error("%s: no kernel for %dx%d tiles", what, sc.bm, sc.bn);
    return 1;
}

int launch_gemm_mid(const GemmArgs& a, const Schedule& sc, hipStream_t st, const char* what) {
    return launch_mid<false>(a, sc, st, what);
}

// The same tiles with packed per-row UE8M0 weight scales (GemmArgs::sWp).
int launch_gemm_mid_roww(const GemmArgs& a, const Schedule& sc, hipStream_t st, const char* what) {
    return launch_mid<true>(a, sc, st, what);
}

}  // namespace kbn
