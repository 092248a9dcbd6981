// hipcc-flags: -mllvm -amdgpu-mfma-vgpr-form=1
// Instantiations of the GEMM for few output tiles (gemm_direct.h), all scaling modes and formats. Its sums
// are read once at the end by every lane, so they live in architectural VGPRs.
#include "gemm_direct.h"

namespace pt {

template <int MODE, bool SB_VEC> static int launch_fmt(const GemmArgs &a, int fa, int fb, int tile, hipStream_t stream) {
    if (fa == 0 && fb == 0)
        return launch_gemm_direct<MODE, SB_VEC, 0, 0>(a, tile, stream);
    if (fa == 0 && fb == 1)
        return launch_gemm_direct<MODE, SB_VEC, 0, 1>(a, tile, stream);
    if (fa == 1 && fb == 0)
        return launch_gemm_direct<MODE, SB_VEC, 1, 0>(a, tile, stream);
    return launch_gemm_direct<MODE, SB_VEC, 1, 1>(a, tile, stream);
}

int gemm_direct_tile(int64_t M, int64_t N, int64_t row_bytes, int mode, bool fp4) {
    return direct_tile(M, N, cdiv(row_bytes, KSTEP), mode, fp4);
}

int launch_gemm_direct_mode(const GemmArgs &a, int mode, bool sb_vec, int fa, int fb, int tile, hipStream_t stream) {
    if (mode == SCALE_VECTOR)
        return launch_fmt<SCALE_VECTOR, false>(a, fa, fb, tile, stream);
    if (mode == SCALE_BLOCK)
        return sb_vec ? launch_fmt<SCALE_BLOCK, true>(a, fa, fb, tile, stream) : launch_fmt<SCALE_BLOCK, false>(a, fa, fb, tile, stream);
    if (fa == 4)
        return launch_gemm_direct<SCALE_MX, false, 4, 4>(a, tile, stream);
    return launch_fmt<SCALE_MX, false>(a, fa, fb, tile, stream);
}

} // namespace pt
