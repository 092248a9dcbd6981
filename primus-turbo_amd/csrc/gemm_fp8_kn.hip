// Dense FP8 products with vector scales (TENSORWISE, ROWWISE) whose operands are not contiguous along the reduction: B stored
// [K, N], and A stored [K, M] as well. Slabs are copied into the LDS as they lie and transposed as they are read
// (read_transposed), where other tiles want a transposed copy in memory. What a TENSORWISE layer's backward products read:
// the forward codes of weight, activation and gradient, whose casts then write one layout (4096^2 17 -> 12 us each). The
// products take 4 (B) and up to 3 % (both) longer than on transposed copies. A whole training step, with copies / in place, us:
// 4096^3 206 / 200, 8192 x 2048 x 8192 422 / 411, 4096 x 8192 x 8192 716 / 705, 8192^3 1298 / 1290, 8192 x 4096 x 4096 379 / 374.
#include "gemm_fp8_kernel.h"

namespace pt {

template <int FA, int FB> static int launch_kn(const GemmArgs &a, bool at, hipStream_t stream) {
    if (at)
        return launch_gemm_cfg<8, 8, SCALE_VECTOR, false, FA, FB, GROUP_NONE, 2, 1, true, true>(a, stream);
    return launch_gemm_cfg<8, 8, SCALE_VECTOR, false, FA, FB, GROUP_NONE, 2, 1, true>(a, stream);
}

int launch_gemm_vector_kn(const GemmArgs &a, int fa, int fb, bool at, hipStream_t stream) {
    if (fa == 0)
        return fb == 0 ? launch_kn<0, 0>(a, at, stream) : launch_kn<0, 1>(a, at, stream);
    return fb == 0 ? launch_kn<1, 0>(a, at, stream) : launch_kn<1, 1>(a, at, stream);
}

} // namespace pt
