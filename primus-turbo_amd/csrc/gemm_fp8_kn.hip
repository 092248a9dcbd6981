// Dense FP8 products with vector scales (TENSORWISE, ROWWISE) whose operands are not contiguous along the reduction: B stored
// [K, N], and A stored [K, M] as well. Slabs are copied into the LDS as they lie and transposed as they are read
// (read_transposed), where other tiles want a transposed copy in memory. What a TENSORWISE layer's backward products read:
// the forward codes of weight, activation and gradient, whose casts then write one layout (4096^2 17 -> 12 us each). The
// products take longer than on transposed copies, 3 to 4 % with B in place, 5 to 6 % with both (us, copies / B / both: 4096^3 52.1 /
// 53.8 / 54.6, 8192 x 4096 x 4096 101.4 / 105.8 / 107.4, 4096 x 8192 x 8192 183.0 / 188.7 / 192.1, 8192^3 365 / 379 / 382): a
// fragment takes four LDS reads instead of two. A whole training step, copies / in place, us: 4096^3 210.1 / 204.4, 8192 x 8192 x 2048
// 428 / 414, 4096 x 8192 x 8192 734 / 716, 8192 x 4096 x 4096 397.5 / 392.6, 16384 x 4096 x 8192 1402 / 1363 (7 runs of either in turn, which
// differ by 1 % or less); adding the weight gradient into fp32 231.3 / 225.4, 450 / 432, 829 / 806, 418.0 / 418.5, 1456 / 1411.
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
