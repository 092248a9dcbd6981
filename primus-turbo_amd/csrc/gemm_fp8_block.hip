// hipcc-flags: -mllvm -amdgpu-mfma-vgpr-form=1
// BLOCK-scale instantiations of the FP8 GEMM kernel. Every MFMA result of this mode is an
// input of VALU FMAs (the per-128-K-block scale is applied outside the matrix core), so this
// translation unit is compiled with MFMA destinations in architectural VGPRs: results in
// accumulation registers would cost one v_accvgpr_read per element on top of each FMA.
#include "gemm_fp8_block8.h"

namespace pt {

template <bool SB_VEC, int FA, int FB>
static int launch_block_tiles(const GemmArgs &a, int tile_cfg, hipStream_t stream) {
    // tile_cfg: 0 = auto, 1 and 4 = 256x256 with eight wavefronts, 2 = 256x128 (per-column B scales: as 3),
    // 3 = 128x128 (two workgroups per CU)
    // (Per-column B scales, the weight gradient of the blockwise recipe, us: 256x256 with eight wavefronts /
    // 256x128 / 128x128: 8192^3 522 / 651 / 661, 4096 x 7168 x 4096 127 / 164 / 144, 2048 x 2048 x 8192 106 / 81
    // / 59, 5120 x 4096 x 2048 66 / 68 / 54; 128 x 128 B blocks: 454 / 566 / 574, 112 / 142 / 131, 87 / 64 / 48,
    // 57 / 56 / 49.)
    if constexpr (!SB_VEC) {
        if (a.b_kn) // (block_nn_in_place has looked at the tile)
            return launch_gemm_block8<FA, FB, GROUP_NONE, false, true>(a, stream);
    }
    if (tile_cfg == 0)
        tile_cfg = dense_tile<SCALE_BLOCK>(a.M, a.N, a.K / KSTEP, !SB_VEC);
    if (tile_cfg == 1 || tile_cfg == 4)
        return launch_gemm_block8<FA, FB, GROUP_NONE, SB_VEC>(a, stream);
    if constexpr (!SB_VEC) {
        if (tile_cfg == 2)
            return launch_gemm_cfg<8, 4, SCALE_BLOCK, SB_VEC, FA, FB>(a, stream);
    }
    if (two_teams(SCALE_BLOCK, SB_VEC, a.M, a.N, a.K / KSTEP))
        return launch_gemm_cfg<4, 4, SCALE_BLOCK, SB_VEC, FA, FB, GROUP_NONE, 2, 2>(a, stream);
    return launch_gemm_cfg<4, 4, SCALE_BLOCK, SB_VEC, FA, FB>(a, stream);
}

template <bool SB_VEC>
static int launch_block_fmt(const GemmArgs &a, int fa, int fb, int tile_cfg, hipStream_t stream) {
    if (fa == 0 && fb == 0)
        return launch_block_tiles<SB_VEC, 0, 0>(a, tile_cfg, stream);
    if (fa == 0 && fb == 1)
        return launch_block_tiles<SB_VEC, 0, 1>(a, tile_cfg, stream);
    if (fa == 1 && fb == 0)
        return launch_block_tiles<SB_VEC, 1, 0>(a, tile_cfg, stream);
    return launch_block_tiles<SB_VEC, 1, 1>(a, tile_cfg, stream);
}

int launch_gemm_block(const GemmArgs &a, int fa, int fb, bool sb_vec, int tile_cfg, hipStream_t stream) {
    return sb_vec ? launch_block_fmt<true>(a, fa, fb, tile_cfg, stream)
                  : launch_block_fmt<false>(a, fa, fb, tile_cfg, stream);
}

} // namespace pt
