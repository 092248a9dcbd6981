// MoE grouped MXFP8 and MXFP4 GEMM over row groups whose weights are stored [G, K, N], N contiguous:
//   out[rows of g] = A[rows of g] . B[g]
// the backward product of a layer that keeps its weights as the forward product reads them (128-byte slabs of
// B are copied into the LDS as they lie and transposed as they are read, see read_transposed). The transposed copy of
// the codes that this saves the weights' quantizer is a quarter of its bytes: 32 x 4096 x 4096 364 -> 257 us, MXFP4 32 x 7168 x 2048
// 280 -> 215. The product against
// that on the transposed codes: 256 x 256 tiles 555 / 559 us (32768 tokens on those weights), 128 x 128 tiles 244 / 252 (8192).
// (Semantics: the dgrad of Primus-Turbo's grouped MXFP8 path, primus_turbo/pytorch/ops/grouped_gemm_fp8.py:604-840, which reads
// a transposed quantization of the same 32 x 32 blocks; the same bits.)
#include "gemm_fp8_kernel.h"

namespace pt {

template <int FA, int FB> static int launch_kn_tiles(const GemmArgs &a, hipStream_t stream) {
    // the tiles of pt_grouped_gemm_mx, by its rule
    if (mx_rows_tile(a, FA == 4) == 1)
        return launch_gemm_cfg<8, 8, SCALE_MX, false, FA, FB, GROUP_ROWS, 2, 1, true>(a, stream);
    // (MXFP4: 128 columns are 64 bytes of a K row, and a copy is paid by the row; 128 x 256 tiles read whole 128-byte lines: 32
    // groups of 256 rows, N 2048, K 7168 156 us on 128 x 128 tiles, 126 on these. Against the transposed codes on 128 x 128: N = K =
    // 4096, 64 rows a group 105 / 77 even, 100 / 92 uneven, 256 rows 132 / 133, 145 / 137; N 2048, K 7168 105 / 126.)
    constexpr int TN = FA == 4 ? 8 : 4;
    return launch_gemm_cfg<4, TN, SCALE_MX, false, FA, FB, GROUP_ROWS, 2, 1, true>(a, stream);
}

} // namespace pt

using namespace pt;

extern "C" int pt_grouped_gemm_mx_kn(const void *a, int a_dtype, const void *a_words, const void *b, int b_dtype,
                                     const void *b_words, void *c, int c_dtype, const int64_t *group_offs,
                                     const int64_t *group_offs_out, int64_t G, int64_t a_rows, int64_t out_rows, int64_t N,
                                     int64_t K, void *stream) {
    const bool fp4 = a_dtype == PT_DTYPE_E2M1X2;
    PT_REQUIRE(fp4 ? b_dtype == PT_DTYPE_E2M1X2 : (is_fp8_dtype(a_dtype) && is_fp8_dtype(b_dtype)),
               "operands must both be fp8 (e4m3 / e5m2) or both e2m1x2");
    PT_REQUIRE(is_hp_dtype(c_dtype), "output must be bf16, fp16 or fp32");
    PT_REQUIRE(G >= 0 && a_rows >= 0 && out_rows >= 0 && N >= 0, "bad dimensions");
    PT_REQUIRE(reads_kn(N, K, fp4), "K must be whole slabs (128, e2m1x2 256), at least four, N a multiple of 16 (32), B below 2^31 bytes a group");
    auto st = static_cast<hipStream_t>(stream);
    if (out_rows == 0 || N == 0)
        return PT_OK;
    PT_REQUIRE(c && group_offs, "NULL pointer");
    PT_REQUIRE(aligned_to(c, 16), "output must be 16-byte aligned");
    if (G == 0 || a_rows == 0)
        return launch_zero_rows(c, group_offs_out ? group_offs_out : group_offs, G, out_rows, N * (c_dtype == PT_DTYPE_F32 ? 4 : 2), st);
    PT_REQUIRE(a && b && a_words && b_words, "NULL tensor pointer");
    PT_REQUIRE(aligned_to(a, 16) && aligned_to(b, 16), "operands must be 16-byte aligned");
    GemmArgs g{};
    g.A              = static_cast<const uint8_t *>(a);
    g.B              = static_cast<const uint8_t *>(b);
    g.C              = c;
    g.sA             = static_cast<const float *>(a_words); // [K / 128, a_rows] words of four E8M0 bytes
    g.sB             = static_cast<const float *>(b_words); // [G, K / 128, N]
    g.M              = a_rows;
    g.N              = N;
    g.K              = fp4 ? K / 2 : K; // bytes
    g.lda            = g.K;
    g.ldb            = fp4 ? N / 2 : N;
    g.b_kn           = true;
    g.sa_wpitch      = a_rows * 4;
    g.sb_wpitch      = N * 4;
    g.kb_valid       = static_cast<int>(K / 32);
    g.out_dtype      = c_dtype;
    g.G              = static_cast<int>(G);
    g.group_offs     = group_offs;
    g.group_offs_out = group_offs_out;
    g.b_gstride      = g.ldb * K;
    g.sb_gstride     = K / 128 * N;
    g.out_rows       = out_rows;
    if (fp4)
        return launch_kn_tiles<4, 4>(g, st);
    const bool fa = a_dtype == PT_DTYPE_E5M2, fb = b_dtype == PT_DTYPE_E5M2;
    if (!fa && !fb)
        return launch_kn_tiles<0, 0>(g, st);
    if (!fa)
        return launch_kn_tiles<0, 1>(g, st);
    return fb ? launch_kn_tiles<1, 1>(g, st) : launch_kn_tiles<1, 0>(g, st);
}
