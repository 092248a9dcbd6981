// Scaled FP8 / MX GEMM for products with few output tiles:  C[M, N] = scale( A . B^T ),  both operands
// K-contiguous, arguments and scaling modes of gemm_fp8_nt_kernel (a decoding step's sixteen tokens against
// a projection, a few hundred tokens against a narrow one).
//
// What bounds the tiled kernel there: its 128 x 128 tile gives such a product a few dozen workgroups, each
// with all of K in front of it and one copy pipeline to hide the memory latency with. 16 x 4096 x 4096 was
// 32 workgroups on 256 CUs walking 32 slabs, 17.5 us, where its 16 MB of weights take 3.1.
//
// This kernel instead
//   * takes tiles of 16 RM x 16 RN, small enough that they fill the machine;
//   * splits K over the wavefronts of the workgroup, slab by slab in turn (consecutive 128-byte pieces of a
//     row are requested side by side), so the chain of every wavefront is K / (128 W) MFMAs long. The
//     partial sums meet in the LDS and are added in a fixed order: no second launch, no workspace, the same
//     bits every time;
//   * loads MFMA fragments straight into registers: no wavefront shares its slab with another, so a stage in
//     the LDS would only add a barrier and a round trip. P slabs per wavefront are in flight;
//   * reads rows of any length that is a multiple of 16 bytes: chunks behind the end of K are out of the
//     buffer's range and read as zero, so nothing is padded by a copy.
// What it pays: a workgroup fetches (RM + RN) rows of 2 KB a slab for RM RN MFMAs, at 40 to 50 bytes a
// nanosecond and CU; direct_tile() below compares that with the tiled kernel.
#pragma once
#include "gemm_fp8_kernel.h"

namespace pt {

template <int RM, int RN, int W, int P, int MODE, bool SB_VEC, int FA, int FB>
__global__ __launch_bounds__(W * 64) void gemm_direct_kernel(const GemmArgs a) {
    constexpr bool F4 = FA == 4;
    static_assert((FA == 4) == (FB == 4), "FP4 operands come in pairs");
    constexpr int NH  = F4 ? 2 : 1; // MFMAs per slab and tile: an MXFP4 slab holds 256 codes of a row
    constexpr int BM  = 16 * RM, BN = 16 * RN;
    constexpr int LDR = BN + 4; // floats per row of a wavefront's partial result
    __shared__ __attribute__((aligned(16))) float red[W * BM * LDR];

    const int tid = threadIdx.x, lane = tid & 63, lm = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int id   = xcd_contiguous_id(blockIdx.x, a.tiles_m * a.tiles_n);
    const int tn = id / a.tiles_m, tm = id - tn * a.tiles_m;

    const int64_t  m0 = static_cast<int64_t>(tm) * BM, n0 = static_cast<int64_t>(tn) * BN;
    const int      rows_a = a.M - m0 < BM ? static_cast<int>(a.M - m0) : BM, rows_b = a.N - n0 < BN ? static_cast<int>(a.N - n0) : BN;
    const uint8_t *Ap = a.A + m0 * a.lda, *Bp = a.B + n0 * a.ldb;
    const uint32_t end_a = static_cast<uint32_t>((rows_a - 1) * a.lda + a.K), end_b = static_cast<uint32_t>((rows_b - 1) * a.ldb + a.K);
    const uint32_t K = static_cast<uint32_t>(a.K), slabs = (K + KSTEP - 1) / KSTEP;
    const uint32_t row_a = lm * static_cast<uint32_t>(a.lda) + lg * 16, row_b = lm * static_cast<uint32_t>(a.ldb) + lg * 16;

    struct Slab {
        i32x8    fa[RM], fb[RN];
        uint32_t sa[RM][NH], sb[RN][SB_VEC ? 4 : NH];
    };
    // Out of range of every buffer: such a load returns zero
    constexpr uint32_t NOWHERE = 0x7f000000u;

    auto load = [&](Slab &s, const uint32_t kt) {
#if defined(__HIP_DEVICE_COMPILE__) // the buffer resource type only exists in the device pass
        constexpr uint32_t RSRC_FLAGS = 0x00020000;
        const bool     on   = kt < slabs;
        const uint32_t k0   = on ? kt * KSTEP : 0u;
        const uint32_t left = K - k0; // bytes of K from the slab on
        const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(Ap + k0), 0, on ? end_a - k0 : 0u, RSRC_FLAGS);
        const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(Bp + k0), 0, on ? end_b - k0 : 0u, RSRC_FLAGS);
        const uint32_t lo = lg * 16u < left ? 0u : NOWHERE, hi = 64u + lg * 16u < left ? 64u : NOWHERE;
        auto frag = [&](const __amdgpu_buffer_rsrc_t &r, const uint32_t off) {
            const u32x4 l = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off + lo, 0, 0));
            const u32x4 h = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off + hi, 0, 0));
            i32x8       f;
            f[0] = l.x; f[1] = l.y; f[2] = l.z; f[3] = l.w;
            f[4] = h.x; f[5] = h.y; f[6] = h.z; f[7] = h.w;
            return f;
        };
#pragma unroll
        for (int j = 0; j < RN; ++j)
            s.fb[j] = frag(rb, row_b + 16 * j * static_cast<uint32_t>(a.ldb));
#pragma unroll
        for (int i = 0; i < RM; ++i)
            s.fa[i] = frag(ra, row_a + 16 * i * static_cast<uint32_t>(a.lda));
        if constexpr (MODE == SCALE_MX) {
            // row-major or word-major scales, each operand for itself (see GemmArgs)
            const uint32_t nkb   = static_cast<uint32_t>(a.kb_valid);
            const uint32_t rowpa = a.sa_wpitch != 0 ? 4u : static_cast<uint32_t>(a.sa_m), rowpb = a.sb_wpitch != 0 ? 4u : static_cast<uint32_t>(a.sb_n);
            const int64_t  wordpa = a.sa_wpitch != 0 ? a.sa_wpitch : 4, wordpb = a.sb_wpitch != 0 ? a.sb_wpitch : 4;
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                const uint32_t word = on ? kt * NH + h : 0u;
                const bool     some = on && 4 * word < nkb;
                const uint8_t *sA = reinterpret_cast<const uint8_t *>(a.sA) + m0 * rowpa + word * wordpa;
                const uint8_t *sB = reinterpret_cast<const uint8_t *>(a.sB) + n0 * rowpb + word * wordpb;
                const __amdgpu_buffer_rsrc_t qa = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(sA), 0, some ? (rows_a - 1) * rowpa + 4u : 0u, RSRC_FLAGS);
                const __amdgpu_buffer_rsrc_t qb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(sB), 0, some ? (rows_b - 1) * rowpb + 4u : 0u, RSRC_FLAGS);
                const uint32_t off = 4 * word + lg < nkb ? static_cast<uint32_t>(lg) : NOWHERE;
#pragma unroll
                for (int i = 0; i < RM; ++i)
                    s.sa[i][h] = __builtin_amdgcn_raw_buffer_load_b8(qa, (16 * i + lm) * rowpa + off, 0, 0);
#pragma unroll
                for (int j = 0; j < RN; ++j)
                    s.sb[j][h] = __builtin_amdgcn_raw_buffer_load_b8(qb, (16 * j + lm) * rowpb + off, 0, 0);
            }
        }
        if constexpr (MODE == SCALE_BLOCK) {
            const float *sA = a.sA + (m0 >> a.sa_shift) * a.sa_m + (on ? kt : 0u) * a.sa_k, *sB = a.sB + (n0 >> a.sb_shift) * a.sb_n + (on ? kt : 0u) * a.sb_k;
            const __amdgpu_buffer_rsrc_t qa = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float *>(sA), 0, on ? static_cast<uint32_t>(((rows_a - 1) >> a.sa_shift) * a.sa_m + 1) * 4u : 0u, RSRC_FLAGS);
            const __amdgpu_buffer_rsrc_t qb = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float *>(sB), 0, on ? static_cast<uint32_t>(((rows_b - 1) >> a.sb_shift) * a.sb_n + 1) * 4u : 0u, RSRC_FLAGS);
#pragma unroll
            for (int i = 0; i < RM; ++i)
                s.sa[i][0] = __builtin_amdgcn_raw_buffer_load_b32(qa, ((16 * i + lm) >> a.sa_shift) * static_cast<uint32_t>(a.sa_m) * 4u, 0, 0);
            if constexpr (SB_VEC) {
#pragma unroll
                for (int j = 0; j < RN; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        s.sb[j][e] = __builtin_amdgcn_raw_buffer_load_b32(qb, (16 * j + 4 * lg + e) * static_cast<uint32_t>(a.sb_n) * 4u, 0, 0);
            } else { // (a tile lies within one 128-wide block of columns)
                s.sb[0][0] = __builtin_amdgcn_raw_buffer_load_b32(qb, 0, 0, 0);
            }
        }
#endif
    };

    f32x4 acc[RM][RN];
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j)
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto multiply = [&](const Slab &s) {
#if defined(__HIP_DEVICE_COMPILE__)
        [[maybe_unused]] constexpr int ONE = 0x7f7f7f7f;
#pragma unroll
        for (int j = 0; j < RN; ++j)
#pragma unroll
            for (int i = 0; i < RM; ++i) {
                if constexpr (MODE == SCALE_VECTOR) {
                    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(s.fb[j], s.fa[i], acc[i][j], FB, FA, 0, ONE, 0, ONE);
                } else if constexpr (MODE == SCALE_MX && !F4) {
                    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(s.fb[j], s.fa[i], acc[i][j], FB, FA, 0, s.sb[j][0], 0, s.sa[i][0]);
                } else if constexpr (MODE == SCALE_MX) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const i32x8 b = h ? __builtin_shufflevector(s.fb[j], s.fb[j], 4, 5, 6, 7, 4, 5, 6, 7) : s.fb[j];
                        const i32x8 c = h ? __builtin_shufflevector(s.fa[i], s.fa[i], 4, 5, 6, 7, 4, 5, 6, 7) : s.fa[i];
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b, c, acc[i][j], 4, 4, 0, s.sb[j][h], 0, s.sa[i][h]);
                    }
                } else {
                    const f32x4 p = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(s.fb[j], s.fa[i], f32x4{0.f, 0.f, 0.f, 0.f}, FB, FA, 0, ONE, 0, ONE);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc[i][j][e] = fmaf(p[e], __uint_as_float(s.sa[i][0]) * __uint_as_float(s.sb[SB_VEC ? j : 0][SB_VEC ? e : 0]), acc[i][j][e]);
                }
            }
#endif
    };

    Slab s[P];
#pragma unroll
    for (int p = 0; p < P; ++p)
        load(s[p], wave + p * W);
    for (uint32_t kt = wave; kt < slabs; kt += P * W) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            multiply(s[p]);
            __builtin_amdgcn_sched_barrier(0);
            load(s[p], kt + (P + p) * W);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    float *mine = red + wave * (BM * LDR);
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j)
            *reinterpret_cast<f32x4 *>(mine + (16 * i + lm) * LDR + 16 * j + 4 * lg) = acc[i][j];
    __syncthreads();

    const bool accu = a.accumulate != 0, quads = (a.N & 3) == 0;
    constexpr int QUADS = BM * BN / 4;
    auto leave = [&](auto tag) {
        using T = decltype(tag);
        for (int q = tid; q < QUADS; q += W * 64) {
            const int m = q / (BN / 4), n = (q % (BN / 4)) * 4;
            if (m >= rows_a || n >= rows_b)
                continue;
            f32x4 v = *reinterpret_cast<const f32x4 *>(red + m * LDR + n);
#pragma unroll
            for (int w = 1; w < W; ++w)
                v += *reinterpret_cast<const f32x4 *>(red + (w * BM + m) * LDR + n);
            if constexpr (MODE == SCALE_VECTOR) {
                const float sa = a.sA[(m0 + m) * a.sa_m];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e] = v[e] * sa * a.sB[(n0 + (n + e < rows_b ? n + e : n)) * a.sb_n];
            }
            uint8_t *p = static_cast<uint8_t *>(a.C) + ((m0 + m) * a.N + n0 + n) * sizeof(T);
            if (quads) {
                store_quad<T>(v, p, accu);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < rows_b)
                        store_elem<T>(v[e], p + e * sizeof(T), accu);
            }
        }
    };
    if (a.out_dtype == PT_DTYPE_BF16)
        leave(bf16_t{});
    else if (a.out_dtype == PT_DTYPE_F16)
        leave(f16_t{});
    else
        leave(0.f);
}

// The tile shapes built, as indices of DIRECT_TILES, W wavefronts and P slabs in flight for each.
struct DirectTile {
    int rm, rn, w, p;
};
constexpr DirectTile DIRECT_TILES[] = {{1, 1, 8, 2}, {1, 2, 8, 2}, {1, 4, 8, 2}, {2, 2, 4, 2}, {2, 4, 4, 2}, {4, 4, 4, 1}};
constexpr int        DIRECT_COUNT   = sizeof(DIRECT_TILES) / sizeof(DIRECT_TILES[0]);

// Index of the tile for an M x N product over `slabs` 128-byte slabs, or -1: the tiled kernel. The cost of a
// tile shape is the rows (in 16s) that a CU fetches each slab; measured (us, 4096 x 4096 weights of random
// codes, vector scales), the tiled kernel -> this one:
//   cost 2 (16 rows) 17.4 -> 6.5, 4 (64 rows) 18.0 -> 10.0, 6 (128 rows) 18.3 -> 14.4, 8 (256 rows) 18.5 -> 18.2
// (64 x 64 tiles; the tiled kernel with four stages: 15.4). Short products pay for the tiled kernel's long
// start as well: 300 x 2880 x 512, cost 8, 6.2 -> 5.9. Block scales fold each product in the VALU, which the
// tiled kernel hides with its two teams only in part: there cost 8 pays at any length (20.6 -> 19.8, a scale per
// column 22.2 -> 20.8, 1024 x 1024 x 16384 61.4 -> 61.0). MXFP4 has half the matrix time for the same bytes (16
// slabs 13.6 -> 13.2, but 32 slabs 21.1 -> 21.8). Cost 16 loses everywhere (512 rows: 19.4 against 33.6).
static inline int direct_tile(int64_t M, int64_t N, int64_t slabs, int mode, bool fp4) {
    int     best = -1;
    int64_t least = 0;
    for (int i = 0; i < DIRECT_COUNT; ++i) {
        const DirectTile t     = DIRECT_TILES[i];
        const int64_t    tiles = cdiv(M, 16 * t.rm) * cdiv(N, 16 * t.rn);
        const int64_t    cost  = cdiv(tiles, device_cu_count()) * (t.rm + t.rn); // 2 KB pieces a CU fetches each slab
        if (best < 0 || cost < least) {
            best  = i;
            least = cost;
        }
    }
    const bool cost8_pays = mode == SCALE_BLOCK || slabs <= (fp4 ? 16 : 8);
    return least <= 6 || (least <= 8 && cost8_pays) ? best : -1;
}

template <int I, int MODE, bool SB_VEC, int FA, int FB>
static int launch_direct_tile(const GemmArgs &args_in, hipStream_t stream) {
    constexpr DirectTile T = DIRECT_TILES[I];
    GemmArgs             a = args_in;
    a.tiles_m              = static_cast<int>(cdiv(a.M, 16 * T.rm));
    a.tiles_n              = static_cast<int>(cdiv(a.N, 16 * T.rn));
    gemm_direct_kernel<T.rm, T.rn, T.w, T.p, MODE, SB_VEC, FA, FB>
        <<<static_cast<unsigned>(a.tiles_m) * static_cast<unsigned>(a.tiles_n), T.w * 64, 0, stream>>>(a);
    return check_launch("gemm_direct_kernel");
}

// `tile`: what direct_tile() gave; a.K: bytes of a row that count (a multiple of 16), a.lda / a.ldb below 2^24.
template <int MODE, bool SB_VEC, int FA, int FB, int I = 0>
static int launch_gemm_direct(const GemmArgs &a, int tile, hipStream_t stream) {
    if (tile == I)
        return launch_direct_tile<I, MODE, SB_VEC, FA, FB>(a, stream);
    if constexpr (I + 1 < DIRECT_COUNT)
        return launch_gemm_direct<MODE, SB_VEC, FA, FB, I + 1>(a, tile, stream);
    return fail(PT_ERR_INVALID_ARGUMENT, "gemm_direct: no such tile");
}

} // namespace pt
