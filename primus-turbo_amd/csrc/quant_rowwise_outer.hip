// Rowwise FP8 quantization along an axis that is not the contiguous one: x viewed as [B, M, N], one
// scale per (b, n), the abs-max taken over M (semantics of Primus-Turbo's quantize_fp8_rowwise for
// axis != -1, csrc/pytorch/quantization/quantization.cpp:110-208).
//
// Two launches: column abs-max of row chunks into a small array of partial maxima, then scale and
// cast. Both walk rows with 8 columns per lane, eight rows requested back to back; the second launch
// reads its columns' partial maxima (at most 64 x 512 floats from the L2) and so needs neither a
// zero-fill and atomics before it nor a scale_inv pass behind it. A wavefront covers 512 columns of one
// row or, in a narrower matrix, several rows; a matrix with more rows than 64 chunks are good for takes a
// third launch, after which the maxima of any number of chunks meet by atomics (outer_plan).
//
// What it reads and how it writes are template choices:
//   * the source is the 16- / 32-bit tensor, or FP8 codes with a scale per row: the value is then the
//     code times its row's scale rounded to the 16- / 32-bit type, i.e. de-quantize + quantize in one
//     step with the same bits (the backward operands of a ROWWISE product are the forward codes
//     quantized again along their other axis);
//   * the codes leave in place ([B, M, N]) or transposed ([B, N, ldt], rows M .. ldt zero): the
//     transposed form is the K-contiguous operand of the products that reduce over M.
//
// Bound by memory traffic. 3001 x 4096 bf16 (24.6 MB in, 12.3 MB out) from memory, same box: the launches
// before these (one 2-byte load in flight per lane, four rows of 64 columns per workgroup and step, 12 row
// chunks) took 33.6 us for the maxima and 66.7 us for the cast, plus 9.5 us of zero-fill and scale
// launches; these take 10.1 and 9.3 us. 16384 x 16384: 307 + 326 us, now 151 + 174 (4.1 TB/s over both
// reads and the write).
#include "pt_common.h"

namespace pt {

// ---- sources: eight (or one) consecutive columns of a row as floats ----
template <typename T> struct OuterSrcHP {
    static constexpr bool IN_PLACE = true; // codes may also leave untransposed
    const T              *x;
    int64_t               ld; // elements from one row to the next
    struct Raw {
        u32x4 v[sizeof(T) / 2];
    };
    __device__ __forceinline__ Raw load8(int64_t /*row*/, int64_t off) const {
        Raw r;
#pragma unroll
        for (unsigned i = 0; i < sizeof(T) / 2; ++i)
            r.v[i] = ld128(reinterpret_cast<const char *>(x + off) + 16 * i);
        return r;
    }
    __device__ __forceinline__ void get8(const Raw &r, float (&f)[8]) const {
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    f[4 * i + e] = __uint_as_float(r.v[i][e]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                unpack2<T>(r.v[0][e], f[2 * e], f[2 * e + 1]);
        }
    }
    __device__ __forceinline__ float get1(int64_t /*row*/, int64_t off) const { return HP<T>::to_f32(x[off]); }
};

template <typename T, bool SRC_E5M2> struct OuterSrcCodes {
    static constexpr bool IN_PLACE = false;
    const uint8_t        *q;
    int64_t               ld;
    const float          *row_scale; // scale_inv of row b * M + m
    struct Raw {
        u32x2 v;
        float s;
    };
    __device__ __forceinline__ Raw load8(int64_t row, int64_t off) const {
        return Raw{*reinterpret_cast<const u32x2 *>(q + off), row_scale[row]};
    }
    static __device__ __forceinline__ float value(float code, float s) { return HP<T>::to_f32(HP<T>::from_f32(code * s)); }
    __device__ __forceinline__ void get8(const Raw &r, float (&f)[8]) const {
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            f[4 * w + 0] = value(fp8_to_f32<SRC_E5M2>(r.v[w], 0), r.s);
            f[4 * w + 1] = value(fp8_to_f32<SRC_E5M2>(r.v[w], 1), r.s);
            f[4 * w + 2] = value(fp8_to_f32<SRC_E5M2>(r.v[w], 2), r.s);
            f[4 * w + 3] = value(fp8_to_f32<SRC_E5M2>(r.v[w], 3), r.s);
        }
    }
    __device__ __forceinline__ float get1(int64_t row, int64_t off) const {
        return value(fp8_to_f32<SRC_E5M2>(q[off], 0), row_scale[row]);
    }
};

constexpr int RO_ROWS = 8; // rows a lane requests back to back

// Abs-max of a row chunk for VEC << lc columns: part[(b * chunks + chunk) * N + n], or an integer atomic
// max into amax[b * N + n] (non-negative floats order like integers). 1 << lc lanes share a row, so a
// wavefront covers 64 >> lc rows at once.
template <typename SRC, int VEC, bool ATOMIC>
__global__ __launch_bounds__(256) void col_amax_kernel(const SRC src, float *__restrict__ out, const int64_t M, const int64_t N,
                                                       const int64_t rows_per, const int lc) {
    __shared__ float s[4][64 * VEC];
    const int        lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int        W = VEC << lc, col = (lane & ((1 << lc) - 1)) * VEC, rows = 64 >> lc; // rows of a wavefront
    const int64_t    b = blockIdx.z, n = static_cast<int64_t>(blockIdx.x) * W + col;
    const int64_t    m0 = blockIdx.y * rows_per, m1 = (m0 + rows_per < M) ? m0 + rows_per : M;
    float            a[VEC] = {};
    if (n < N) {
        for (int64_t m = m0 + wave * rows + (lane >> lc); m < m1; m += 4 * RO_ROWS * rows) {
            // (a row behind the chunk's end re-reads the first one of the run: the maximum is the same)
            if constexpr (VEC == 8) {
                typename SRC::Raw r[RO_ROWS];
#pragma unroll
                for (int k = 0; k < RO_ROWS; ++k) {
                    const int64_t row = b * M + (m + 4 * k * rows < m1 ? m + 4 * k * rows : m);
                    r[k]              = src.load8(row, row * src.ld + n);
                }
#pragma unroll
                for (int k = 0; k < RO_ROWS; ++k) {
                    float f[8];
                    src.get8(r[k], f);
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        a[e] = fmaxf(a[e], fabsf(f[e]));
                }
            } else {
                float f[RO_ROWS];
#pragma unroll
                for (int k = 0; k < RO_ROWS; ++k) {
                    const int64_t row = b * M + (m + 4 * k * rows < m1 ? m + 4 * k * rows : m);
                    f[k]              = src.get1(row, row * src.ld + n);
                }
#pragma unroll
                for (int k = 0; k < RO_ROWS; ++k)
                    a[0] = fmaxf(a[0], fabsf(f[k]));
            }
        }
    }
    for (int d = 1 << lc; d < 64; d <<= 1) // the rows of the wavefront
#pragma unroll
        for (int e = 0; e < VEC; ++e)
            a[e] = fmaxf(a[e], __shfl_xor(a[e], d));
    if (lane < 1 << lc)
#pragma unroll
        for (int e = 0; e < VEC; ++e)
            s[wave][col + e] = a[e];
    __syncthreads();
    for (int c = threadIdx.x; c < W; c += 256) {
        const int64_t nc = static_cast<int64_t>(blockIdx.x) * W + c;
        if (nc < N) {
            const float v = fmaxf(fmaxf(s[0][c], s[1][c]), fmaxf(s[2][c], s[3][c]));
            if constexpr (ATOMIC)
                __hip_atomic_fetch_max(reinterpret_cast<uint32_t *>(out) + b * N + nc, __float_as_uint(v), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            else
                out[(b * gridDim.y + blockIdx.y) * N + nc] = v;
        }
    }
}

// The scale of column n: given, or from the partial maxima of its `chunks` row chunks.
__device__ __forceinline__ float outer_scale(const float *__restrict__ amax_or_scale, bool dynamic, int64_t b, int64_t n,
                                             int64_t N, int chunks, float qmax) {
    if (!dynamic)
        return amax_or_scale[b * N + n];
    float a = 0.f;
#pragma unroll 8
    for (int c = 0; c < chunks; ++c)
        a = fmaxf(a, amax_or_scale[(b * chunks + c) * N + n]);
    return qmax / fmaxf(a, 1e-12f);
}

// Codes in place. scale_inv == nullptr: another launch writes it (the maxima or scales sit in its storage).
template <typename SRC, bool E5M2, int VEC>
__global__ __launch_bounds__(256) void quant_outer_kernel(const SRC src, uint8_t *__restrict__ q,
                                                          const float *__restrict__ amax_or_scale, const bool dynamic,
                                                          const int chunks, float *__restrict__ scale_inv, const int64_t M,
                                                          const int64_t N, const int64_t rows_per, const int lc,
                                                          const float qmax) {
    __shared__ float s[64 * VEC];
    const int        lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int        W = VEC << lc, col = (lane & ((1 << lc) - 1)) * VEC, rows = 64 >> lc; // (as col_amax_kernel)
    const int64_t    b = blockIdx.z, nb = static_cast<int64_t>(blockIdx.x) * W;
    for (int c = threadIdx.x; c < W; c += 256) {
        if (nb + c < N) {
            const float sc = outer_scale(amax_or_scale, dynamic, b, nb + c, N, chunks, qmax);
            s[c]           = sc;
            if (scale_inv != nullptr && blockIdx.y == 0)
                scale_inv[b * N + nb + c] = 1.0f / sc;
        }
    }
    __syncthreads();
    const int64_t n  = nb + col;
    const int64_t m0 = blockIdx.y * rows_per, m1 = (m0 + rows_per < M) ? m0 + rows_per : M;
    if (n >= N)
        return;
    float sc[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e)
        sc[e] = s[col + e];
    for (int64_t m = m0 + wave * rows + (lane >> lc); m < m1; m += 4 * RO_ROWS * rows) {
        if constexpr (VEC == 8) {
            typename SRC::Raw r[RO_ROWS];
#pragma unroll
            for (int k = 0; k < RO_ROWS; ++k) {
                const int64_t row = b * M + (m + 4 * k * rows < m1 ? m + 4 * k * rows : m);
                r[k]              = src.load8(row, row * src.ld + n);
            }
#pragma unroll
            for (int k = 0; k < RO_ROWS; ++k) {
                float f[8];
                src.get8(r[k], f);
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    f[e] = scale_clamp(f[e], sc[e], qmax);
                if (m + 4 * k * rows < m1)
                    st64_nt(q + (b * M + m + 4 * k * rows) * N + n,
                            u32x2{cvt4_fp8<E5M2>(f[0], f[1], f[2], f[3]), cvt4_fp8<E5M2>(f[4], f[5], f[6], f[7])});
            }
        } else {
            float f[RO_ROWS];
#pragma unroll
            for (int k = 0; k < RO_ROWS; ++k) {
                const int64_t row = b * M + (m + 4 * k * rows < m1 ? m + 4 * k * rows : m);
                f[k]              = src.get1(row, row * src.ld + n);
            }
#pragma unroll
            for (int k = 0; k < RO_ROWS; ++k)
                if (m + 4 * k * rows < m1)
                    q[(b * M + m + 4 * k * rows) * N + n] =
                        static_cast<uint8_t>(cvt_pk_fp8<E5M2>(scale_clamp(f[k], sc[0], qmax), 0.f, 0u, false));
        }
    }
}

// Codes transposed: a workgroup turns a 128 x 128 tile around. A thread holds four rows of eight
// columns at a time: the conversion packs the four rows of a column into one word (no byte shuffles),
// the words of a column meet in the LDS and leave as whole 128-byte rows of the transposed matrix.
// 3001 x 4096 codes quantized again along their other axis: de-quantize, maxima, cast and byte transpose
// (seven launches over 24.6 MB of bf16) took 118 us, the maxima launch and this one take 6.2 + 11.6 us;
// 3001 x 2880 bf16 gradients 112 -> 6.1 + 11.1 us.
template <typename SRC, bool E5M2, bool VEC8>
__global__ __launch_bounds__(256) void quant_outer_t_kernel(const SRC src, uint8_t *__restrict__ qt,
                                                            const float *__restrict__ part, const int chunks,
                                                            float *__restrict__ scale_inv, const int64_t M, const int64_t N,
                                                            const int64_t ldt, const float qmax) {
    constexpr int       P = 33; // words per LDS row
    __shared__ uint32_t t[128 * P];
    __shared__ float    s[128];
    const int           tid = threadIdx.x;
    // (tiles numbered along x, columns first: the y extent of a grid ends at 65535, 8.4 million rows)
    const uint32_t      nt = static_cast<uint32_t>((N + 127) / 128), tn = blockIdx.x % nt, tm = blockIdx.x / nt;
    const int64_t       b = blockIdx.z, n0 = static_cast<int64_t>(tn) * 128, m0 = static_cast<int64_t>(tm) * 128;
    const int           cc = tid & 15, rg = tid >> 4; // eight columns, four rows (two rounds of 64 rows)
    const int64_t       n = n0 + cc * 8;
    typename SRC::Raw   raw[VEC8 ? 8 : 1];
    if constexpr (VEC8) {
        // all eight loads are requested before the partial maxima are looked at
        const int64_t nn = n < N ? n : 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int64_t m = m0 + (k >> 2) * 64 + rg * 4 + (k & 3), row = b * M + (m < M ? m : 0);
            raw[k] = src.load8(row, row * src.ld + nn);
        }
    }
    if (tid < 128) {
        float sc = 0.f;
        if (n0 + tid < N) {
            sc = outer_scale(part, true, b, n0 + tid, N, chunks, qmax);
            if (tm == 0)
                scale_inv[b * N + n0 + tid] = 1.0f / sc;
        }
        s[tid] = sc;
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float f[4][8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int64_t m = m0 + h * 64 + rg * 4 + k;
            if constexpr (VEC8) {
                src.get8(raw[h * 4 + k], f[k]);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    f[k][e] = (m < M && n + e < N) ? src.get1(b * M + m, (b * M + m) * src.ld + n + e) : 0.f;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) // (rows behind the end: code 0)
                f[k][e] = m < M ? scale_clamp(f[k][e], s[cc * 8 + e], qmax) : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e)
            t[(cc * 8 + e) * P + h * 16 + rg] = cvt4_fp8<E5M2>(f[0][e], f[1][e], f[2][e], f[3][e]);
    }
    __syncthreads();
    const int j = tid & 7; // 16-byte chunk of a transposed row
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int     c  = (tid >> 3) + 32 * p;
        const int64_t mr = m0 + j * 16;
        if (n0 + c < N && mr < ldt) {
            u32x4 v;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                v[k] = t[c * P + j * 4 + k];
            st128(qt + (b * N + n0 + c) * ldt + mr, v);
        }
    }
}

__global__ void zero_u32_kernel(uint32_t *p, const int64_t n) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = 0u;
}

// column maxima (dynamic) or given scales -> scale_inv in place: for the form without a workspace, and for
// scales that are given in scale_inv's own storage
__global__ void finish_scale_inv_kernel(float *scale_inv, const bool dynamic, const int64_t n, const float qmax) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        scale_inv[i] = 1.0f / (dynamic ? qmax / fmaxf(scale_inv[i], 1e-12f) : scale_inv[i]);
}

// How a problem is split: 1 << lc lanes across a row (as many as its columns need, at most 64), strips of
// columns, row chunks for about OUTER_BLOCKS workgroups over all strips; a chunk is at least one round of
// requests of its workgroup. The second launch reads each chunk's maxima for every column, so there are
// at most OUTER_PARTS of them, unless a matrix is so tall and narrow that twice as many would pay (lanes
// that request two bytes need more workgroups than those that request sixteen) and each of OUTER_PARTS
// chunks had more than 12 (32) rounds: then the maxima meet by atomics behind a zero-fill, one launch more,
// and the cast is split as if there were none to read. bf16 from memory, in place / transposed, us:
//   512 columns    16384 rows (8 rounds): two launches 29 / 23, three 25 / 28; 32768 (16): two 54 / 37, three 31 / 34
//   33 columns, one per lane    32768 rows (16 rounds): two 27 / 25, three 26 / 32; 130, 70000 (34): 67 / 55, 36 / 45
//   64 columns, 1048576 rows: 64 lanes across a row and two launches 2410 / 834, eight lanes and three 89 / 97
constexpr int64_t OUTER_BLOCKS = 1024, OUTER_PARTS = 64;
struct OuterPlan {
    int     lc;
    int64_t strips;                 // workgroups along the columns
    int64_t chunks, rows;           // chunks of the maxima, rows of each
    int64_t cast_chunks, cast_rows; // the same of a cast behind one maximum (or given scale) per column
    bool    meet;
};
static OuterPlan outer_plan(int64_t B, int64_t M, int64_t N, int vec) {
    OuterPlan p{};
    while (p.lc < 6 && (int64_t{vec} << p.lc) < N)
        ++p.lc;
    p.strips            = cdiv(N, int64_t{vec} << p.lc);
    const int64_t round = 4 * RO_ROWS * (64 >> p.lc), most = cdiv(M, round), across = p.strips * B;
    auto          split = [&](int64_t want, int64_t &chunks, int64_t &rows) {
        const int64_t c = want < most ? want : most;
        rows            = cdiv(M, c < 1 ? 1 : c);
        chunks          = cdiv(M, rows);
    };
    const int64_t blocks = cdiv(OUTER_BLOCKS, across), tall = cdiv(vec == 1 ? 1024 : 256, across);
    p.meet               = tall >= 2 * OUTER_PARTS && cdiv(M, OUTER_PARTS) > (vec == 1 ? 32 : 12) * round;
    split(p.meet ? tall : (blocks < OUTER_PARTS ? blocks : OUTER_PARTS), p.chunks, p.rows);
    split(blocks, p.cast_chunks, p.cast_rows);
    return p;
}

template <typename SRC, bool E5M2>
static int launch_outer(const SRC &src, bool vec, int64_t B, int64_t M, int64_t N, [[maybe_unused]] uint8_t *q, uint8_t *qt,
                        int64_t ldt, [[maybe_unused]] const float *scale_in, float *scale_inv, float *ws, hipStream_t st) {
    const float     qmax    = E5M2 ? 57344.0f : 448.0f;
    const OuterPlan p       = outer_plan(B, M, N, vec ? 8 : 1);
    const bool      dynamic = scale_in == nullptr, meet = p.meet || ws == nullptr;
    float          *amax    = ws != nullptr ? ws : scale_inv; // (without a workspace the maxima meet in scale_inv's storage)
    const int       parts   = meet ? 1 : static_cast<int>(p.chunks);
    const dim3      g(static_cast<unsigned>(p.strips), static_cast<unsigned>(p.chunks), static_cast<unsigned>(B));
    const unsigned  gs = static_cast<unsigned>(cdiv(B * N, 256));
    if (dynamic) {
        if (meet) {
            zero_u32_kernel<<<gs, 256, 0, st>>>(reinterpret_cast<uint32_t *>(amax), B * N);
            if (vec)
                col_amax_kernel<SRC, 8, true><<<g, 256, 0, st>>>(src, amax, M, N, p.rows, p.lc);
            else
                col_amax_kernel<SRC, 1, true><<<g, 256, 0, st>>>(src, amax, M, N, p.rows, p.lc);
        } else if (vec) {
            col_amax_kernel<SRC, 8, false><<<g, 256, 0, st>>>(src, amax, M, N, p.rows, p.lc);
        } else {
            col_amax_kernel<SRC, 1, false><<<g, 256, 0, st>>>(src, amax, M, N, p.rows, p.lc);
        }
    }
    if (qt != nullptr) {
        const dim3 gt(static_cast<unsigned>(cdiv(N, 128) * cdiv(ldt, 128)), 1, static_cast<unsigned>(B));
        if (vec)
            quant_outer_t_kernel<SRC, E5M2, true><<<gt, 256, 0, st>>>(src, qt, amax, parts, scale_inv, M, N, ldt, qmax);
        else
            quant_outer_t_kernel<SRC, E5M2, false><<<gt, 256, 0, st>>>(src, qt, amax, parts, scale_inv, M, N, ldt, qmax);
        return check_launch("quant_outer_t_kernel");
    }
    if constexpr (SRC::IN_PLACE) {
        const float *from = dynamic ? amax : scale_in;
        float       *to   = from != scale_inv ? scale_inv : nullptr;
        const bool   one  = !dynamic || meet;
        const dim3   gc(g.x, static_cast<unsigned>(one ? p.cast_chunks : p.chunks), g.z);
        const int64_t rows = one ? p.cast_rows : p.rows;
        if (vec)
            quant_outer_kernel<SRC, E5M2, 8><<<gc, 256, 0, st>>>(src, q, from, dynamic, parts, to, M, N, rows, p.lc, qmax);
        else
            quant_outer_kernel<SRC, E5M2, 1><<<gc, 256, 0, st>>>(src, q, from, dynamic, parts, to, M, N, rows, p.lc, qmax);
        if (to == nullptr)
            finish_scale_inv_kernel<<<gs, 256, 0, st>>>(scale_inv, dynamic, B * N, qmax);
    }
    return check_launch("quant_outer_kernel");
}

template <typename T>
static int launch_outer_hp(const void *x, int64_t B, int64_t M, int64_t N, void *q, void *qt, int64_t ldt, bool e5m2,
                           const float *scale_in, float *scale_inv, float *ws, hipStream_t st) {
    const OuterSrcHP<T> src{static_cast<const T *>(x), N};
    const bool          vec = N % 8 == 0 && aligned_to(x, 16) && (q == nullptr || aligned_to(q, 8));
    auto *qp = static_cast<uint8_t *>(q), *tp = static_cast<uint8_t *>(qt);
    return e5m2 ? launch_outer<OuterSrcHP<T>, true>(src, vec, B, M, N, qp, tp, ldt, scale_in, scale_inv, ws, st)
                : launch_outer<OuterSrcHP<T>, false>(src, vec, B, M, N, qp, tp, ldt, scale_in, scale_inv, ws, st);
}

// codes quantized again keep their format
template <typename T>
static int launch_outer_codes(const void *x, int64_t ld, const float *row_scale, int64_t B, int64_t M, int64_t N, void *qt,
                              int64_t ldt, bool e5m2, float *scale_inv, float *ws, hipStream_t st) {
    const bool vec = N % 8 == 0 && ld % 8 == 0 && aligned_to(x, 8);
    auto      *xp  = static_cast<const uint8_t *>(x);
    auto      *tp  = static_cast<uint8_t *>(qt);
    if (e5m2)
        return launch_outer<OuterSrcCodes<T, true>, true>({xp, ld, row_scale}, vec, B, M, N, nullptr, tp, ldt, nullptr, scale_inv, ws, st);
    return launch_outer<OuterSrcCodes<T, false>, false>({xp, ld, row_scale}, vec, B, M, N, nullptr, tp, ldt, nullptr, scale_inv, ws, st);
}

// the form behind pt_quantize_fp8_rowwise (quant_fp8.hip); ws may be NULL
int launch_quant_rowwise_outer(const void *x, int x_dtype, int64_t B, int64_t M, int64_t N, void *q, bool e5m2,
                               const float *scale_in, float *scale_inv, float *ws, hipStream_t st) {
    if (x_dtype == PT_DTYPE_BF16)
        return launch_outer_hp<bf16_t>(x, B, M, N, q, nullptr, 0, e5m2, scale_in, scale_inv, ws, st);
    if (x_dtype == PT_DTYPE_F16)
        return launch_outer_hp<f16_t>(x, B, M, N, q, nullptr, 0, e5m2, scale_in, scale_inv, ws, st);
    return launch_outer_hp<float>(x, B, M, N, q, nullptr, 0, e5m2, scale_in, scale_inv, ws, st);
}

} // namespace pt

using namespace pt;

extern "C" {

size_t pt_quantize_fp8_rowwise_outer_workspace_bytes(int64_t B, int64_t M, int64_t N) {
    if (B <= 0 || M <= 0 || N <= 0)
        return 0;
    // (the wider lanes' plan may not be taken, so the workspace serves either)
    int64_t parts = 1;
    for (const int vec : {8, 1}) {
        const OuterPlan p = outer_plan(B, M, N, vec);
        if (!p.meet && p.chunks > parts)
            parts = p.chunks;
    }
    return static_cast<size_t>(B * parts * N) * sizeof(float);
}

int pt_quantize_fp8_rowwise_outer(const void *x, int x_dtype, const float *row_scale_inv, int hp_dtype, int64_t B, int64_t M,
                                  int64_t N, void *q, void *q_t, int64_t ld_t, int q_dtype, float *scale_inv, void *workspace,
                                  size_t workspace_bytes, void *stream) {
    return pt_quantize_fp8_rowwise_outer_ld(x, N, x_dtype, row_scale_inv, hp_dtype, B, M, N, q, q_t, ld_t, q_dtype, scale_inv,
                                            workspace, workspace_bytes, stream);
}

int pt_quantize_fp8_rowwise_outer_ld(const void *x, int64_t ld_x, int x_dtype, const float *row_scale_inv, int hp_dtype,
                                     int64_t B, int64_t M, int64_t N, void *q, void *q_t, int64_t ld_t, int q_dtype,
                                     float *scale_inv, void *workspace, size_t workspace_bytes, void *stream) {
    const bool codes = is_fp8_dtype(x_dtype);
    PT_REQUIRE(codes || is_hp_dtype(x_dtype), "input must be bf16, fp16, fp32 or fp8 codes");
    PT_REQUIRE(is_fp8_dtype(q_dtype), "output must be e4m3 or e5m2");
    PT_REQUIRE(B >= 0 && M >= 0 && N >= 0, "dimensions must be non-negative");
    PT_REQUIRE((q != nullptr) != (q_t != nullptr), "one of q and q_t is written");
    PT_REQUIRE(codes ? ld_x >= N : ld_x == N, "only rows of codes may be longer than the matrix is wide");
    if (codes) {
        PT_REQUIRE(row_scale_inv != nullptr && is_hp_dtype(hp_dtype), "codes need their row scales and the type they stand for");
        PT_REQUIRE(q_t != nullptr && q_dtype == x_dtype, "codes are quantized again into their own format, transposed");
    }
    if (B * M * N == 0)
        return PT_OK;
    PT_REQUIRE(x && scale_inv, "NULL tensor pointer");
    PT_REQUIRE(q_t == nullptr || (ld_t >= M && ld_t % 16 == 0 && aligned_to(q_t, 16)),
               "transposed rows must be 16-byte aligned and hold M codes");
    // (the rows that pt_quantize_fp8_rowwise takes; transposed, 2^32 threads along x)
    PT_REQUIRE(B < 65536 && cdiv(M, 256) < 65536 && (q_t == nullptr || cdiv(N, 128) * cdiv(ld_t, 128) < (1LL << 24)),
               "grid dimension out of range");
    if (workspace == nullptr || workspace_bytes < pt_quantize_fp8_rowwise_outer_workspace_bytes(B, M, N) || !aligned_to(workspace, 16))
        return fail(PT_ERR_WORKSPACE, "pt_quantize_fp8_rowwise_outer: workspace missing, too small or misaligned");
    auto       st = static_cast<hipStream_t>(stream);
    auto      *ws = static_cast<float *>(workspace);
    const bool e5 = q_dtype == PT_DTYPE_E5M2;
    const int  hp = codes ? hp_dtype : x_dtype;
    if (codes) {
        if (hp == PT_DTYPE_BF16)
            return launch_outer_codes<bf16_t>(x, ld_x, row_scale_inv, B, M, N, q_t, ld_t, e5, scale_inv, ws, st);
        if (hp == PT_DTYPE_F16)
            return launch_outer_codes<f16_t>(x, ld_x, row_scale_inv, B, M, N, q_t, ld_t, e5, scale_inv, ws, st);
        return launch_outer_codes<float>(x, ld_x, row_scale_inv, B, M, N, q_t, ld_t, e5, scale_inv, ws, st);
    }
    if (hp == PT_DTYPE_BF16)
        return launch_outer_hp<bf16_t>(x, B, M, N, q, q_t, ld_t, e5, nullptr, scale_inv, ws, st);
    if (hp == PT_DTYPE_F16)
        return launch_outer_hp<f16_t>(x, B, M, N, q, q_t, ld_t, e5, nullptr, scale_inv, ws, st);
    return launch_outer_hp<float>(x, B, M, N, q, q_t, ld_t, e5, nullptr, scale_inv, ws, st);
}

} // extern "C"
