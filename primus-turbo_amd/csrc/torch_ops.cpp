// The host side of the dense operators in C++: checks, output and workspace allocation, and the call of the C entry
// point. Bound by host time: a 16-token serving product spends 13 us in kernels, and its two operators took 24 us to
// issue from Python, a training step makes six to eight such calls. Host us a call, body in Python / here: product 14.2 / 6.8 (the
// launch is 3.9 of them), tensorwise cast 9.7 / 6.2, with the transposed codes 13.7 / 7.6, rowwise cast along the columns 17.1 / 10.4.
// The serving call 33.7 -> 21.3, a ROWWISE training step of 3001 x 2880 x 4096 298 -> 200, where kernels bound it.
//
// Each operator is registered from Python (schema, tracing, autograd) with a Python body; here its CUDA kernel is
// registered. It handles the forms that the layers make, and hands every other one (other layouts, unusual dtypes,
// a current device that is not the tensors', errors) to the operator "<name>_general", which is the Python
// body. So what an operator accepts, refuses and says is decided in one place.
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <hip/hip_runtime_api.h>
#include <torch/library.h>

#include <atomic>
#include <dlfcn.h>

#include "../../include/primus_turbo_amd.h"

namespace {

using at::ScalarType;
using at::Tensor;

// Entry points of the library that Python loaded (by path: there is one of them in the process).
struct Api {
#define PT_FN(name) decltype(&::name) name
    PT_FN(pt_last_error);
    PT_FN(pt_gemm_fp8);
    PT_FN(pt_gemm_fp8_workspace_bytes);
    PT_FN(pt_gemm_fp8_vec_in_place);
    PT_FN(pt_gemm_fp8_nn_in_place);
    PT_FN(pt_gemm_mx);
    PT_FN(pt_gemm_mx_workspace_bytes);
    PT_FN(pt_quantize_fp8_tensorwise_static);
    PT_FN(pt_quantize_fp8_tensorwise_t);
    PT_FN(pt_dequantize_fp8_tensorwise);
    PT_FN(pt_quantize_fp8_rowwise);
    PT_FN(pt_quantize_fp8_rowwise_padded);
    PT_FN(pt_quantize_fp8_rowwise_outer_ld);
    PT_FN(pt_quantize_fp8_rowwise_outer_workspace_bytes);
    PT_FN(pt_quantize_fp8_blockwise_kmajor);
    PT_FN(pt_quantize_mx);
#undef PT_FN
};
Api               api;
std::atomic<bool> bound{false};
// the launch structure of the tensorwise quantizer: 0 automatic, 1 fused, 2 two passes
std::atomic<int64_t> tensorwise_mode{0};

void bind_native(std::string path) {
    void *lib = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    TORCH_CHECK(lib != nullptr, "primus_turbo: cannot load ", path, ": ", dlerror());
    Api a;
#define PT_FN(name)                                                                                                       \
    a.name = reinterpret_cast<decltype(a.name)>(dlsym(lib, #name));                                                       \
    TORCH_CHECK(a.name != nullptr, "primus_turbo: ", path, " does not export " #name)
    PT_FN(pt_last_error);
    PT_FN(pt_gemm_fp8);
    PT_FN(pt_gemm_fp8_workspace_bytes);
    PT_FN(pt_gemm_fp8_vec_in_place);
    PT_FN(pt_gemm_fp8_nn_in_place);
    PT_FN(pt_gemm_mx);
    PT_FN(pt_gemm_mx_workspace_bytes);
    PT_FN(pt_quantize_fp8_tensorwise_static);
    PT_FN(pt_quantize_fp8_tensorwise_t);
    PT_FN(pt_dequantize_fp8_tensorwise);
    PT_FN(pt_quantize_fp8_rowwise);
    PT_FN(pt_quantize_fp8_rowwise_padded);
    PT_FN(pt_quantize_fp8_rowwise_outer_ld);
    PT_FN(pt_quantize_fp8_rowwise_outer_workspace_bytes);
    PT_FN(pt_quantize_fp8_blockwise_kmajor);
    PT_FN(pt_quantize_mx);
#undef PT_FN
    api = a;
    bound.store(true, std::memory_order_release);
}

void set_tensorwise_mode(int64_t mode) {
    tensorwise_mode.store(mode, std::memory_order_relaxed);
}

// Whether a call of the C library was carried out. What it refuses (arguments, a form, a workspace), it refuses before it
// launches the kernel that writes the results: the Python body then refuses as well, or finds another way. Any other status
// raises here: a failed launch is found by the error that HIP holds after it, which may be one that an earlier call of
// this thread left while this kernel runs, and an accumulating product that is issued again adds twice.
bool carried_out(int status) {
    if (status == PT_OK)
        return true;
    TORCH_CHECK(status == PT_ERR_INVALID_ARGUMENT || status == PT_ERR_UNSUPPORTED || status == PT_ERR_WORKSPACE,
                "primus_turbo native error ", status, ": ", api.pt_last_error());
    return false;
}

bool is_fp8(ScalarType t) {
    return t == at::kFloat8_e4m3fn || t == at::kFloat8_e5m2;
}
bool is_hp(ScalarType t) {
    return t == at::kBFloat16 || t == at::kHalf || t == at::kFloat;
}
int code_of(ScalarType t) {
    switch (t) {
    case at::kBFloat16: return PT_DTYPE_BF16;
    case at::kHalf: return PT_DTYPE_F16;
    case at::kFloat: return PT_DTYPE_F32;
    case at::kFloat8_e4m3fn: return PT_DTYPE_E4M3;
    case at::kFloat8_e5m2: return PT_DTYPE_E5M2;
    default: return PT_DTYPE_E2M1X2; // (callers admit no other type)
    }
}
int64_t cdiv(int64_t a, int64_t b) {
    return (a + b - 1) / b;
}
int64_t round_up(int64_t a, int64_t b) {
    return cdiv(a, b) * b;
}

// Plain dense memory on the current device: what the forms below are written for.
bool on_current_device(const Tensor &t) {
    int dev = -1;
    return bound.load(std::memory_order_acquire) && t.is_cuda() && hipGetDevice(&dev) == hipSuccess && t.get_device() == dev;
}
bool plain(const Tensor &t, const Tensor &like) {
    return t.is_cuda() && t.is_contiguous() && t.get_device() == like.get_device();
}
hipStream_t stream_of(const Tensor &t) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.get_device()).stream();
}
bool capturing(hipStream_t s) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &status) != hipSuccess || status != hipStreamCaptureStatusNone;
}
Tensor empty(at::IntArrayRef shape, ScalarType t, const Tensor &like) {
    return at::empty(shape, at::TensorOptions().dtype(t).device(like.device()));
}

// The Python body of an operator. (The callers' stack holds the operator's arguments in order.)
template <typename... Args> torch::jit::Stack general(const char *name, Args &&...args) {
    auto              op = c10::Dispatcher::singleton().findSchemaOrThrow(name, "");
    torch::jit::Stack stack;
    torch::jit::push(stack, std::forward<Args>(args)...);
    op.callBoxed(stack);
    return stack;
}

// ---- products -------------------------------------------------------------------------------------------------------
enum : int64_t { TENSORWISE = 1, ROWWISE = 2, BLOCKWISE = 3, MX_BLOCKWISE = 4 }; // ScalingGranularity

// Bytes from one row's scales to the next row's, 0 for word-major ones; -1: not the scales of `rows` rows of K values.
int64_t mx_scale_pitch(const Tensor &s, int64_t rows, int64_t K) {
    if (s.dim() != 2 || !s.is_contiguous())
        return -1;
    if (s.scalar_type() == at::kInt)
        return K % 128 == 0 && s.size(0) == K / 128 && s.size(1) == rows ? 0 : -1;
    return s.element_size() == 1 && s.size(0) == rows && s.size(1) >= K / 32 && s.size(1) > 0 ? s.size(1) : -1;
}

// A product into `out` (MX: NT); false: a form for the Python body.
bool launch_mx(const Tensor &a, const Tensor &a_s, const Tensor &b, const Tensor &b_s, Tensor &out, bool accumulate) {
    const bool fp4 = a.scalar_type() == at::kFloat4_e2m1fn_x2;
    if (fp4 ? b.scalar_type() != at::kFloat4_e2m1fn_x2 : !is_fp8(a.scalar_type()) || !is_fp8(b.scalar_type()))
        return false;
    const int64_t pack = fp4 ? 2 : 1, M = a.size(0), N = b.size(0), ld = a.size(1), K = ld * pack;
    if (b.size(1) != ld || K % 32 != 0)
        return false;
    const int64_t sa_ld = mx_scale_pitch(a_s, M, K), sb_ld = mx_scale_pitch(b_s, N, K);
    if (sa_ld < 0 || sb_ld < 0)
        return false;
    // (word-major scales of both operands and rows of whole slabs: nothing is copied)
    const bool   ready    = sa_ld == 0 && sb_ld == 0 && ld % 128 == 0 && ld >= 512;
    const size_t ws_bytes = ready ? 0 : api.pt_gemm_mx_workspace_bytes(M, N, K, ld, ld, fp4);
    Tensor       ws;
    if (ws_bytes)
        ws = empty({static_cast<int64_t>(ws_bytes)}, at::kByte, a);
    return carried_out(api.pt_gemm_mx(a.data_ptr(), a_s.data_ptr(), b.data_ptr(), b_s.data_ptr(), code_of(a.scalar_type()),
                                      a.scalar_type() == at::kFloat8_e5m2, b.scalar_type() == at::kFloat8_e5m2, out.data_ptr(),
                                      code_of(out.scalar_type()), M, N, K, ld, ld, sa_ld, sb_ld, accumulate, ws_bytes ? ws.data_ptr() : nullptr,
                                      ws_bytes, 0, stream_of(a)));
}

bool launch_scaled(const Tensor &a, const Tensor &a_s, bool trans_a, const Tensor &b, const Tensor &b_s, bool trans_b, Tensor &out,
                   bool trans_c, int64_t granularity, bool accumulate) {
    if (!is_fp8(a.scalar_type()) || !is_fp8(b.scalar_type()) || a_s.scalar_type() != at::kFloat || b_s.scalar_type() != at::kFloat)
        return false;
    int64_t M = a.size(trans_a), N = b.size(!trans_b);
    const int64_t K = a.size(!trans_a), kb = cdiv(K, 128);
    if (b.size(trans_b) != K)
        return false;
    int     mode = 0, sa_blk = 1, sb_blk = 1;
    int64_t sa_m = 0, sa_k = 0, sb_n = 0, sb_k = 0;
    if (granularity == TENSORWISE) {
        if (a_s.numel() != 1 || b_s.numel() != 1)
            return false;
    } else if (granularity == ROWWISE) {
        if (a_s.numel() != M || b_s.numel() != N || !a_s.is_contiguous() || !b_s.is_contiguous())
            return false;
        sa_m = sb_n = 1;
    } else if (granularity == BLOCKWISE) {
        if (trans_a || a_s.dim() != 2 || b_s.dim() != 2 || !b_s.is_contiguous())
            return false;
        mode = 1;
        // row blocks: the view of a block-major tensor that the activation's quantizer made
        const int64_t nb        = cdiv(N, 128);
        const bool    row_major = a_s.size(0) == M && a_s.size(1) == kb;
        const bool    rows      = row_major && kb > 1 && a_s.stride(0) == 1 && a_s.stride(1) == M;
        if (trans_b && row_major && b_s.size(0) == nb && b_s.size(1) == kb) {
            if (!rows)
                return false;
            sa_m = 1, sa_k = M, sb_n = kb, sb_k = 1, sb_blk = 128;
        } else if (!trans_b && rows && b_s.size(0) == kb && b_s.size(1) == nb) {
            // the input gradient: the weight's codes and tiles as the forward product reads them
            sa_m = 1, sa_k = M, sb_n = 1, sb_k = nb, sb_blk = 128;
        } else if (trans_b && a_s.is_contiguous() && a_s.size(0) == kb && a_s.size(1) == M && b_s.size(0) == kb && b_s.size(1) == N) {
            // both operands transposed 128 x 1 column quantizations: a scale per row of either
            sa_m = 1, sa_k = M, sb_n = 1, sb_k = N;
        } else {
            return false;
        }
    } else {
        return false;
    }
    const Tensor *pa = &a, *pb = &b, *psa = &a_s, *psb = &b_s;
    if (trans_c) { // C^T = B . A^T
        std::swap(pa, pb);
        std::swap(psa, psb);
        std::swap(M, N);
        std::swap(sa_m, sb_n);
        std::swap(sa_k, sb_k);
        std::swap(sa_blk, sb_blk);
        const bool was_a = trans_a;
        trans_a          = !trans_b;
        trans_b          = !was_a;
    }
    const bool   in_place = mode == 0 && !trans_b && api.pt_gemm_fp8_vec_in_place(M, N, K, trans_a);
    const bool   b_as_is  = trans_b || (mode == 1 && !trans_a && sa_blk == 1 && sb_blk == 128 && api.pt_gemm_fp8_nn_in_place(M, N, K));
    const size_t ws_bytes = in_place ? 0 : api.pt_gemm_fp8_workspace_bytes(M, N, K, trans_a, b_as_is);
    Tensor       ws;
    if (ws_bytes)
        ws = empty({static_cast<int64_t>(ws_bytes)}, at::kByte, a);
    return carried_out(api.pt_gemm_fp8(pa->data_ptr(), code_of(pa->scalar_type()), static_cast<const float *>(psa->data_ptr()), pb->data_ptr(),
                                       code_of(pb->scalar_type()), static_cast<const float *>(psb->data_ptr()), out.data_ptr(),
                                       code_of(out.scalar_type()), M, N, K, trans_a, trans_b, mode, sa_m, sa_k, sb_n, sb_k, sa_blk, sb_blk, accumulate,
                                       ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, 0, stream_of(a)));
}

bool launch_product(const Tensor &a, const Tensor &a_s, bool trans_a, const Tensor &b, const Tensor &b_s, bool trans_b, Tensor &out,
                    bool trans_c, int64_t granularity, bool accumulate) {
    if (granularity == MX_BLOCKWISE)
        return !trans_a && trans_b && trans_c ? launch_mx(b, b_s, a, a_s, out, accumulate)
               : !trans_a && trans_b          ? launch_mx(a, a_s, b, b_s, out, accumulate)
                                              : false;
    return launch_scaled(a, a_s, trans_a, b, b_s, trans_b, out, trans_c, granularity, accumulate);
}

bool product_form(const Tensor &a, const Tensor &a_s, const Tensor &b, const Tensor &b_s) {
    return on_current_device(a) && a.dim() == 2 && b.dim() == 2 && plain(a, a) && plain(b, a) &&
           a_s.is_cuda() && b_s.is_cuda() && a_s.get_device() == a.get_device() && b_s.get_device() == a.get_device();
}

Tensor gemm_fp8(const Tensor &a, const Tensor &a_s, bool trans_a, const Tensor &b, const Tensor &b_s, bool trans_b,
                ScalarType out_dtype, bool trans_c, int64_t granularity, int64_t backend) {
    if (product_form(a, a_s, b, b_s) && is_hp(out_dtype)) {
        const int64_t M = a.size(trans_a), N = b.size(!trans_b);
        Tensor        out = trans_c ? empty({N, M}, out_dtype, a) : empty({M, N}, out_dtype, a);
        if ((granularity != MX_BLOCKWISE || (plain(a_s, a) && plain(b_s, a))) &&
            launch_product(a, a_s, trans_a, b, b_s, trans_b, out, trans_c, granularity, false))
            return out;
    }
    return general("primus_turbo::gemm_fp8_impl_general", a, a_s, trans_a, b, b_s, trans_b, out_dtype, trans_c, granularity,
                   backend)[0].toTensor();
}

// out += the product; false: nothing was done
bool gemm_fp8_into(const Tensor &a, const Tensor &a_s, bool trans_a, const Tensor &b, const Tensor &b_s, bool trans_b,
                   bool trans_c, int64_t granularity, Tensor out) {
    if (!product_form(a, a_s, b, b_s) || !is_hp(out.scalar_type()) || out.dim() != 2 || !plain(out, a) ||
        out.size(trans_c) != a.size(trans_a) || out.size(!trans_c) != b.size(!trans_b))
        return false;
    if (granularity == MX_BLOCKWISE && (!plain(a_s, a) || !plain(b_s, a)))
        return false;
    return launch_product(a, a_s, trans_a, b, b_s, trans_b, out, trans_c, granularity, true);
}

// ---- quantizers -----------------------------------------------------------------------------------------------------
bool castable(const Tensor &x, ScalarType dtype) {
    return on_current_device(x) && is_hp(x.scalar_type()) && is_fp8(dtype) && x.is_contiguous();
}

std::vector<Tensor> quantize_fp8_tensorwise(const Tensor &x, ScalarType dtype, const std::optional<Tensor> &scale) {
    if (!scale.has_value() && castable(x, dtype) && tensorwise_mode.load(std::memory_order_relaxed) != 2) {
        const hipStream_t st = stream_of(x);
        if (!capturing(st)) {
            Tensor q = at::empty_like(x, x.options().dtype(dtype)), scale_inv = empty({}, at::kFloat, x);
            if (carried_out(api.pt_quantize_fp8_tensorwise_static(x.data_ptr(), code_of(x.scalar_type()), x.numel(), q.data_ptr(), code_of(dtype),
                                                                  nullptr, static_cast<float *>(scale_inv.data_ptr()), nullptr, st)))
                return {q, scale_inv};
        }
    }
    return general("primus_turbo_cpp_extension::quantize_fp8_tensorwise_general", x, dtype, scale)[0].toTensorVector();
}

std::tuple<Tensor, Tensor, Tensor> quantize_fp8_tensorwise_t(const Tensor &x, ScalarType dtype, int64_t width, int64_t width_t) {
    if (castable(x, dtype) && x.dim() == 2 && tensorwise_mode.load(std::memory_order_relaxed) != 2) {
        const int64_t     R = x.size(0), C = x.size(1);
        const hipStream_t st = stream_of(x);
        if (C % 16 == 0 && width % 16 == 0 && width_t % 16 == 0 && (width == C || width == round_up(C, 128)) &&
            (width_t == R || width_t == round_up(R, 128)) && x.numel() > 0 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
            !capturing(st)) {
            Tensor q = empty({R, width}, dtype, x), q_t = empty({C, width_t}, dtype, x), scale_inv = empty({}, at::kFloat, x);
            if (carried_out(api.pt_quantize_fp8_tensorwise_t(x.data_ptr(), code_of(x.scalar_type()), R, C, q.data_ptr(), width, q_t.data_ptr(),
                                                             width_t, code_of(dtype), static_cast<float *>(scale_inv.data_ptr()), nullptr, 0,
                                                             st)))
                return {q, q_t, scale_inv};
        }
    }
    auto s = general("primus_turbo::quantize_fp8_tensorwise_t_general", x, dtype, width, width_t);
    return {s[0].toTensor(), s[1].toTensor(), s[2].toTensor()};
}

Tensor dequantize_fp8_tensorwise(const Tensor &x, const Tensor &scale_inv, ScalarType dtype) {
    if (on_current_device(x) && is_fp8(x.scalar_type()) && x.is_contiguous() && is_hp(dtype) && scale_inv.is_cuda() &&
        scale_inv.get_device() == x.get_device() && scale_inv.numel() == 1 && scale_inv.scalar_type() == at::kFloat) {
        Tensor out = at::empty_like(x, x.options().dtype(dtype));
        if (carried_out(api.pt_dequantize_fp8_tensorwise(x.data_ptr(), code_of(x.scalar_type()), x.numel(),
                                                         static_cast<const float *>(scale_inv.data_ptr()), out.data_ptr(), code_of(dtype),
                                                         stream_of(x))))
            return out;
    }
    return general("primus_turbo_cpp_extension::dequantize_fp8_tensorwise_general", x, scale_inv, dtype)[0].toTensor();
}

// Along the last axis; other axes and given scales are the Python body's.
std::vector<Tensor> quantize_fp8_rowwise(const Tensor &x, ScalarType dtype, int64_t axis, const std::optional<Tensor> &scale) {
    if (!scale.has_value() && castable(x, dtype) && x.dim() >= 1 && (axis == -1 || axis == x.dim() - 1)) {
        const int64_t M = x.size(-1);
        int64_t       B = 1;
        for (int64_t d = 0; d + 1 < x.dim(); ++d)
            B *= x.size(d);
        auto shape   = x.sizes().vec();
        shape.back() = 1;
        Tensor q = at::empty_like(x, x.options().dtype(dtype)), scale_inv = empty(shape, at::kFloat, x);
        if (carried_out(api.pt_quantize_fp8_rowwise(x.data_ptr(), code_of(x.scalar_type()), B, M, 1, q.data_ptr(), code_of(dtype), nullptr,
                                                    static_cast<float *>(scale_inv.data_ptr()), stream_of(x))))
            return {q, scale_inv};
    }
    return general("primus_turbo_cpp_extension::quantize_fp8_rowwise_general", x, dtype, axis, scale)[0].toTensorVector();
}

std::tuple<Tensor, Tensor> quant_fp8_rowwise_padded(const Tensor &x, ScalarType dtype, int64_t width) {
    if (castable(x, dtype) && x.dim() == 2 && width >= x.size(1)) {
        Tensor q = empty({x.size(0), width}, dtype, x), scale_inv = empty({x.size(0), 1}, at::kFloat, x);
        if (carried_out(api.pt_quantize_fp8_rowwise_padded(x.data_ptr(), code_of(x.scalar_type()), x.size(0), x.size(1), q.data_ptr(), width,
                                                           code_of(dtype), static_cast<float *>(scale_inv.data_ptr()), stream_of(x))))
            return {q, scale_inv};
    }
    auto s = general("primus_turbo::quant_fp8_rowwise_padded_impl_general", x, dtype, width);
    return {s[0].toTensor(), s[1].toTensor()};
}

std::tuple<Tensor, Tensor> quant_fp8_rowwise_t(const Tensor &x, const std::optional<Tensor> &row_scale, ScalarType hp, ScalarType dtype,
                                               int64_t pad, std::optional<int64_t> cols) {
    const bool codes = row_scale.has_value();
    if (on_current_device(x) && x.dim() == 2 && x.is_contiguous() && is_fp8(dtype) && is_hp(hp) && pad > 0 && pad % 16 == 0 &&
        x.scalar_type() == (codes ? dtype : hp) && (codes || !cols.has_value()) &&
        (!cols.has_value() || (*cols >= 0 && *cols <= x.size(1))) &&
        (!codes || (plain(*row_scale, x) && row_scale->scalar_type() == at::kFloat && row_scale->dim() == 2 &&
                    row_scale->size(0) == x.size(0) && row_scale->size(1) == 1))) {
        const int64_t M = x.size(0), N = cols.value_or(x.size(1)), Mp = round_up(M, pad);
        Tensor        q_t = empty({N, Mp}, dtype, x), scale_inv = empty({1, N}, at::kFloat, x);
        Tensor        ws  = empty({static_cast<int64_t>(api.pt_quantize_fp8_rowwise_outer_workspace_bytes(1, M, N))}, at::kByte, x);
        if (carried_out(api.pt_quantize_fp8_rowwise_outer_ld(
                x.data_ptr(), codes ? x.size(1) : N, code_of(x.scalar_type()),
                codes ? static_cast<const float *>(row_scale->data_ptr()) : nullptr, code_of(hp), 1, M, N, nullptr, q_t.data_ptr(),
                Mp, code_of(dtype), static_cast<float *>(scale_inv.data_ptr()), ws.data_ptr(), ws.numel(), stream_of(x))))
            return {q_t, scale_inv};
    }
    auto s = general("primus_turbo::quant_fp8_rowwise_t_impl_general", x, row_scale, hp, dtype, pad, cols);
    return {s[0].toTensor(), s[1].toTensor()};
}

std::tuple<Tensor, Tensor, Tensor, Tensor> quant_fp8_blockwise_kmajor(const Tensor &x, ScalarType dtype, int64_t block,
                                                                      bool with_col_t) {
    if (castable(x, dtype) && x.dim() == 2 && block == 128) {
        const int64_t M = x.size(0), N = x.size(1), Mp = round_up(M, block);
        Tensor        q = empty({M, N}, dtype, x), s = empty({cdiv(N, block), M}, at::kFloat, x);
        Tensor        q_t = with_col_t ? empty({N, Mp}, dtype, x) : empty({0}, dtype, x);
        Tensor        s_t = with_col_t ? empty({cdiv(M, block), N}, at::kFloat, x) : empty({0}, at::kFloat, x);
        if (carried_out(api.pt_quantize_fp8_blockwise_kmajor(x.data_ptr(), code_of(x.scalar_type()), M, N, code_of(dtype), q.data_ptr(),
                                                             static_cast<float *>(s.data_ptr()), with_col_t ? q_t.data_ptr() : nullptr,
                                                             with_col_t ? Mp : 0, with_col_t ? static_cast<float *>(s_t.data_ptr()) : nullptr,
                                                             stream_of(x))))
            return {q, s, q_t, s_t};
    }
    auto r = general("primus_turbo::quant_fp8_blockwise_kmajor_impl_general", x, dtype, block, with_col_t);
    return {r[0].toTensor(), r[1].toTensor(), r[2].toTensor(), r[3].toTensor()};
}

// The codes and scales of one direction, `rows` rows of `width` values each (both a multiple of what the kernel pads
// to): E8M0 bytes [rows, width / 32] or, word-major (8), words [width / 128, rows]. Empty tensors for one not wanted.
std::pair<Tensor, Tensor> mx_direction(const Tensor &x, ScalarType dtype, bool wanted, int64_t flags, int64_t rows, int64_t width) {
    if (!wanted)
        return {empty({0}, dtype, x), empty({0}, at::kFloat8_e8m0fnu, x)};
    const int64_t        pack = dtype == at::kFloat4_e2m1fn_x2 ? 2 : 1;
    std::vector<int64_t> q(x.sizes().begin(), x.sizes().end() - 2), s = q;
    q.insert(q.end(), {rows, width / pack});
    if (flags & 8) {
        s.insert(s.end(), {width / 128, rows});
        return {empty(q, dtype, x), empty(s, at::kInt, x)};
    }
    s.insert(s.end(), {rows, width / 32});
    return {empty(q, dtype, x), empty(s, at::kFloat8_e8m0fnu, x)};
}

// Stochastic rounding (4) takes its seed in the Python body.
std::tuple<Tensor, Tensor, Tensor, Tensor> quantize_mx(const Tensor &x, ScalarType dtype, bool row, bool col, int64_t row_flags,
                                                       int64_t col_flags) {
    if ((row || col) && (row_flags & 4) == 0 && (col_flags & 4) == 0 && on_current_device(x) && x.is_contiguous() &&
        (x.dim() == 2 || x.dim() == 3) && (x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kHalf) &&
        (dtype == at::kFloat4_e2m1fn_x2 || is_fp8(dtype)) && x.size(-1) % 32 == 0) {
        const int64_t B = x.dim() == 3 ? x.size(0) : 1, M = x.size(-2), N = x.size(-1);
        auto [rq, rs] = mx_direction(x, dtype, row, row_flags, M, round_up(N, 128));
        auto [cq, cs] = mx_direction(x, dtype, col, col_flags, N, round_up(M, 128));
        if (carried_out(api.pt_quantize_mx(x.data_ptr(), code_of(x.scalar_type()), B, M, N, code_of(dtype), row ? rq.data_ptr() : nullptr,
                                           row ? static_cast<uint8_t *>(rs.data_ptr()) : nullptr, static_cast<int>(row_flags),
                                           col ? cq.data_ptr() : nullptr, col ? static_cast<uint8_t *>(cs.data_ptr()) : nullptr,
                                           static_cast<int>(col_flags), 0, stream_of(x))))
            return {rq, rs, cq, cs};
    }
    auto r = general("primus_turbo::quantize_mx_general", x, dtype, row, col, row_flags, col_flags);
    return {r[0].toTensor(), r[1].toTensor(), r[2].toTensor(), r[3].toTensor()};
}

} // namespace

TORCH_LIBRARY_FRAGMENT(primus_turbo, m) {
    m.def("_bind_native(str path) -> ()", &bind_native);
    m.def("_native_tensorwise_mode(int mode) -> ()", &set_tensorwise_mode);
    m.def("_gemm_fp8_into(Tensor a, Tensor a_scale_inv, bool trans_a, Tensor b, Tensor b_scale_inv, bool trans_b, bool trans_c, "
          "int granularity, Tensor(a!) out) -> bool");
}

TORCH_LIBRARY_IMPL(primus_turbo, CUDA, m) {
    m.impl("_gemm_fp8_into", &gemm_fp8_into);
    m.impl("gemm_fp8_impl", &gemm_fp8);
    m.impl("quantize_fp8_tensorwise_t", &quantize_fp8_tensorwise_t);
    m.impl("quant_fp8_rowwise_padded_impl", &quant_fp8_rowwise_padded);
    m.impl("quant_fp8_rowwise_t_impl", &quant_fp8_rowwise_t);
    m.impl("quant_fp8_blockwise_kmajor_impl", &quant_fp8_blockwise_kmajor);
    m.impl("quantize_mx", &quantize_mx);
}

TORCH_LIBRARY_IMPL(primus_turbo_cpp_extension, CUDA, m) {
    m.impl("quantize_fp8_tensorwise", &quantize_fp8_tensorwise);
    m.impl("dequantize_fp8_tensorwise", &dequantize_fp8_tensorwise);
    m.impl("quantize_fp8_rowwise", &quantize_fp8_rowwise);
}
