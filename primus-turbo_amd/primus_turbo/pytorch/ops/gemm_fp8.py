"""``gemm_fp8``: FP8 GEMM with autograd (reference: primus_turbo/pytorch/ops/gemm_fp8.py).

Which quantizer feeds which GEMM layout, per granularity (same recipes as the reference):

  TENSORWISE  fwd  C = Aq . Bq            one scale per tensor; both backward products read the forward
                   codes along their other axis in place where the kernels can, else they are
                   NT products on physically transposed fp8 copies (ref :96-276)
  ROWWISE     fwd  A, B quantized along K; backward re-quantizes the de-quantized
                   operands along the other axis and quantizes grad_out twice (ref :278-426)
  BLOCKWISE   fwd  A 1x128 (+128x1 for wgrad from the same read), B 128x128 tiles;
                   dgrad = NN with the same weight tiles, wgrad = TN on the 128x1 casts
                   (ref :429-553)
  MX_BLOCKWISE     A 1x32, B 32x32 two-direction MXFP8 casts, every GEMM is NT (ref :556-717)

HYBRID format: forward operands E4M3, gradients E5M2.
"""

from __future__ import annotations

from typing import Optional, Union

import torch

from primus_turbo.pytorch.core.backend import BackendType
from primus_turbo.pytorch.core.low_precision import (
    Float8QuantConfig,
    ScalingGranularity,
    ScalingRecipe,
    check_mxfp8_support,
)
from primus_turbo.pytorch.core.quantized_tensor import (
    QuantizedTensor,
    QuantizedTensorPair,
    check_quantized_tensor,
    transpose_last_two,
)
from primus_turbo.pytorch.kernels.gemm.gemm_fp8_impl import (
    gemm_fp8_accum_impl,
    gemm_fp8_impl,
    get_gemm_logical_shape,
    kn_layer_pays,
    reads_kn_in_place,
    vec_reads_in_place,
)
from primus_turbo.pytorch.kernels.quantization.quantization_impl import (
    quant_fp8_blockwise_dual_t_impl,
    quant_fp8_blockwise_kmajor_impl,
    quant_fp8_blockwise_for_weight_dual_impl,
    quant_fp8_rowwise_padded_impl,
    quant_fp8_rowwise_t_impl,
    quantize_fp8_tensorwise_t_impl,
    quantize_mx_operands,
)
from primus_turbo.pytorch.ops.quantization import dequantize_fp8, quantize_fp8, quantize_fp8_with_trans
from primus_turbo.pytorch.ops.utils import _get_dummy_wgrad, _get_fp8_dtype, _setup_fused_grad_accum, _traced

__all__ = ["gemm_fp8"]

_NATIVE = BackendType.TURBO.value  # single backend; the value is informational


def _gemm(a, a_s, trans_a, b, b_s, trans_b, out_dtype, trans_c, granularity):
    return gemm_fp8_impl(a, a_s, trans_a, b, b_s, trans_b, out_dtype, trans_c, granularity.value, _NATIVE)


def _wgrad_gemm(a, a_s, trans_a, b, b_s, trans_b, out_dtype, trans_c, granularity, accumulate_into=None):
    """Weight-gradient GEMM; with ``accumulate_into`` the result is added to that buffer in
    the GEMM epilogue and a cached dummy tensor of the weight's shape is returned (the
    framework's own accumulation was switched off in forward)."""
    if accumulate_into is None:
        return _gemm(a, a_s, trans_a, b, b_s, trans_b, out_dtype, trans_c, granularity)
    gemm_fp8_accum_impl(a, a_s, trans_a, b, b_s, trans_b, accumulate_into.dtype, trans_c, granularity.value,
                        accumulate_into, _NATIVE)
    return _get_dummy_wgrad(accumulate_into.shape, out_dtype)


def _quantized_parts(x, config, fwd: bool, axis):
    """-> ``(codes, scale_inv, original dtype)`` of an operand: the fields of a ``QuantizedTensor``
    that the caller quantized already, else a fresh quantization along ``axis``. Plain tensors, not
    wrappers, so that ``torch.compile`` traces the functions below into one graph."""
    if isinstance(x, QuantizedTensor):
        check_quantized_tensor(x, config, axis=axis)
        return x.qdata, x.scale_inv, x.dtype
    q, s = quantize_fp8(x.contiguous(), _get_fp8_dtype(config.format, fwd), config.granularity, axis=axis % x.ndim,
                        block_size=config.block_size)
    return q, s, x.dtype


def _whole_slabs(n: int) -> int:
    """``n`` codes padded to what the products read as they are: whole 128-byte slabs of a row."""
    return -(-n // 128) * 128


class FP8GemmTensorFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, a, b, a_t, b_t, trans_a, trans_b, out_dtype, config, fuse_bgrad_accum_pattern=None):
        fuse, main_grad = _setup_fused_grad_accum(b, fuse_bgrad_accum_pattern)
        # NT forward: keep physically transposed fp8 copies so that both backward GEMMs
        # are NT as well (contiguous-K operands need no transposition pass inside the GEMM);
        # they only feed backward: skipped when nothing asks for a gradient. A tensorwise transpose
        # shares the scalar scale; the cast of a plain operand emits it from the same read
        nt_bwd = (not trans_a) and trans_b
        need_bwd = any(ctx.needs_input_grad[:2])
        # (rows are padded to whole slabs of the products where both operands of a product are made here, in
        # one launch each: codes in 16-byte groups along K and N)
        plain = not any(isinstance(t, QuantizedTensor) for t in (a, b, a_t, b_t)) and b.shape[0] % 16 == 0 and b.shape[1] % 16 == 0
        if plain:
            get_gemm_logical_shape(a, b, trans_a, trans_b)  # (padded to the same length different ones look alike)

        # (the large tile reads the forward codes as they lie in both backward products: no transposed copies)
        # (where the forward product needs no padding of its rows)
        if (nt_bwd and plain and need_bwd and b.shape[1] % 128 == 0 and not _traced(a, b) and a.is_cuda
                and vec_reads_in_place(a.shape[0], b.shape[1], b.shape[0], False)
                and vec_reads_in_place(b.shape[0], b.shape[1], a.shape[0], True)):
            nt_bwd = False

        def operand(x, x_t):
            want_t = need_bwd and nt_bwd and not isinstance(x_t, QuantizedTensor)
            if want_t and not isinstance(x, QuantizedTensor):
                pad = _whole_slabs if plain else (lambda n: n)
                q, q_t, q_s = quantize_fp8_tensorwise_t_impl(x.contiguous(), _get_fp8_dtype(config.format, True),
                                                             pad(x.shape[1]), pad(x.shape[0]))
                return q, q_s, q_t, q_s
            q, q_s, _ = _quantized_parts(x, config, True, -1)
            if want_t:
                return q, q_s, transpose_last_two(q), q_s
            return (q, q_s, x_t.qdata, x_t.scale_inv) if isinstance(x_t, QuantizedTensor) else (q, q_s, None, None)

        qa, qa_s, sa, sa_s = operand(a, a_t)
        qb, qb_s, sb, sb_s = operand(b, b_t)
        out = _gemm(qa, qa_s, trans_a, qb, qb_s, trans_b, out_dtype, False, config.granularity)
        if not need_bwd:
            pass
        elif nt_bwd:
            ctx.save_for_backward(sa, sa_s, sb, sb_s)
        else:
            ctx.save_for_backward(qa, qa_s, qb, qb_s)
        ctx.meta = (trans_a, trans_b, out_dtype, config, nt_bwd, fuse, main_grad)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        trans_a, trans_b, out_dtype, config, nt_bwd, fuse, main_grad = ctx.meta
        sa, sa_s, sb, sb_s = ctx.saved_tensors
        gran = config.granularity
        gdt = _get_fp8_dtype(config.format, False)
        acc = main_grad if fuse else None
        if nt_bwd:
            # saved: A^T [K, M], B^T [K, N] (rows as long as the gradient's have to be)
            g, g_t, g_s = quantize_fp8_tensorwise_t_impl(grad_out.contiguous(), gdt, sb.shape[1], sa.shape[1])
            grad_a = _gemm(g, g_s, False, sb, sb_s, True, out_dtype, False, gran)
            grad_b = _wgrad_gemm(sa, sa_s, False, g_t, g_s, True, out_dtype, trans_b, gran, acc)
        else:
            g, g_s = quantize_fp8(grad_out.contiguous(), gdt, gran)
            grad_a = _gemm(g, g_s, False, sb, sb_s, not trans_b, out_dtype, trans_a, gran)
            grad_b = _wgrad_gemm(sa, sa_s, not trans_a, g, g_s, False, out_dtype, trans_b, gran, acc)
        return grad_a, grad_b, None, None, None, None, None, None, None


class FP8GemmRowFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, a, b, a_t, b_t, trans_a, trans_b, out_dtype, config):
        assert trans_a == False, "trans_a has to be False"  # noqa: E712
        gran = config.granularity
        b_axis = -1 if trans_b else -2
        # operands made here have rows of whole slabs: no product copies them to pad them
        plain = trans_b and not any(isinstance(t, QuantizedTensor) for t in (a, b))
        K = a.shape[1]
        if plain:
            get_gemm_logical_shape(a, b, trans_a, trans_b)  # (padded to the same length different ones look alike)

        def along_rows(x, axis):
            if not plain or K % 128 == 0:
                return _quantized_parts(x, config, True, axis)
            return (*quant_fp8_rowwise_padded_impl(x.contiguous(), _get_fp8_dtype(config.format, True), _whole_slabs(K)), x.dtype)

        qa, qa_s, a_hp = along_rows(a, -1)
        qb, qb_s, b_hp = along_rows(b, b_axis)
        cols = K if qa.shape[1] != K else None

        def other_axis(q, q_s, hp_dtype, from_axis, given, axis):
            # the operand as backward reads it: what the forward codes stand for, quantized again
            # along the other axis -> (codes, scales, whether the codes are stored transposed, i.e.
            # contiguous along the axis that the backward product reduces over)
            if given is not None:
                assert isinstance(given, QuantizedTensor)
                return given.qdata, given.scale_inv, False
            # (a transposed operand carries the padding of the product's reduction: tokens in wgrad, N in dgrad;
            # the other one has not been padded)
            if axis == -2:
                return (*quant_fp8_rowwise_t_impl(q, q_s, hp_dtype, q.dtype, 128, cols), True)
            hp = dequantize_fp8(q, hp_dtype, gran, axis=from_axis % q.ndim, scale_inv=q_s, block_size=config.block_size)
            return (*quantize_fp8(hp, q.dtype, gran, axis=axis % q.ndim, block_size=config.block_size), False)

        out = _gemm(qa, qa_s, trans_a, qb, qb_s, trans_b, out_dtype, False, gran)
        # the operands quantized along their other axis only feed backward: skip them when no
        # input asks for a gradient (same outputs, two quantizer passes less)
        a_t_ready = b_t_ready = False
        if any(ctx.needs_input_grad[:2]):
            a_c, a_cs, a_t_ready = other_axis(qa, qa_s, a_hp, -1, a_t, -2)
            b_c, b_cs, b_t_ready = other_axis(qb, qb_s, b_hp, b_axis, b_t, -2 if trans_b else -1)
            ctx.save_for_backward(a_c, a_cs, b_c, b_cs)
        ctx.meta = (trans_a, trans_b, out_dtype, config, a_t_ready, b_t_ready)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        trans_a, trans_b, out_dtype, config, a_t_ready, b_t_ready = ctx.meta
        a_c, a_cs, b_c, b_cs = ctx.saved_tensors
        grad_out = grad_out.contiguous()
        gdt = _get_fp8_dtype(config.format, False)
        gran = config.granularity
        if b_t_ready:
            g_row, g_row_s = quant_fp8_rowwise_padded_impl(grad_out, gdt, b_c.shape[1])
        else:
            g_row, g_row_s = quantize_fp8(grad_out, gdt, gran, axis=1, block_size=config.block_size)
        grad_a = _gemm(g_row, g_row_s, False, b_c, b_cs, True if b_t_ready else not trans_b, out_dtype, trans_a, gran)
        if a_t_ready:
            g_col, g_col_s = quant_fp8_rowwise_t_impl(grad_out, None, grad_out.dtype, gdt, 128)
            grad_b = _gemm(a_c, a_cs, False, g_col, g_col_s, True, out_dtype, trans_b, gran)
        else:
            g_col, g_col_s = quantize_fp8(grad_out, gdt, gran, axis=0, block_size=config.block_size)
            grad_b = _gemm(a_c, a_cs, not trans_a, g_col, g_col_s, False, out_dtype, trans_b, gran)
        return grad_a, grad_b, None, None, None, None, None, None


class FP8GemmBlockFunction(torch.autograd.Function):
    """BLOCKWISE (128): activations and gradients in 1 x 128 blocks along the reduction of each
    product, the weight in 128 x 128 tiles that serve forward and backward. When a gradient is
    wanted the quantizers also emit, from the same read, the operands of the backward products with
    their reduction axis contiguous (the transposed 128 x 1 column codes of ``a`` and ``grad_out``).
    The input gradient reads the forward weight codes ``[N, K]`` in place; where its product cannot
    (``reads_kn_in_place``) or that does not pay (``kn_layer_pays``) the weight's quantizer writes transposed codes too."""

    @staticmethod
    def forward(ctx, a, b, a_t, b_t, trans_a, trans_b, out_dtype, config):
        assert trans_a == False, "trans_a has to be False"  # noqa: E712
        fdt = _get_fp8_dtype(config.format, True)
        gran, bs = config.granularity, config.block_size
        need_bwd = any(ctx.needs_input_grad[:2])
        a_col = a_col_s = None
        a_kmajor = False
        if isinstance(a, QuantizedTensor):
            check_quantized_tensor(a, config, axis=-1)
            a_row, a_row_s = a.qdata, a.scale_inv
            if need_bwd:
                if a_t is None:
                    a_t = QuantizedTensor.quantize(a.dequantize(), fdt, gran, axis=-2, block_size=bs)
                a_col, a_col_s = a_t.qdata, a_t.scale_inv
        elif a.dim() == 2:
            # row scales block-major, as the GEMM reads them; the column-direction copy of `a` only
            # feeds wgrad: skipped when nothing asks for a gradient
            a_row, a_row_s_km, a_col, a_col_s = quant_fp8_blockwise_kmajor_impl(a.contiguous(), fdt, bs, need_bwd)
            a_row_s = a_row_s_km.t()
            a_kmajor = need_bwd
        else:
            a_row, a_row_s = quantize_fp8(a, fdt, gran, axis=-1, block_size=bs)
        w_recipe = ScalingRecipe(use_2d_block=True)  # weight tiles serve forward and backward unchanged
        b_q_t = None
        if isinstance(b, QuantizedTensor):
            check_quantized_tensor(b, config, scaling_recipe=w_recipe)
            b_q, b_s = b.qdata, b.scale_inv
        elif ((need_bwd or not trans_b) and b.dim() == 2 and b.size(0) % 16 == 0
              and not (trans_b and a.dim() == 2 and not _traced(a, b) and b.is_cuda
                       and kn_layer_pays(a.shape[0]) and reads_kn_in_place(a.shape[0], b.shape[1], b.shape[0]))):
            b_q, b_q_t, b_s = quant_fp8_blockwise_for_weight_dual_impl(b, fdt, bs)
        else:
            b_q, b_s = quantize_fp8(b, fdt, gran, block_size=bs, scaling_recipe=w_recipe)
        b_s_t = b_s.t().contiguous() if b_q_t is not None else None
        # forward reduces over b's last axis when trans_b, dgrad over the other one
        fwd_b, fwd_s, dgrad_b, dgrad_s = (b_q, b_s, b_q_t, b_s_t) if trans_b else (b_q_t, b_s_t, b_q, b_s)
        if fwd_b is not None:
            out = _gemm(a_row, a_row_s, False, fwd_b, fwd_s, True, out_dtype, False, gran)
        else:
            out = _gemm(a_row, a_row_s, False, b_q, b_s, trans_b, out_dtype, False, gran)
        if need_bwd:
            b_ready = dgrad_b is not None
            ctx.save_for_backward(a_col, a_col_s, dgrad_b if b_ready else b_q, dgrad_s if b_ready else b_s)
            ctx.meta = (trans_a, trans_b, out_dtype, config, a_kmajor, b_ready)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        trans_a, trans_b, out_dtype, config, a_kmajor, b_ready = ctx.meta
        a_col, a_col_s, b_q, b_s = ctx.saved_tensors
        gran = config.granularity
        gdt = _get_fp8_dtype(config.format, False)
        g = grad_out.contiguous()
        if a_kmajor:
            g_row, g_row_s_km, g_col_t, g_col_s = quant_fp8_blockwise_kmajor_impl(g, gdt, config.block_size, True)
            g_row_s = g_row_s_km.t()
        else:
            g_row, g_row_s, g_col, g_col_s = quantize_fp8_with_trans(g, gdt, gran, block_size=config.block_size)
        grad_a = _gemm(g_row, g_row_s, False, b_q, b_s, True if b_ready else not trans_b, out_dtype, False, gran)
        if a_kmajor:
            # [K, M_pad] x [N, M_pad]^T: both read in place; trans_c gives the [N, K] weight layout
            grad_b = _gemm(a_col, a_col_s, False, g_col_t, g_col_s, True, out_dtype, trans_b, gran)
        else:
            grad_b = _gemm(a_col, a_col_s, not trans_a, g_col, g_col_s, False, out_dtype, trans_b, gran)
        return grad_a, grad_b, None, None, None, None, None, None


class FP8GemmMXFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, a, b, a_t, b_t, trans_a, trans_b, out_dtype, config, fuse_bgrad_accum_pattern=None):
        from primus_turbo.pytorch.kernels.quantization.quantization_impl import quantize_mxfp8_impl

        ok, why = check_mxfp8_support()
        assert ok, why
        assert trans_a == False and trans_b == True, "trans_a has to be False and trans_b has to be True"  # noqa: E712
        fuse, main_grad = _setup_fused_grad_accum(b, fuse_bgrad_accum_pattern)
        fdt = _get_fp8_dtype(config.format, True)
        gran, bs = config.granularity, config.block_size

        need_bwd = any(ctx.needs_input_grad[:2])

        def both_ways(x, x_t, recipe):
            if isinstance(x, QuantizedTensor):
                check_quantized_tensor(x, config, axis=-1, scaling_recipe=recipe)
                if not need_bwd:
                    return x.qdata, x.scale_inv, None, None
                if x_t is None:
                    x_t = QuantizedTensor.quantize(x.dequantize(), x.real_dtype, gran, axis=-2, block_size=bs,
                                                   scaling_recipe=recipe)
                return x.qdata, x.scale_inv, x_t.qdata, x_t.scale_inv
            if not need_bwd:
                # the transposed copies only feed backward: skip them when nothing asks for a gradient
                q, sc = quantize_mxfp8_impl(x, fdt, x.dim() - 1, bs, scaling_recipe=recipe)
                return q, sc, None, None
            assert bs == 32, "The block size must be 32 for MXFP8 quantization"
            return quantize_mx_operands(x, fdt, recipe, recipe, "MXFP8")

        a_row, a_row_s, a_col, a_col_s = both_ways(a, a_t, ScalingRecipe())
        b_row, b_row_s, b_col, b_col_s = both_ways(b, b_t, ScalingRecipe(use_2d_block=True))
        out = _gemm(a_row, a_row_s, False, b_row, b_row_s, True, out_dtype, False, gran)
        if need_bwd:
            ctx.save_for_backward(a_col, a_col_s, b_col, b_col_s)
        ctx.meta = (out_dtype, config, fuse, main_grad)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        out_dtype, config, fuse, main_grad = ctx.meta
        a_col, a_col_s, b_col, b_col_s = ctx.saved_tensors
        gran = config.granularity
        g = grad_out.reshape(grad_out.shape[0], -1).contiguous()
        g_row, g_row_s, g_col, g_col_s = quantize_mx_operands(g, _get_fp8_dtype(config.format, False), ScalingRecipe(),
                                                              ScalingRecipe(), "MXFP8")
        # the two-direction casts are stored transposed, so dgrad and wgrad are NT GEMMs too
        grad_a = _gemm(g_row, g_row_s, False, b_col, b_col_s, True, out_dtype, False, gran)
        grad_b = _wgrad_gemm(g_col, g_col_s, False, a_col, a_col_s, True, out_dtype, False, gran,
                             main_grad if fuse else None)
        return grad_a, grad_b, None, None, None, None, None, None, None


def gemm_fp8(
    a: Union[torch.Tensor, QuantizedTensor, QuantizedTensorPair],
    b: Union[torch.Tensor, QuantizedTensor, QuantizedTensorPair],
    trans_a: bool = False,
    trans_b: bool = False,
    out_dtype: Optional[torch.dtype] = None,
    config: Optional[Float8QuantConfig] = None,
    fuse_bgrad_accum_pattern: Optional[str] = None,
) -> torch.Tensor:
    """FP8 GEMM with autograd: ``a`` is ``(M, K)``, ``b`` is ``(K, N)`` or, with
    ``trans_b``, ``(N, K)``; returns ``(M, N)`` in ``out_dtype``.

    ``config`` selects format (E4M3 / E5M2 / HYBRID) and granularity (TENSORWISE default,
    ROWWISE, BLOCKWISE with ``block_size=128``, MX_BLOCKWISE with ``block_size=32`` and E8M0
    scales). Operands may be pre-quantized ``QuantizedTensor`` / ``QuantizedTensorPair``.
    ``fuse_bgrad_accum_pattern="megatron"`` (TENSORWISE and MX_BLOCKWISE) adds the weight
    gradient into ``b.main_grad`` inside the wgrad GEMM epilogue.
    """
    if config is None:
        config = Float8QuantConfig()
    a_data, a_t = (a.data, a.data_t) if isinstance(a, QuantizedTensorPair) else (a, None)
    b_data, b_t = (b.data, b.data_t) if isinstance(b, QuantizedTensorPair) else (b, None)
    assert a_data.ndim == 2, "Only 2D tensors are supported"
    assert b_data.ndim == 2, "Only 2D tensors are supported"
    if out_dtype is None:
        out_dtype = torch.promote_types(a_data.dtype, b_data.dtype)

    g = config.granularity
    if g == ScalingGranularity.TENSORWISE:
        return FP8GemmTensorFunction.apply(a_data, b_data, a_t, b_t, trans_a, trans_b, out_dtype, config,
                                           fuse_bgrad_accum_pattern)
    if g == ScalingGranularity.MX_BLOCKWISE:
        return FP8GemmMXFunction.apply(a_data, b_data, a_t, b_t, trans_a, trans_b, out_dtype, config,
                                       fuse_bgrad_accum_pattern)
    assert fuse_bgrad_accum_pattern is None, f"fuse_bgrad_accum_pattern is not supported for {g}"
    if g == ScalingGranularity.ROWWISE:
        return FP8GemmRowFunction.apply(a_data, b_data, a_t, b_t, trans_a, trans_b, out_dtype, config)
    if g == ScalingGranularity.BLOCKWISE:
        return FP8GemmBlockFunction.apply(a_data, b_data, a_t, b_t, trans_a, trans_b, out_dtype, config)
    raise ValueError(f"Unsupported FP8 ScalingGranularity: {g}")
