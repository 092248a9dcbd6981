"""The scale layouts that meet in the grouped MX weight gradient: the variable-K product reads both operands' scales
in one layout, so the gradient is quantized in that of the activation, which the caller may have quantized."""

import importlib

import pytest
import torch

import primus_turbo.pytorch as turbo
from primus_turbo.pytorch.core.low_precision import Float4QuantConfig, Float8QuantConfig, Format, ScaleDtype, ScalingRecipe
from primus_turbo.pytorch.core.low_precision import ScalingGranularity as G
from primus_turbo.pytorch.core.quantized_tensor import QuantizedTensor, QuantizedTensorPair

FP4 = getattr(torch, "float4_e2m1fn_x2", None)


@pytest.mark.parametrize("given", [False, True])
@pytest.mark.parametrize("fp4", [False, pytest.param(True, marks=pytest.mark.skipif(FP4 is None, reason="no float4_e2m1fn_x2"))])
def test_one_layout_for_both_operands(fp4, given, native_lib, monkeypatch):
    import primus_turbo.pytorch.core.low_precision as LP

    monkeypatch.setattr(LP, "_needs", lambda *a: (True, ""))
    mod = importlib.import_module("primus_turbo.pytorch.ops.grouped_gemm_fp4" if fp4 else "primus_turbo.pytorch.ops.grouped_gemm_fp8")
    wrapper = "_bgrad_grouped_gemm_fp4_impl_wrapper" if fp4 else "_grouped_gemm_fp8_variable_k_impl_wrapper"
    scales, product = [], getattr(mod, wrapper)

    def recorded(a, b, a_s, b_s, *rest, **kw):
        scales.append((a_s.dtype, b_s.dtype))
        return product(a, b, a_s, b_s, *rest, **kw)

    monkeypatch.setattr(mod, wrapper, recorded)
    if fp4:
        op, dt, config = turbo.ops.grouped_gemm_fp4, FP4, Float4QuantConfig()
    else:
        op, dt = turbo.ops.grouped_gemm_fp8, turbo.float8_e4m3
        config = Float8QuantConfig(format=Format.E4M3, granularity=G.MX_BLOCKWISE, block_size=32, scale_dtype=ScaleDtype.E8M0)
    lens = torch.empty(4, device="meta", dtype=torch.int64)
    a = torch.empty(512, 256, device="meta", dtype=torch.bfloat16)
    b = torch.empty(4, 384, 256, device="meta", dtype=torch.bfloat16, requires_grad=True)
    if given:
        from primus_turbo.pytorch.kernels.quantization import quantization_impl as Q

        offs = torch.empty(5, device="meta", dtype=torch.int64)
        recipes = ScalingRecipe(), ScalingRecipe(use_rht=fp4)
        q = (Q.grouped_quantize_mxfp4_impl if fp4 else Q.grouped_quantize_mxfp8_impl)(
            a, dt, None, 32, lens, offs, True, *recipes)

        def wrapped(data, scale, lens_padded, offs_padded, axis, recipe):
            return QuantizedTensor(data, scale, shape=a.shape, orig_dtype=a.dtype, dest_dtype=dt, granularity=G.MX_BLOCKWISE,
                                   orig_group_lens=lens, orig_group_offs=offs, group_lens=lens_padded, group_offs=offs_padded,
                                   is_grouped_tensor=True, block_size=32, scaling_recipe=recipe, quantized_axis=axis)

        a = QuantizedTensorPair(wrapped(q[0], q[1], q[4], q[5], 1, recipes[0]), wrapped(q[2], q[3], q[6], q[7], 0, recipes[1]))
    out = op(a, b, lens, trans_b=True, config=config)
    out.backward(torch.empty_like(out))
    assert len(scales) == 1
    of_grad, of_activation = scales[0]
    assert of_grad == of_activation
    assert (of_activation != torch.int32) == given  # quantized here: the word-major layout that products read
