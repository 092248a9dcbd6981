"""A product that no gradient is asked of makes its forward operands only; its result is the one that the
same call gives when gradients are wanted, and a gradient asked of either operand still arrives."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _cfg(recipe):
    from primus_turbo.pytorch.core.low_precision import Float4QuantConfig, Float8QuantConfig, ScaleDtype, ScalingGranularity as G

    if recipe == "mxfp4":
        return Float4QuantConfig()
    if recipe == "mxfp8":
        return Float8QuantConfig(granularity=G.MX_BLOCKWISE, block_size=32, scale_dtype=ScaleDtype.E8M0)
    return Float8QuantConfig(granularity=G.TENSORWISE)


@pytest.mark.parametrize("recipe", ["tensorwise", "mxfp8", "mxfp4"])
@pytest.mark.parametrize("quantized", [False, True])
@pytest.mark.parametrize("M,N,K", [(32, 96, 160), (288, 512, 1024)])
def test_forward_only(native_lib, recipe, quantized, M, N, K):
    import primus_turbo.pytorch as turbo
    from primus_turbo.pytorch.core.quantized_tensor import create_quantized_weight

    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    w = torch.randn(N, K, generator=g).to(torch.bfloat16).cuda()
    cfg = _cfg(recipe)
    op = turbo.ops.gemm_fp4 if recipe == "mxfp4" else turbo.ops.gemm_fp8
    if quantized:
        w = create_quantized_weight(w, turbo.float4_e2m1fn_x2 if recipe == "mxfp4" else turbo.float8_e4m3, cfg)[0]
    plain = op(x, w, trans_b=True, config=cfg)
    xg = x.clone().requires_grad_(True)
    out = op(xg, w, trans_b=True, config=cfg)
    assert torch.equal(plain, out.detach()) and not plain.requires_grad
    (gx,) = torch.autograd.grad(out, (xg,), torch.ones_like(out))
    ref = torch.ones(M, N) @ (w.dequantize() if quantized else w).float().cpu()
    # E4M3 carries 4 significant bits, E2M1 two: operands rounded to half a unit, both operands
    bound = 2 ** -2 if recipe == "mxfp4" else 2 ** -4
    assert (gx.float().cpu() - ref).norm() / ref.norm() < bound
    if quantized:
        return
    wg = w.clone().requires_grad_(True)  # the weight alone
    out = op(x, wg, trans_b=True, config=cfg)
    assert torch.equal(plain, out.detach())
    (gw,) = torch.autograd.grad(out, (wg,), torch.ones_like(out))
    ref = torch.ones(N, M) @ x.float().cpu()
    assert (gw.float().cpu() - ref).norm() / ref.norm() < bound
