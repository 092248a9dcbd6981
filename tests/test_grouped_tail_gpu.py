"""Grouped products over more rows than the groups hold: the rows behind the last group come back zero from every
tile, and neither they nor a wanted gradient change the others. Padded offsets of two alignments from one launch."""

import pytest
import torch

pytestmark = pytest.mark.gpu

LENS = [300, 0, 131, 7, 259]


def _setup(recipe, N, K, extra):
    import primus_turbo.pytorch as turbo
    from primus_turbo.pytorch.core.low_precision import Float4QuantConfig, Float8QuantConfig, ScaleDtype
    from primus_turbo.pytorch.core.low_precision import ScalingGranularity as G

    cfg = {"rowwise": lambda: Float8QuantConfig(granularity=G.ROWWISE),
           "blockwise": lambda: Float8QuantConfig(granularity=G.BLOCKWISE, block_size=128),
           "mxfp8": lambda: Float8QuantConfig(granularity=G.MX_BLOCKWISE, block_size=32, scale_dtype=ScaleDtype.E8M0),
           "mxfp4": Float4QuantConfig}[recipe]()
    op = turbo.ops.grouped_gemm_fp4 if recipe == "mxfp4" else turbo.ops.grouped_gemm_fp8
    g = torch.Generator().manual_seed(N + K)
    x = torch.randn(sum(LENS) + extra, K, generator=g).to(torch.bfloat16).cuda()
    w = torch.randn(len(LENS), N, K, generator=g).to(torch.bfloat16).cuda()
    return op, x, w, torch.tensor(LENS, device="cuda"), cfg


@pytest.mark.parametrize("extra", [1, 77])
@pytest.mark.parametrize("recipe,N,tile", [("rowwise", 262, 1), ("rowwise", 262, 3), ("blockwise", 262, 2), ("blockwise", 262, 3),
                                           ("blockwise", 262, 4), ("mxfp8", 262, 1), ("mxfp8", 262, 3), ("mxfp8", 262, 4),
                                           ("mxfp4", 288, 1), ("mxfp4", 288, 3), ("mxfp4", 288, 4)])
def test_rows_behind_the_groups(native_lib, recipe, N, tile, extra):
    from primus_turbo.pytorch.kernels.grouped_gemm import grouped_gemm_fp8_impl as impl

    op, x, w, lens, cfg = _setup(recipe, N, 640, extra)
    used = sum(LENS)
    pin = "TILE_CFG" if recipe == "blockwise" else "MX_TILE_CFG"
    try:
        setattr(impl, pin, tile)
        tight = op(x[:used].contiguous(), w, lens, trans_b=True, config=cfg)
        junk = [torch.full((x.shape[0] + 512, N), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(4)]
        del junk  # (what the next allocations of this size find)
        out = op(x, w, lens, trans_b=True, config=cfg)
        with_grad = op(x.clone().requires_grad_(True), w, lens, trans_b=True, config=cfg)
    finally:
        setattr(impl, pin, 0)
    assert torch.equal(out[:used], tight)
    assert out.shape[0] == x.shape[0] and not out[used:].any()
    assert torch.equal(out, with_grad.detach())


@pytest.mark.parametrize("lens", [[5], [0, 0, 0], [1, 32, 33, 0, 127, 128, 129], list(range(0, 300, 2))])
def test_two_paddings_of_the_offsets(native_lib, lens):
    from primus_turbo.pytorch.kernels.quantization.quantization_impl import _group_offs_pair

    got = _group_offs_pair(torch.tensor(lens, device="cuda"), 32, 128)
    for align, got_lens, got_offs in ((32, *got[:2]), (128, *got[2:])):
        want = [-(-n // align) * align for n in lens]
        assert got_lens.tolist() == want
        assert got_offs.tolist() == [sum(want[:i]) for i in range(len(want) + 1)]
