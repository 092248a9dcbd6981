"""GPU parity of the GEMM kernels at sizes that hang over a tile: columns, rows and K that are no multiple of
anything a tile is made of. Operands hold small whole numbers, so every product is exact in fp32 and the
result is the whole-number product rounded once to the output type."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

G = None


@pytest.fixture(scope="module", autouse=True)
def _impl(native_lib):
    global G, impl
    from primus_turbo.pytorch.core.low_precision import ScalingGranularity as G
    from primus_turbo.pytorch.kernels.gemm import gemm_fp8_impl as impl


def _whole(rows, cols, seed):
    """fp8 codes of whole numbers in [-4, 4] and the numbers."""
    g = torch.Generator().manual_seed(seed)
    v = torch.randint(-4, 5, (rows, cols), generator=g).float()
    return v.to(torch.float8_e4m3fn).cuda(), v


def _vec(M, N, K, out_dtype, accumulate, cfg, seed=0):
    (a, av), (b, bv) = _whole(M, K, seed), _whole(N, K, seed + 1)
    sa = 2.0 ** torch.randint(-2, 3, (M, 1)).float()
    sb = 2.0 ** torch.randint(-2, 3, (N, 1)).float()
    ref = (av.double() * sa.double()) @ (bv.double() * sb.double()).T
    old = torch.randint(-8, 9, (M, N)).to(out_dtype)
    out = old.cuda().clone()
    impl.TILE_CFG = cfg
    try:
        impl._launch(a, sa.cuda(), False, b, sb.cuda(), True, out, False, G.ROWWISE, accumulate)
    finally:
        impl.TILE_CFG = 0
    want = (ref + old.double() if accumulate else ref).float().to(out_dtype)
    return out.cpu(), want


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("N", [264, 268, 262, 40, 7])  # 8-, 4- and 2-column groups at the edge; less than a sub-tile
@pytest.mark.parametrize("cfg", [1, 2, 3])
def test_ragged_columns(out_dtype, accumulate, N, cfg):
    got, want = _vec(333, N, 512, out_dtype, accumulate, cfg)
    assert torch.equal(got, want), f"{(got != want).sum().item()} of {got.numel()} differ"


@pytest.mark.parametrize("M,N", [(1, 16), (333, 264)])
@pytest.mark.parametrize("K", [16, 144, 272, 2000, 40, 257])  # padded in 16-byte groups, byte by byte
def test_ragged_reduction(M, N, K):
    got, want = _vec(M, N, K, torch.float32, False, 0)
    assert torch.equal(got, want), f"{(got != want).sum().item()} of {got.numel()} differ"


def _exact_operand(recipe, rows, K, seed):
    """Codes and scales of an operand on the GPU and the whole numbers that they stand for (scales are 1)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    v = torch.randint(-4, 5, (rows, K), generator=g, device="cuda")
    if recipe == "mxfp4":  # E2M1 codes of 0..4 and the sign bit, even element in the low nibble
        nib = torch.tensor([0, 2, 4, 5, 6], device="cuda")[v.abs()] + 8 * (v < 0)
        codes = (nib[:, 0::2] + 16 * nib[:, 1::2]).to(torch.uint8).view(torch.float4_e2m1fn_x2)
    else:
        codes = v.to(torch.float8_e4m3fn)
    scale = (torch.ones(rows, 1, device="cuda") if recipe == "rowwise"
             else torch.full((rows, K // 32), 127, dtype=torch.uint8, device="cuda"))
    return codes, scale, v.float()


@pytest.mark.parametrize("recipe,out_dtype,accumulate", [("rowwise", torch.bfloat16, False), ("rowwise", torch.float32, True),
                                                         ("mxfp8", torch.bfloat16, False), ("mxfp4", torch.bfloat16, False)])
def test_output_above_2_gib(recipe, out_dtype, accumulate):
    """Eight columns in the last tile and more than 2 GiB of result behind the first tiles: every element is
    the product of its own row and column (csrc/store_window.h, walked on the host for more sizes)."""
    N, K = 16 * 1024 + 8, 128
    M = (1 << 31) // (N * out_dtype.itemsize) + 700
    a, sa, av = _exact_operand(recipe, M, K, 1)
    b, sb, bv = _exact_operand(recipe, N, K, 2)
    out = torch.full((M, N), 3.0, dtype=out_dtype, device="cuda")
    impl._launch(a, sa, False, b, sb, True, out, False, G.ROWWISE if recipe == "rowwise" else G.MX_BLOCKWISE, accumulate)
    for m in range(0, M, 8192):  # (whole numbers up to 2^11 are exact in fp32; both sides round once)
        want = av[m : m + 8192] @ bv.T
        want = (want + 3.0 if accumulate else want).to(out_dtype)
        assert torch.equal(out[m : m + 8192], want), f"rows {m}..: {(out[m : m + 8192] != want).sum().item()} differ"
