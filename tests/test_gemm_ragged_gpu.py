"""GPU parity of the GEMM kernels at sizes that hang over a tile: columns, rows and K that are no multiple of
anything a tile is made of. Operands hold small whole numbers and powers of two as scales, so every product
is exact in fp32 and the result is the exact product rounded once to the output type."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _impl(native_lib):
    global GRAN, impl, grouped
    from primus_turbo.pytorch.core.low_precision import ScalingGranularity as G
    from primus_turbo.pytorch.kernels.gemm import gemm_fp8_impl as impl
    from primus_turbo.pytorch.kernels.grouped_gemm import grouped_gemm_fp8_impl as grouped

    GRAN = {"rowwise": G.ROWWISE, "blockwise": G.BLOCKWISE, "mxfp8": G.MX_BLOCKWISE, "mxfp4": G.MX_BLOCKWISE}


def _exact_operand(recipe, rows, K, seed, scaled=False, weight=False):
    """Codes and scales of an operand on the GPU and the values that they stand for: whole numbers, with
    ``scaled`` times powers of two (BLOCKWISE ``weight``: scales of 128 x 128 tiles)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    v = torch.randint(-4, 5, (rows, K), generator=g, device="cuda")
    if recipe == "mxfp4":  # E2M1 codes of 0..4 and the sign bit, even element in the low nibble
        nib = torch.tensor([0, 2, 4, 5, 6], device="cuda")[v.abs()] + 8 * (v < 0)
        codes = (nib[:, 0::2] + 16 * nib[:, 1::2]).to(torch.uint8).view(torch.float4_e2m1fn_x2)
    else:
        codes = v.to(torch.float8_e4m3fn)
    block = {"rowwise": K, "blockwise": 128}.get(recipe, 32)
    height = 128 if weight and recipe == "blockwise" else 1
    e = torch.randint(-2, 3, (-(-rows // height), -(-K // block)), generator=g, device="cuda") * int(scaled)
    scale = 2.0**e if recipe in ("rowwise", "blockwise") else (e + 127).to(torch.uint8)
    values = v * (2.0**e).repeat_interleave(height, 0)[:rows].repeat_interleave(block, 1)[:, :K]
    return codes, scale, values


def _dense(recipe, M, N, K, out_dtype, accumulate, cfg):
    a, sa, av = _exact_operand(recipe, M, K, 0, True)
    b, sb, bv = _exact_operand(recipe, N, K, 1, True, weight=True)
    ref = av.double().cpu() @ bv.double().cpu().T
    old = torch.randint(-8, 9, (M, N), generator=torch.Generator().manual_seed(2)).to(out_dtype)
    out = old.cuda()
    impl.TILE_CFG = cfg
    try:
        impl._launch(a, sa, False, b, sb, True, out, False, GRAN[recipe], accumulate)
    finally:
        impl.TILE_CFG = 0
    want = (ref + old.double() if accumulate else ref).float().to(out_dtype)
    return out.cpu(), want


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("N", [264, 268, 262, 40, 7])  # 8-, 4- and 2-column groups at the edge; less than a sub-tile
@pytest.mark.parametrize("recipe,cfg", [(r, c) for r in ("rowwise", "mxfp8", "mxfp4", "blockwise") for c in (1, 2, 3, 4)
                                        if (r, c) != ("rowwise", 4)])
def test_ragged_columns(out_dtype, accumulate, N, recipe, cfg):
    got, want = _dense(recipe, 333, N, 512, out_dtype, accumulate, cfg)
    assert torch.equal(got, want), f"{(got != want).sum().item()} of {got.numel()} differ"


@pytest.mark.parametrize("M,N", [(1, 16), (333, 264)])
@pytest.mark.parametrize("K", [16, 144, 272, 2000, 40, 257])  # padded in 16-byte groups, byte by byte
def test_ragged_reduction(M, N, K):
    got, want = _dense("rowwise", M, N, K, torch.float32, False, 0)
    assert torch.equal(got, want), f"{(got != want).sum().item()} of {got.numel()} differ"


@pytest.mark.parametrize("cfg", [1, 2, 3, 4])
@pytest.mark.parametrize("recipe", ["mxfp8", "mxfp4"])
def test_blocks_that_end_inside_a_scale_word(recipe, cfg):
    """38 blocks of 32: the last word of the last row of either operand holds two of them."""
    M, N, K = 333, 264, 1216
    (a, sa, av), (b, sb, bv) = (_exact_operand(recipe, rows, K, seed, True) for rows, seed in ((M, 0), (N, 1)))
    sa, sb = (torch.nn.functional.pad(s, (0, 2)) for s in (sa, sb))
    out = torch.empty(M, N, dtype=torch.float32, device="cuda")
    impl.TILE_CFG = cfg
    try:
        impl._launch(a, sa, False, b, sb, True, out, False, GRAN[recipe], False)
    finally:
        impl.TILE_CFG = 0
    want = (av.double() @ bv.double().T).float()
    assert torch.equal(out, want), f"{(out != want).sum().item()} of {out.numel()} differ"


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
    impl._launch(a, sa, False, b, sb, True, out, False, GRAN[recipe], accumulate)
    for m in range(0, M, 8192):  # (whole numbers up to 2^11 are exact in fp32; both sides round once)
        want = av[m : m + 8192] @ bv.T
        want = (want + 3.0 if accumulate else want).to(out_dtype)
        assert torch.equal(out[m : m + 8192], want), f"rows {m}..: {(out[m : m + 8192] != want).sum().item()} differ"


LENS = [300, 0, 130, 7, 256]  # rows of the groups (MX variable K: elements in whole 256-blocks)


@pytest.mark.parametrize("recipe", ["rowwise", "mxfp8", "mxfp4", "blockwise"])
@pytest.mark.parametrize("N", [264, 268, 262, 7])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_ragged_columns_of_groups(recipe, N, out_dtype):
    if recipe == "blockwise" and out_dtype == torch.float32:
        pytest.skip("grouped block-scaled results are 16-bit")
    K, M = 512, sum(LENS)
    offs = torch.tensor([0, *LENS]).cumsum(0).cuda()
    a, sa, av = _exact_operand(recipe, M, K, 3, True)
    bs = [_exact_operand(recipe, N, K, 4 + g, True, weight=True) for g in range(len(LENS))]
    b, sb = (torch.stack([t[i].view(torch.uint8) if i == 0 else t[i] for t in bs]) for i in range(2))
    out = grouped.grouped_gemm_fp8_impl(a, b.view(a.dtype), sa.t().contiguous() if recipe == "blockwise" else sa, sb,
                                        torch.tensor(LENS).cuda(), offs, False, True, out_dtype, GRAN[recipe].value, None, 0)
    for g, n in enumerate(LENS):
        rows = slice(int(offs[g]), int(offs[g]) + n)
        want = (av[rows].double().cpu() @ bs[g][2].double().cpu().T).float().to(out_dtype)
        assert torch.equal(out[rows].cpu(), want), f"group {g}"


@pytest.mark.parametrize("recipe", ["rowwise", "mxfp8", "mxfp4"])
@pytest.mark.parametrize("N", [264, 268, 262, 7])
@pytest.mark.parametrize("out_dtype,accumulate", [(torch.bfloat16, False), (torch.float32, True)])
def test_ragged_columns_of_variable_k(recipe, N, out_dtype, accumulate):
    M, lens = 72, ([256, 0, 512] if recipe.startswith("mx") else [256, 0, 333])
    K = sum(lens)
    offs = torch.tensor([0, *lens]).cumsum(0).cuda()
    a, sa, av = _exact_operand(recipe, M, K, 5, True)
    b, sb, bv = _exact_operand(recipe, N, K, 6, True)
    old = torch.randint(-8, 9, (len(lens), M, N), generator=torch.Generator().manual_seed(2)).to(out_dtype)
    out = old.cuda()
    if recipe == "rowwise":
        grouped._variable_k_vec(a.t().contiguous(), b.t().contiguous(), sa, sb, offs, True, False, False, out, accumulate)
    else:
        grouped._variable_k_mx(a, b, sa, sb, offs, False, False, False, out, accumulate)
    for g, n in enumerate(lens):
        k = slice(int(offs[g]), int(offs[g]) + n)
        want = av[:, k].double().cpu() @ bv[:, k].double().cpu().T + (old[g].double() if accumulate else 0.0)
        assert torch.equal(out[g].cpu(), want.float().to(out_dtype)), f"group {g}"
