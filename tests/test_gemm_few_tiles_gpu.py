"""GPU parity of dense products with few output tiles: the kernel that splits K over the wavefronts of a
workgroup (csrc/gemm_direct.h) at the edges of each of its tiles and of K, and the 128 x 128 tiles whose copies
run three slabs ahead. Operands hold small whole numbers and powers of two as scales, so every product is
exact in fp32 and the result is the exact product rounded once to the output type."""

import pytest
import torch

from test_gemm_ragged_gpu import _exact_operand

pytestmark = pytest.mark.gpu

RECIPES = ("rowwise", "blockwise", "vectors", "mxfp8", "mxfp4")  # vectors: 1 x 128 scales on both operands
# tile of 16 x 16, x 32, x 64, 32 x 32, 32 x 64, 64 x 64 (up to eight slabs) on 256 CUs; less than a tile
SHAPES = [(16, 512), (1, 40), (9, 8190), (13, 16380), (61, 4091), (120, 4090), (200, 4084), (3, 7)]


@pytest.fixture(scope="module", autouse=True)
def _impl(native_lib):
    global G, impl
    from primus_turbo.pytorch.core.low_precision import ScalingGranularity as G
    from primus_turbo.pytorch.kernels.gemm import gemm_fp8_impl as impl


def _check(recipe, M, N, K, out_dtype=torch.bfloat16, accumulate=False, dtypes=None, special=None):
    """``recipe`` of RECIPES, or mxfp8 / mxfp4 with " words": scales word-major."""
    recipe, words = recipe.split()[0], recipe.endswith(" words")
    a, sa, av = _exact_operand("blockwise" if recipe == "vectors" else recipe, M, K, 0, True)
    b, sb, bv = _exact_operand("blockwise" if recipe == "vectors" else recipe, N, K, 1, True, weight=recipe == "blockwise")
    if dtypes:  # (the whole numbers are exact in either format)
        a, b = a.float().to(dtypes[0]), b.float().to(dtypes[1])
    if special:
        _make_special(special, a, sa, av)
        _make_special(special, b, sb, bv)
    if recipe == "vectors":
        sa, sb = sa.t().contiguous(), sb.t().contiguous()
    if recipe.startswith("mx"):  # rows of whole words, as the quantizers leave them
        sa, sb = (torch.nn.functional.pad(s, (0, -s.shape[1] % 4)) for s in (sa, sb))
    if words:
        sa, sb = (s.contiguous().view(torch.int32).t().contiguous() for s in (sa, sb))
    gran = {"rowwise": G.ROWWISE, "blockwise": G.BLOCKWISE, "vectors": G.BLOCKWISE}.get(recipe, G.MX_BLOCKWISE)
    old = torch.randint(-8, 9, (M, N), device="cuda").to(out_dtype)
    out = old.clone()
    impl._launch(a, sa, False, b, sb, True, out, False, gran, accumulate)
    want = av.double() @ bv.double().T
    want = (want + old.double() if accumulate else want).float().to(out_dtype)
    wrong = (out != want) & ~(out.isnan() & want.isnan())
    assert not wrong.any(), f"{wrong.sum().item()} of {out.numel()} differ"


def _make_special(special, codes, scales, values):
    """"zero": every code 0. "nan" / "inf": such a code in two rows, the last one among them (MXFP4 has none: a NaN scale)."""
    rows, k = [codes.shape[0] // 3, codes.shape[0] - 1], values.shape[1] // 2
    if special == "zero":
        codes.view(torch.uint8).zero_()
        values.zero_()
    elif codes.shape[1] == values.shape[1]:
        codes.view(torch.uint8)[rows, k] = 0x7F if special == "nan" else 0x7C
        values[rows, k] = float(special)
    else:
        scales.view(torch.uint8)[rows, -1] = 0xFF
        values[rows, -32:] = float(special)


@pytest.mark.parametrize("K", [32, 512, 1024, 992])
@pytest.mark.parametrize("M,N", SHAPES)
@pytest.mark.parametrize("recipe", RECIPES)
def test_tiles(recipe, M, N, K):
    _check(recipe, M, N, K)


@pytest.mark.parametrize("K", [16, 40, 257, 1296, 4208, 16384])  # rows of 16-byte groups or padded; many slabs
@pytest.mark.parametrize("M,N", [(16, 512), (61, 4091)])
@pytest.mark.parametrize("recipe", ["rowwise", "blockwise", "vectors"])
def test_reductions(recipe, M, N, K):
    _check(recipe, M, N, K)


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("N", [40, 42])
@pytest.mark.parametrize("recipe", RECIPES)
def test_outputs(recipe, N, accumulate, out_dtype):
    _check(recipe, 21, N, 640, out_dtype, accumulate)


@pytest.mark.parametrize("da", [torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("db", [torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("recipe", RECIPES[:-1])
def test_formats(recipe, da, db):
    _check(recipe, 61, 4091, 640, dtypes=(da, db))


@pytest.mark.parametrize("M,N,K", [(700, 1032, 1216), (257, 4090, 2048), (1024, 4096, 1152)])
@pytest.mark.parametrize("recipe", RECIPES)
def test_one_large_tile_per_cu(recipe, M, N, K):
    _check(recipe, M, N, K)


# the direct kernel, four stages or two teams, with edges in every direction; rows that are not special stay exact
@pytest.mark.parametrize("special", ["zero", "nan", "inf"])
@pytest.mark.parametrize("M,N,K", [(13, 1020, 992), (61, 4091, 640), (700, 1032, 2176)])
@pytest.mark.parametrize("recipe", RECIPES)
def test_special_values(recipe, M, N, K, special):
    if special == "inf" and recipe == "mxfp4":
        pytest.skip("E2M1 and E8M0 have no infinity")
    _check(recipe, M, N, K, torch.float32, dtypes=(torch.float8_e5m2,) * 2 if special == "inf" else None, special=special)
