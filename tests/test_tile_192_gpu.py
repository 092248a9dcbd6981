"""GPU parity of the 192 x 256 tile (dense products with vector scales, MXFP8): the operands make every product exact (see
test_gemm_few_tiles_gpu)."""

import pytest
import torch

import test_gemm_few_tiles_gpu as few

pytestmark = pytest.mark.gpu
_impl = few._impl  # the fixture that loads the operators


@pytest.fixture
def pinned(_impl):
    few.impl.TILE_CFG = 5
    yield
    few.impl.TILE_CFG = 0


# one tile exactly; one row over and short of it; ragged on both sides, unaligned columns among them; fewer rows than a wavefront's
@pytest.mark.parametrize("M,N,K", [(192, 256, 512), (193, 264, 640), (191, 520, 576), (578, 1002, 1216), (70, 254, 4000), (1, 512, 1024)])
@pytest.mark.parametrize("recipe", ["rowwise", "mxfp8", "mxfp8 words"])
def test_edges(recipe, M, N, K, pinned):
    few._check(recipe, M, N, K // 128 * 128 if "words" in recipe else K // 32 * 32)


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("recipe", ["rowwise", "mxfp8"])
def test_outputs(recipe, accumulate, out_dtype, pinned):
    few._check(recipe, 300, 520, 640, out_dtype, accumulate)


@pytest.mark.parametrize("da", [torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("db", [torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("recipe", ["rowwise", "mxfp8"])
def test_formats(recipe, da, db, pinned):
    few._check(recipe, 300, 520, 640, dtypes=(da, db))


@pytest.mark.parametrize("special", ["zero", "nan"])
@pytest.mark.parametrize("recipe", ["rowwise", "mxfp8"])
def test_special_values(recipe, special, pinned):
    few._check(recipe, 510, 1002, 1216, torch.float32, special=special)


# where the rule takes the tile: 16 x 12, 16 x 16 and 15 x 16 tiles of it on 256 CUs, and more rounds than one (with vector scales not
# of as few slabs)
@pytest.mark.parametrize("M,N,K", [(3001, 2880, 1024), (3001, 4096, 1024), (2880, 4096, 1024), (5760, 4096, 544), (5760, 4096, 1056)])
@pytest.mark.parametrize("recipe", ["rowwise", "mxfp8"])
def test_rule(recipe, M, N, K, native_lib):
    assert (native_lib.pt_gemm_mx_tile(M, N, K, 0) if recipe == "mxfp8" else native_lib.pt_gemm_fp8_tile(M, N, K)) == (
        3 if recipe == "rowwise" and K == 544 else 5)
    few._check(recipe, M, N, K)
