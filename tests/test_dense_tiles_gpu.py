"""GPU parity of the tiles a dense product may take (256 x 256 with eight wavefronts, also with a scale per
column; 256 x 128; 128 x 128) at sizes where the rule changes its choice and where a tile hangs over an edge.
The operands make every product exact (see test_gemm_few_tiles_gpu)."""

import pytest
import torch

import test_gemm_few_tiles_gpu as few

pytestmark = pytest.mark.gpu
_impl = few._impl  # the fixture that loads the operators


@pytest.fixture(params=[0, 1, 2, 3, 4])
def tile(request, _impl):
    few.impl.TILE_CFG = request.param
    yield request.param
    few.impl.TILE_CFG = 0


# exactly one tile of 256; one element over an edge; ragged on both sides; fewer rows than half a tile
@pytest.mark.parametrize("M,N,K", [(256, 256, 512), (257, 520, 640), (510, 1002, 1216), (100, 264, 4000)])
@pytest.mark.parametrize("recipe", few.RECIPES)
def test_edges(recipe, M, N, K, tile):
    few._check(recipe, M, N, K // 32 * 32)


@pytest.mark.parametrize("special", ["zero", "nan"])
@pytest.mark.parametrize("recipe", few.RECIPES)
def test_special_values(recipe, special, tile):
    few._check(recipe, 510, 1002, 1216, torch.float32, special=special)


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("recipe", ["vectors", "blockwise", "mxfp8"])
def test_outputs(recipe, accumulate, out_dtype):
    few.impl.TILE_CFG = 1
    try:
        few._check(recipe, 300, 520, 640, out_dtype, accumulate)
    finally:
        few.impl.TILE_CFG = 0


@pytest.mark.parametrize("da", [torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("db", [torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("recipe", ["vectors", "mxfp8"])
def test_formats(recipe, da, db):
    few.impl.TILE_CFG = 1
    try:
        few._check(recipe, 300, 520, 640, dtypes=(da, db))
    finally:
        few.impl.TILE_CFG = 0


# 64, 128 (both ways round), 192 and 320 tiles of 256 x 256 on 256 CUs, and whole rounds of them
@pytest.mark.parametrize("M,N,K", [(2048, 2048, 512), (4090, 2048, 544), (2040, 4104, 512), (3001, 4096, 512), (5000, 4096, 512),
                                   (16384, 1024, 544), (8192, 4096, 512)])
@pytest.mark.parametrize("recipe", few.RECIPES)
def test_rule(recipe, M, N, K):
    few._check(recipe, M, N, K)


# two teams of wavefronts share the slabs: odd and even numbers of them, the shortest K of each recipe and the lines of the
# rule
@pytest.mark.parametrize("out_dtype,accumulate", [(torch.bfloat16, False), (torch.float16, True), (torch.float32, False), (torch.float32, True)])
@pytest.mark.parametrize("K", [512, 640, 896, 1024, 2048, 2176, 4096, 4352])
@pytest.mark.parametrize("M,N", [(600, 2056), (513, 2047)])
@pytest.mark.parametrize("recipe", ["vectors", "blockwise", "mxfp8", "mxfp4", "mxfp8 words", "mxfp4 words"])
def test_teams(recipe, M, N, K, out_dtype, accumulate):
    few._check(recipe, M, N, K, out_dtype, accumulate)


@pytest.mark.parametrize("da", [torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("db", [torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("recipe", ["vectors", "blockwise", "mxfp8"])
def test_team_formats(recipe, da, db):
    few._check(recipe, 600, 2056, 2176, dtypes=(da, db))
