"""Word-major MX scales, which pass between this package's quantizers and its products: the same bytes as the
row-major scales in another order, and the same products bit for bit, in every tile and beside a row-major operand
(whose products the other MX tests hold against the oracle)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

FP4 = getattr(torch, "float4_e2m1fn_x2", None)
LENS = [300, 0, 131, 7, 259]


@pytest.fixture(scope="module", autouse=True)
def _impl(native_lib):
    global Q, D, GG, Recipe, GRAN
    from primus_turbo.pytorch.core.low_precision import ScalingGranularity, ScalingRecipe as Recipe
    from primus_turbo.pytorch.kernels.gemm import gemm_fp8_impl as D
    from primus_turbo.pytorch.kernels.grouped_gemm import grouped_gemm_fp8_impl as GG
    from primus_turbo.pytorch.kernels.quantization import quantization_impl as Q

    GRAN = ScalingGranularity.MX_BLOCKWISE.value


def _x(*shape, dtype=torch.bfloat16):
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _bytes(words):
    """int32 words [.., W, R] -> the scale bytes [.., R, 4 W]"""
    return words.transpose(-2, -1).clone(memory_format=torch.contiguous_format).view(torch.uint8)


def _same(a, b):
    assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("shape", [(1, 32), (130, 160), (384, 512), (3, 100, 96), (2, 256, 384)])
@pytest.mark.parametrize("dtype", [torch.float8_e4m3fn, torch.float8_e5m2, FP4])
@pytest.mark.parametrize("recipe", [{}, {"use_2d_block": True}])
def test_dense_scales(shape, dtype, recipe):
    what = "MXFP4" if dtype == FP4 else "MXFP8"
    x, r = _x(*shape), Recipe(**recipe)
    q, s, qt, st = Q._quantize_mx_impl(x, dtype, None, 32, True, r, r, what)
    wq, ws, wqt, wst = Q.quantize_mx_operands(x, dtype, r, r, what)
    for plain, words in ((q, wq), (qt, wqt)):
        _same(plain, words)
    for plain, words in ((s, ws), (st, wst)):
        _same(plain, _bytes(words))


# zeros, an infinity and a NaN; stochastic rounding from one seed
@pytest.mark.parametrize("recipe", [{}, {"use_sr": True}, {"use_sr": True, "use_rht": True}])
@pytest.mark.parametrize("values", [(0.0,), (float("inf"),), (float("nan"), float("-inf"))])
@pytest.mark.parametrize("dtype", [torch.float8_e4m3fn, FP4])
def test_special_values_and_stochastic_rounding(dtype, values, recipe, monkeypatch):
    if recipe and dtype != FP4:
        pytest.skip("belongs to the MXFP4 recipe")
    monkeypatch.setattr(Q, "_next_sr_seed", lambda *flags: 12345)
    what, r = "MXFP4" if dtype == FP4 else "MXFP8", Recipe(**recipe)
    x = _x(130, 160)
    x[32:64, 32:64] = 0
    for i, v in enumerate(values):
        x[129 - i, 159 - i] = v
    q, s, qt, st = Q._quantize_mx_impl(x, dtype, None, 32, True, r, r, what)
    wq, ws, wqt, wst = Q.quantize_mx_operands(x, dtype, r, r, what)
    for plain, words in ((q, wq), (qt, wqt), (s, _bytes(ws)), (st, _bytes(wst))):
        _same(plain, words)


@pytest.mark.parametrize("N", [96, 384])
@pytest.mark.parametrize("dtype", [torch.float8_e4m3fn, FP4])
@pytest.mark.parametrize("glu", [False, True])
def test_grouped_scales(N, dtype, glu):
    lens = torch.tensor(LENS, device="cuda")
    offs = torch.cat([lens.new_zeros(1), lens.cumsum(0)])
    x = _x(sum(LENS), 2 * N if glu else N)
    what = "MXFP4" if dtype == FP4 else "MXFP8"
    if glu:
        p = torch.rand(sum(LENS), device="cuda")
        plain = Q.glu_grouped_quantize_mx_impl(x, p, None, "silu", dtype, lens, offs, True, 0)
        words = Q.glu_grouped_quantize_mx_impl(x, p, None, "silu", dtype, lens, offs, True, Q._MX_WORDS)
    else:
        plain = Q._grouped_mx_quantize(x, dtype, lens, offs, True, True)
        words = Q.grouped_quantize_mx_operands(x, dtype, lens, offs, None, None, what)
        again = Q.grouped_quantize_mx_operands(x, dtype, lens, offs, None, None, what, known=words[4:])
        for a, b in zip(words[5:], again[5:]):
            assert torch.equal(a, b)
        for a, b in zip(words[:4], again[:4]):
            assert a.shape == b.shape and a.dtype == b.dtype
    cols = sum(-(-n // (256 if dtype == FP4 else 128)) for n in LENS) * (256 if dtype == FP4 else 128)
    starts = (plain[5] if dtype != FP4 else offs).tolist()
    rows = torch.cat([torch.arange(n, device="cuda") + s for n, s in zip(LENS, starts)])
    _same(plain[0].view(torch.uint8)[rows], words[0].view(torch.uint8)[rows])
    _same(plain[1].view(torch.uint8)[rows], _bytes(words[1])[rows])
    _same(plain[3].view(torch.uint8)[:, : cols // 32].contiguous(), _bytes(words[3])[:, : cols // 32].contiguous())


@pytest.mark.parametrize("cfg", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("M,N,K", [(21, 260, 640), (333, 520, 896), (1100, 1030, 1152)])
@pytest.mark.parametrize("dtype", [torch.float8_e4m3fn, FP4])
def test_dense_products(cfg, M, N, K, dtype):
    what = "MXFP4" if dtype == FP4 else "MXFP8"
    a, b = _x(M, K), _x(N, K)
    (qa, wa, _, _), (qb, wb, _, _) = (Q.quantize_mx_operands(t, dtype, None, None, what) for t in (a, b))
    sa, sb = _bytes(wa), _bytes(wb)
    outs = []
    D.TILE_CFG = cfg
    try:
        for s, t in ((sa, sb), (wa, wb), (wa, sb), (sa, wb)):
            outs.append(D.launch_mx(qa, s, qb, t, torch.empty(M, N, device="cuda", dtype=torch.float32), False, False))
    finally:
        D.TILE_CFG = 0
    for o in outs[1:]:
        assert torch.equal(o, outs[0])


@pytest.mark.parametrize("cfg", [0, 1, 3, 4])
@pytest.mark.parametrize("dtype", [torch.float8_e4m3fn, FP4])
def test_grouped_products(cfg, dtype):
    N, K, G = 262, 640, len(LENS)
    what = "MXFP4" if dtype == FP4 else "MXFP8"
    lens = torch.tensor(LENS, device="cuda")
    offs = torch.cat([lens.new_zeros(1), lens.cumsum(0)])
    qa, wa, qat, wat, _, offs_row, _, offs_col = Q.grouped_quantize_mx_operands(_x(sum(LENS), K), dtype, lens, offs, None, None, what)
    _, _, qgt, wgt, _, _, _, _ = Q.grouped_quantize_mx_operands(_x(sum(LENS), 288), dtype, lens, offs, None, None, what)
    qb, wb, _, _ = Q.quantize_mx_operands(_x(G, N, K), dtype, Recipe(use_2d_block=True), Recipe(use_2d_block=True), what)
    GG.MX_TILE_CFG = cfg
    try:
        outs = [GG._grouped_mx(qa, qb, s, t, offs_row, offs, False, True, torch.bfloat16)
                for s, t in ((_bytes(wa), _bytes(wb)), (wa, wb), (wa, _bytes(wb)), (_bytes(wa), wb))]
        if cfg != 4:
            grads = [GG._variable_k_mx(qgt, qat, s, t, offs_col, False, False, False,
                                       torch.empty(G, 288, K, device="cuda", dtype=torch.float32), False)
                     for s, t in ((_bytes(wgt), _bytes(wat)), (wgt, wat), (wgt, _bytes(wat)))]
    finally:
        GG.MX_TILE_CFG = 0
    for o in outs[1:]:
        assert torch.equal(o[: sum(LENS)], outs[0][: sum(LENS)])
    if cfg != 4:
        for g in grads[1:]:
            assert torch.equal(g, grads[0])
