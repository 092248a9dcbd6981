"""Block-scaled products that read a weight stored [K, N] where it lies (256 x 256 tile, transposed reads from the LDS): the bits
of the product of the transposed copy, at the edges of the tile and of the matrix, and the same gradients of the layers."""

import numpy as np
import pytest
import torch

from helpers import bf16_randn

pytestmark = pytest.mark.gpu
E4M3, E5M2 = torch.float8_e4m3fn, torch.float8_e5m2


@pytest.fixture(scope="module", autouse=True)
def _turbo(native_lib):
    global turbo, G, impl, gimpl, Q, LP
    import primus_turbo.pytorch as turbo
    from primus_turbo.pytorch.core import low_precision as LP
    from primus_turbo.pytorch.core.low_precision import ScalingGranularity as G
    from primus_turbo.pytorch.kernels.gemm import gemm_fp8_impl as impl
    from primus_turbo.pytorch.kernels.grouped_gemm import grouped_gemm_fp8_impl as gimpl
    from primus_turbo.pytorch.kernels.quantization import quantization_impl as Q


def _operands(M, N, K, da=E4M3, db=E4M3, lead=()):
    x, w = bf16_randn((M, K), seed=1).cuda(), bf16_randn((*lead, K, N), seed=2).cuda()
    a, sa, _, _ = Q.quant_fp8_blockwise_kmajor_impl(x, da, 128, False)
    b, sb = Q.quant_fp8_blockwise_for_weight_impl(w, db, 128)
    return a, sa, b, sb


def _dense(a, sa, b, sb, out, accumulate=False):
    """(read in place, on the transposed copy)"""
    outs = [out.clone(), out.clone()]
    impl._launch(a, sa, False, b, sb, False, outs[0], False, G.BLOCKWISE, accumulate)
    impl._launch(a, sa, False, b.t().contiguous(), sb.t().contiguous(), True, outs[1], False, G.BLOCKWISE, accumulate)
    return outs


@pytest.fixture
def pinned():
    impl.TILE_CFG = 4
    yield
    impl.TILE_CFG = 0


# one tile; columns that end inside a tile, a fragment's and a copy's width before its end; rows of less than a tile
@pytest.mark.parametrize("N", [16, 112, 128, 240, 256, 272, 528, 1008])
@pytest.mark.parametrize("M,K", [(256, 512), (300, 640), (1, 1152)])
def test_edges(M, N, K, pinned):
    a, sa, b, sb = _operands(M, N, K)
    got, want = _dense(a, sa.t(), b, sb, torch.zeros(M, N, dtype=torch.bfloat16, device="cuda"))
    assert torch.equal(got, want)


@pytest.mark.parametrize("da", [E4M3, E5M2])
@pytest.mark.parametrize("db", [E4M3, E5M2])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("accumulate", [False, True])
def test_forms(da, db, out_dtype, accumulate, pinned):
    a, sa, b, sb = _operands(520, 784, 1024, da, db)
    old = torch.randn(520, 784, device="cuda").to(out_dtype)
    for scales in (sa.t(), sa.t().contiguous()):  # block-major, row-major
        got, want = _dense(a, scales, b, sb, old, accumulate)
        assert torch.equal(got, want)


def test_special_values_stay_in_their_column(pinned):
    a, sa, b, sb = _operands(300, 528, 640)
    b.view(torch.uint8)[639, 5] = 0x7F
    b.view(torch.uint8)[0, 527] = 0x7F
    got, want = _dense(a, sa.t(), b, sb, torch.zeros(300, 528, dtype=torch.float32, device="cuda"))
    assert torch.equal(got.nan_to_num(nan=7e9), want.nan_to_num(nan=7e9))
    assert got.isnan().any(0).nonzero().flatten().tolist() == [5, 527]


# reductions and widths that the tile does not read in place take the copy
@pytest.mark.parametrize("M,N,K", [(300, 520, 640), (300, 528, 600), (300, 528, 384), (4096, 4096, 512), (8192, 4080, 1024)])
def test_rule(M, N, K):
    a, sa, b, sb = _operands(M, N, K)
    assert impl.reads_kn_in_place(M, N, K) == (M > 300)
    got, want = _dense(a, sa.t(), b, sb, torch.zeros(M, N, dtype=torch.bfloat16, device="cuda"))
    assert torch.equal(got, want)


@pytest.mark.parametrize("lens", [[256, 0, 255, 1, 257], [700, 513, 0, 300]])
@pytest.mark.parametrize("N", [256, 400, 2064])
@pytest.mark.parametrize("da", [E4M3, E5M2])
@pytest.mark.parametrize("tile", [0, 4])
def test_grouped(lens, N, da, tile):
    M, K = sum(lens), 640
    a, sa, b, sb = _operands(M + 70, N, K, da, E4M3, (len(lens),))  # (rows behind the last group read as zero)
    gl = torch.from_numpy(np.array(lens, dtype=np.int64)).cuda()
    offs = torch.ops.primus_turbo_cpp_extension.grouped_gemm_compute_offs(gl)
    outs = []
    for w, s, tb in ((b, sb, False), (b.transpose(1, 2).contiguous(), sb.transpose(1, 2).contiguous(), True)):
        gimpl.TILE_CFG = tile
        try:
            outs.append(gimpl.grouped_gemm_fp8_impl(a, w, sa, s, gl, offs, False, tb, torch.bfloat16, G.BLOCKWISE.value, None, 0))
        finally:
            gimpl.TILE_CFG = 0
    assert torch.equal(*outs)
    assert not outs[0][M:].any()


@pytest.mark.parametrize("hybrid", [False, True])
@pytest.mark.parametrize("grouped", [False, True])
def test_layer_gradients(grouped, hybrid, monkeypatch):
    import importlib

    ops = importlib.import_module("primus_turbo.pytorch.ops." + ("grouped_gemm_fp8" if grouped else "gemm_fp8"))
    config = LP.Float8QuantConfig(granularity=G.BLOCKWISE, block_size=128, format=LP.Format.HYBRID if hybrid else LP.Format.E4M3)
    lens = torch.tensor([1500, 0, 700, 1896], device="cuda")
    k = 2064 if grouped else 4080
    x = bf16_randn((4096, k), seed=1).cuda().requires_grad_()
    w = bf16_randn((4, 2176, k) if grouped else (4224, k), seed=2).cuda().requires_grad_()
    g = bf16_randn((4096, w.shape[-2]), seed=3).cuda()
    used, grads = [], []
    for on in (True, False):
        real = (gimpl if grouped else impl).reads_kn_in_place
        monkeypatch.setattr(ops, "reads_kn_in_place", lambda *a: used.append(real(*a)) or (on and used[-1]))
        out = ops.grouped_gemm_fp8(x, w, lens, trans_b=True, config=config) if grouped else ops.gemm_fp8(x, w, trans_b=True, config=config)
        grads.append((out, *torch.autograd.grad(out, (x, w), g)))
    assert used == [True, True]
    assert all(torch.equal(p, q) for p, q in zip(*grads))


def _mx_weight(G_, n, k, fmt=E4M3, special=True):
    w = bf16_randn((G_, n, k), seed=4).cuda() * torch.rand(G_, n // 32, k // 32, device="cuda").exp2().repeat_interleave(32, 1).repeat_interleave(32, 2)
    w = w.to(torch.bfloat16)
    if special:
        w[0, :32, :64], w[-1, n - 1, k - 1], w[0, 40, 3] = 0, float("nan"), float("inf")
    return w


@pytest.mark.parametrize("shape", [(1, 128, 128), (3, 256, 640), (2, 1152, 384)])
@pytest.mark.parametrize("fmt", [E4M3, E5M2])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_mx_weight_quantizer(shape, fmt, dtype):
    """The codes of both directions are each other's transposition, and the scales those of the two-direction quantizer."""
    w, recipe = _mx_weight(*shape).to(dtype), LP.ScalingRecipe(use_2d_block=True)
    q, words, words_t = Q.quantize_mx_weight_impl(w, fmt)
    rq, rs, cq, cs = Q.quantize_mx_operands(w, fmt, recipe, recipe, "MXFP8")
    u8 = lambda t: t.contiguous().view(torch.uint8)  # noqa: E731
    assert torch.equal(u8(q), u8(rq)) and torch.equal(u8(q.transpose(1, 2)), u8(cq))
    assert torch.equal(words, rs) and torch.equal(words_t, cs)


# rows of less than a tile, of a whole one, one over; columns that end inside a tile; both tiles (128 x 128 and 256 x 256)
@pytest.mark.parametrize("lens", [[128, 0, 127, 1, 129], [700, 513, 0, 460], [33, 95, 256]])
@pytest.mark.parametrize("n,k", [(128, 512), (1152, 640), (1408, 768)])
@pytest.mark.parametrize("da", [E4M3, E5M2])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_mx_grouped(lens, n, k, da, out_dtype):
    """grad [rows, k] x weight [G, k, n] as it lies against the product on the transposed quantization."""
    w, recipe = _mx_weight(len(lens), k, n, special=False), LP.ScalingRecipe(use_2d_block=True)
    x = bf16_randn((sum(lens), k), seed=5).cuda()
    gl = torch.from_numpy(np.array(lens, dtype=np.int64)).cuda()
    offs = torch.ops.primus_turbo_cpp_extension.grouped_gemm_compute_offs(gl)
    xq, xs, _, _, _, orow, _, _ = Q.grouped_quantize_mx_operands(x, da, gl, offs, None, None, "MXFP8")
    q, _, words_t = Q.quantize_mx_weight_impl(w, E4M3)
    _, _, cq, cs = Q.quantize_mx_operands(w, E4M3, recipe, recipe, "MXFP8")
    got = gimpl.grouped_gemm_mx_kn_impl(xq, q, xs, words_t, orow, offs, out_dtype)
    want = gimpl.grouped_gemm_fp8_impl(xq, cq, xs, cs, gl, orow, False, True, out_dtype, G.MX_BLOCKWISE.value, None, 0, False, offs)
    assert torch.equal(got, want)


@pytest.mark.parametrize("hybrid", [False, True])
@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("n,k", [(640, 384), (512, 416)])  # (the second: blocks of 32, not of 128)
def test_mx_layer_gradients(glu, hybrid, n, k, monkeypatch):
    import importlib

    ops = importlib.import_module("primus_turbo.pytorch.ops.grouped_gemm_fp8")
    config = LP.Float8QuantConfig(granularity=G.MX_BLOCKWISE, block_size=32, scale_dtype=LP.ScaleDtype.E8M0,
                                  format=LP.Format.HYBRID if hybrid else LP.Format.E4M3)
    lens = torch.tensor([300, 0, 213, 87], device="cuda")
    x = bf16_randn((600, 2 * k if glu else k), seed=1).cuda().requires_grad_()
    w = bf16_randn((4, n, k), seed=2).cuda().requires_grad_()
    p = torch.rand(600, device="cuda").requires_grad_()
    g = bf16_randn((600, n), seed=3).cuda()
    used, grads = [], []
    for on in (True, False):
        monkeypatch.setattr(ops, "mx_reads_kn", lambda *a: used.append(gimpl.mx_reads_kn(*a)) or (on and used[-1]))
        out = (ops.glu_grouped_gemm_fp8(x, p, w, lens, trans_b=True, config=config, act_type="silu") if glu else
               ops.grouped_gemm_fp8(x, w, lens, trans_b=True, config=config))
        grads.append((out, *torch.autograd.grad(out, (x, w, p) if glu else (x, w), g)))
    assert used == ([True, True] if k % 128 == 0 else [])
    assert all(torch.equal(a, b) for a, b in zip(*grads))


@pytest.mark.parametrize("M,N,K", [(256, 256, 512), (272, 528, 640), (16, 1008, 1152), (528, 112, 768)])
@pytest.mark.parametrize("trans_a,trans_c", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("granularity", ["TENSORWISE", "ROWWISE"])
@pytest.mark.parametrize("out_dtype,accumulate", [(torch.bfloat16, False), (torch.float16, True), (torch.float32, False), (torch.float32, True)])
def test_vector_scales(M, N, K, trans_a, trans_c, granularity, out_dtype, accumulate, pinned):
    a, b = bf16_randn((M, K), seed=1).cuda().to(E4M3), bf16_randn((N, K), seed=2).cuda().to(E5M2)
    one = torch.full((), 0.5, device="cuda")
    sa, sb = (torch.rand(M, 1, device="cuda"), torch.rand(N, 1, device="cuda")) if granularity == "ROWWISE" else (one, one)
    old = torch.randn((N, M) if trans_c else (M, N), device="cuda").to(out_dtype)
    got, want = old.clone(), old.clone()
    impl._launch(a.t().contiguous() if trans_a else a, sa, trans_a, b.t().contiguous(), sb, False, got, trans_c, G[granularity], accumulate)
    impl._launch(a, sa, False, b, sb, True, want, trans_c, G[granularity], accumulate)
    assert torch.equal(got, want)


@pytest.mark.parametrize("da", [E4M3, E5M2])
@pytest.mark.parametrize("db", [E4M3, E5M2])
def test_vector_scales_by_the_rule(da, db):
    """Taken at a whole round of 256 x 256 tiles; in the operator as in its Python body."""
    a, b = bf16_randn((4096, 1024), seed=1).cuda().to(da), bf16_randn((4096, 1024), seed=2).cuda().to(db)
    one = torch.full((), 0.5, device="cuda")
    assert impl.vec_reads_in_place(4096, 4096, 1024, True) and impl.vec_reads_in_place(4096, 4096, 1024, False)
    args = (torch.bfloat16, False, G.TENSORWISE.value, 1)
    want = impl.gemm_fp8_impl(a, one, False, b, one, True, *args)
    bt = b.t().contiguous()
    for op in (impl.gemm_fp8_impl, torch.ops.primus_turbo.gemm_fp8_impl_general):
        assert torch.equal(op(a, one, False, bt, one, False, *args), want)
        assert torch.equal(op(a.t().contiguous(), one, True, bt, one, False, *args), want)


@pytest.mark.parametrize("hybrid", [False, True])
@pytest.mark.parametrize("main_grad", [False, True])
@pytest.mark.parametrize("M,N,K", [(4096, 4096, 4096), (4096, 4096, 4080)])  # (the second: rows that are no whole slabs)
def test_tensorwise_layer_gradients(M, N, K, main_grad, hybrid, monkeypatch):
    import importlib

    ops = importlib.import_module("primus_turbo.pytorch.ops.gemm_fp8")
    config = LP.Float8QuantConfig(format=LP.Format.HYBRID if hybrid else LP.Format.E4M3)
    x, g = bf16_randn((M, K), seed=1).cuda().requires_grad_(), bf16_randn((M, N), seed=3).cuda()
    used, grads = [], []
    for on in (True, False):
        monkeypatch.setattr(ops, "vec_reads_in_place", lambda *a: used.append(impl.vec_reads_in_place(*a)) or (on and used[-1]))
        w = torch.nn.Parameter(bf16_randn((N, K), seed=2).cuda())
        if main_grad:
            w.main_grad, w.grad_added_to_main_grad = torch.full(w.shape, 0.25, device="cuda"), False
        out = ops.gemm_fp8(x, w, trans_b=True, config=config, fuse_bgrad_accum_pattern="megatron" if main_grad else None)
        gx, gw = torch.autograd.grad(out, (x, w), g)
        grads.append((out, gx, w.main_grad if main_grad else gw))
    assert used == ([True, True, True] if K % 128 == 0 else [])  # (the patched rule is asked once, and says no)
    assert all(torch.equal(a, b) for a, b in zip(*grads))


F4 = torch.float4_e2m1fn_x2


def _nibbles(q):
    """Codes of ``[.., rows, cols / 2]`` packed bytes, one a byte."""
    u = q.contiguous().view(torch.uint8)
    return torch.stack((u & 15, u >> 4), -1).flatten(-2)


@pytest.mark.parametrize("shape", [(1, 128, 128), (3, 256, 640), (2, 1152, 384)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_mxfp4_weight_quantizer(shape, dtype):
    w, recipe = _mx_weight(*shape).to(dtype), LP.ScalingRecipe(use_2d_block=True)
    q, words, words_t = Q.quantize_mx_weight_impl(w, F4)
    rq, rs, cq, cs = Q.quantize_mx_operands(w, F4, recipe, recipe, "MXFP4")
    assert torch.equal(_nibbles(q), _nibbles(rq)) and torch.equal(_nibbles(q).transpose(1, 2), _nibbles(cq))
    assert torch.equal(words, rs) and torch.equal(words_t, cs)


@pytest.mark.parametrize("lens", [[128, 0, 127, 1, 129], [900, 513, 0, 460], [33, 95, 256]])
@pytest.mark.parametrize("n,k", [(128, 1024), (1152, 1280), (1408, 1536)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_mxfp4_grouped(lens, n, k, out_dtype):
    from primus_turbo.pytorch.kernels.grouped_gemm import grouped_gemm_fp4_impl as gimpl4

    w, recipe = _mx_weight(len(lens), k, n, special=False), LP.ScalingRecipe(use_2d_block=True)
    x = bf16_randn((sum(lens), k), seed=5).cuda()
    gl = torch.from_numpy(np.array(lens, dtype=np.int64)).cuda()
    offs = torch.ops.primus_turbo_cpp_extension.grouped_gemm_compute_offs(gl)
    xq, xs, _, _, _, orow, _, _ = Q.grouped_quantize_mx_operands(x, F4, gl, offs, LP.ScalingRecipe(), LP.ScalingRecipe(), "MXFP4")
    q, _, words_t = Q.quantize_mx_weight_impl(w, F4)
    _, _, cq, cs = Q.quantize_mx_operands(w, F4, recipe, recipe, "MXFP4")
    got = gimpl.grouped_gemm_mx_kn_impl(xq, q, xs, words_t, orow, offs, out_dtype)
    want = gimpl4.grouped_gemm_fp4_impl(xq, cq, xs, cs, gl, orow, False, True, out_dtype, G.MX_BLOCKWISE.value, None, 0, False, offs)
    assert torch.equal(got, want)


@pytest.mark.parametrize("glu", [False, True])
# (the second: an odd number of half slabs; the third: blocks of 32, not of 128)
@pytest.mark.parametrize("n,k", [(1280, 384), (1152, 384), (1280, 416)])
def test_mxfp4_layer_gradients(glu, n, k, monkeypatch):
    import importlib

    ops = importlib.import_module("primus_turbo.pytorch.ops.grouped_gemm_fp4")
    config, lens = LP.Float4QuantConfig(), torch.tensor([300, 0, 213, 87], device="cuda")
    x = bf16_randn((600, 2 * k if glu else k), seed=1).cuda().requires_grad_()
    w = bf16_randn((4, n, k), seed=2).cuda().requires_grad_()
    p = torch.rand(600, device="cuda").requires_grad_()
    g = bf16_randn((600, n), seed=3).cuda()
    used, grads = [], []
    monkeypatch.setattr(Q, "_next_sr_seed", lambda *flags: 12345)
    for on in (True, False):
        monkeypatch.setattr(ops, "mx_reads_kn", lambda *a: used.append(gimpl.mx_reads_kn(*a)) or (on and used[-1]))
        out = (ops.glu_grouped_gemm_fp4(x, p, w, lens, trans_b=True, config=config, act_type="silu") if glu else
               ops.grouped_gemm_fp4(x, w, lens, trans_b=True, config=config))
        grads.append((out, *torch.autograd.grad(out, (x, w, p) if glu else (x, w), g)))
    assert used == ([n % 256 == 0] * 2 if k % 128 == 0 else [])
    assert all(torch.equal(a, b) for a, b in zip(*grads))


# both sides of the line at which a bank's weight gets its transposed copy again: the same bits, and the copy's path where it pays
@pytest.mark.parametrize("recipe,rows", [("MX_BLOCKWISE", 2 * 5120 - 1), ("MX_BLOCKWISE", 2 * 5120), ("BLOCKWISE", 2 * 8192 - 1), ("BLOCKWISE", 2 * 8192)])
def test_rows_a_weight(recipe, rows, monkeypatch):
    import importlib

    ops = importlib.import_module("primus_turbo.pytorch.ops.grouped_gemm_fp8")
    mx = recipe == "MX_BLOCKWISE"
    more = dict(block_size=32, scale_dtype=LP.ScaleDtype.E8M0) if mx else dict(block_size=128)
    config = LP.Float8QuantConfig(granularity=G[recipe], **more)
    lens = torch.tensor([700, rows - 700], device="cuda")
    x, g = bf16_randn((rows, 2048), seed=1).cuda().requires_grad_(), bf16_randn((rows, 512), seed=3).cuda()
    w = bf16_randn((2, 512, 2048), seed=2).cuda().requires_grad_()
    name = "quantize_mx_weight_impl" if mx else "quant_fp8_blockwise_for_weight_impl"
    calls, real, pays = [], getattr(ops, name), ops.kn_layer_pays
    monkeypatch.setattr(ops, name, lambda *a, **kw: calls.append(1) or real(*a, **kw))
    grads = []
    for on in (True, False):
        monkeypatch.setattr(ops, "kn_layer_pays", lambda *a: on and pays(*a))
        out = ops.grouped_gemm_fp8(x, w, lens, trans_b=True, config=config)
        grads.append((out, *torch.autograd.grad(out, (x, w), g)))
    assert len(calls) == (rows // 2 < (5120 if mx else 8192))
    assert all(torch.equal(a, b) for a, b in zip(*grads))
