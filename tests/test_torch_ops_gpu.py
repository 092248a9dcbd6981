"""The CUDA kernels of the dense operators in csrc/torch_ops.cpp against the operators' Python bodies (``<name>_general``): the same
bytes, shapes, strides and types for every form, and the same refusal where the body refuses."""

import pytest
import torch

from helpers import bf16_randn

pytestmark = pytest.mark.gpu

E4M3, E5M2, F4 = torch.float8_e4m3fn, torch.float8_e5m2, torch.float4_e2m1fn_x2
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.fixture(scope="module", autouse=True)
def _turbo(native_lib):
    global G, impl, Q
    from primus_turbo.pytorch.core.low_precision import ScalingGranularity as G
    from primus_turbo.pytorch.kernels.gemm import gemm_fp8_impl as impl
    from primus_turbo.pytorch.kernels.quantization import quantization_impl as Q


def _run(op, args):
    try:
        out = op(*args)
    except Exception as e:  # noqa: BLE001
        return str(e).split("\n")[0]
    return list(out) if isinstance(out, (list, tuple)) else [out]


def _same(namespace, name, *args):
    ops = getattr(torch.ops, namespace)
    got, want = _run(getattr(ops, name), args), _run(getattr(ops, name + "_general"), args)
    if isinstance(want, str) or isinstance(got, str):
        assert got == want
        return
    assert len(got) == len(want)
    for g, w in zip(got, want):
        assert (g.dtype, g.shape, g.stride(), g.device) == (w.dtype, w.shape, w.stride(), w.device)
        assert torch.equal(*(t.contiguous().flatten().view(torch.uint8) for t in (g, w)))


def _inputs(dtype):
    x = bf16_randn((97, 160), seed=1).cuda().to(dtype)
    return [x, x[:, :96].contiguous(), x[:1], x[:, :40], x.t(), x[:0], x[:, :0].contiguous(), x[0], x.reshape(97, 4, 40),
            x[:, 1:17].contiguous(), x.flatten()[1:97 * 32 + 1].view(97, 32), x.cpu()]


@pytest.mark.parametrize("to", [E4M3, E5M2, F4, BF16])
@pytest.mark.parametrize("dtype", [BF16, F16, F32, torch.float64])
def test_quantizers(dtype, to):
    ext, own = "primus_turbo_cpp_extension", "primus_turbo"
    one = torch.full((), 0.5, device="cuda")
    for x in _inputs(dtype):
        if not x.is_cuda:
            continue  # (refused by the operators' kernels for CPU tensors, which the general ones do not have)
        _same(ext, "quantize_fp8_tensorwise", x, to, None)
        _same(ext, "quantize_fp8_tensorwise", x, to, one)
        for axis in (-1, 0, 1, 2):
            if x.numel():  # (an empty reduction has no maximum)
                _same(ext, "quantize_fp8_rowwise", x, to, axis, None)
        if x.dim() != 2:
            continue
        R, C = x.shape
        for w, wt in ((C, R), (-(-C // 128) * 128, -(-R // 128) * 128), (C + 16, R)):
            _same(own, "quantize_fp8_tensorwise_t", x, to, w, wt)
        if x.numel():
            _same(own, "quant_fp8_rowwise_padded_impl", x, to, -(-C // 128) * 128)
            _same(own, "quant_fp8_rowwise_padded_impl", x, to, C - 1)
            _same(own, "quant_fp8_rowwise_t_impl", x, None, dtype, to, 128, None)
            _same(own, "quant_fp8_rowwise_t_impl", x, None, BF16, to, 24, None)
            for t in (False, True):
                _same(own, "quant_fp8_blockwise_kmajor_impl", x, to, 128, t)
            _same(own, "quant_fp8_blockwise_kmajor_impl", x, to, 64, True)
            for flags in ((8, 8), (9, 9), (0, 0), (8, 0), (8, 10)):
                _same(own, "quantize_mx", x, to, True, True, *flags)
            _same(own, "quantize_mx", x, to, True, False, 8, 0)


def test_quantizer_modes_and_codes():
    ext, own = "primus_turbo_cpp_extension", "primus_turbo"
    x = bf16_randn((97, 160), seed=1).cuda()
    for mode in ("fused", "two_pass", "auto"):
        before = Q.set_tensorwise_mode(mode)
        try:
            _same(ext, "quantize_fp8_tensorwise", x, E4M3, None)
            _same(own, "quantize_fp8_tensorwise_t", x, E4M3, 256, 128)
        finally:
            Q.set_tensorwise_mode(before)
    q, s = torch.ops.primus_turbo.quant_fp8_rowwise_padded_impl(x, E4M3, 256)
    for cols in (160, 33, None, 300):
        _same(own, "quant_fp8_rowwise_t_impl", q, s, BF16, E4M3, 128, cols)
    _same(own, "quant_fp8_rowwise_t_impl", q, s[:50], BF16, E4M3, 128, None)
    for hp in (BF16, F16, F32, E4M3):
        for scale in (s[:1, 0], s, s[:1].double()):
            _same(ext, "dequantize_fp8_tensorwise", q, scale, hp)
            _same(ext, "dequantize_fp8_tensorwise", q.t(), scale, hp)


@pytest.mark.parametrize("shape", [(1, 32), (97, 160), (128, 128), (130, 1024), (1, 33, 96), (3, 96, 160), (0, 64)])
@pytest.mark.parametrize("to", [E4M3, E5M2, F4])
def test_mx_directions(shape, to):
    """Each direction alone and both, scales of either layout, also batched."""
    x = bf16_randn(shape, seed=2).cuda()
    for row, col in ((True, False), (False, True), (True, True), (False, False)):
        for flags in ((0, 0), (8, 8), (1, 9), (0, 8), (2, 2)):
            _same("primus_turbo", "quantize_mx", x, to, row, col, *flags)
            _same("primus_turbo", "quantize_mx", x.half(), to, row, col, *flags)


@pytest.mark.parametrize("out_dtype", [BF16, F16, F32, torch.float64])
@pytest.mark.parametrize("trans_c", [False, True])
@pytest.mark.parametrize("M,N,K", [(16, 256, 512), (300, 520, 640), (1, 1, 128), (129, 128, 129), (5, 640, 640), (0, 64, 128), (1100, 1040, 1056)])
def test_products(M, N, K, trans_c, out_dtype):
    a, b = (bf16_randn((r, K), seed=i).cuda() for i, r in enumerate((M, N)))
    one, Kp = torch.full((), 0.5, device="cuda"), -(-K // 128) * 128

    def product(a, sa, ta, b, sb, tb, g):
        _same("primus_turbo", "gemm_fp8_impl", a, sa, ta, b, sb, tb, out_dtype, trans_c, g.value, 1)
        if M == 0 or out_dtype == torch.float64:
            return
        shape = (N, M) if trans_c else (M, N)
        outs = [torch.full(shape, 1.0, dtype=out_dtype, device="cuda") for _ in range(2)]
        impl.gemm_fp8_accum_impl(a, sa, ta, b, sb, tb, out_dtype, trans_c, g.value, outs[0], 1)
        impl._launch(a, sa, ta, b, sb, tb, outs[1], trans_c, g, True)
        assert torch.equal(*outs)

    qa, qb = a.to(E4M3), b.to(E5M2)
    product(qa, one, False, qb, one, True, G.TENSORWISE)
    product(qa.t().contiguous(), one, True, qb, one, True, G.TENSORWISE)
    product(qa, one, False, qb.t().contiguous(), one, False, G.TENSORWISE)
    ra, rb = torch.rand(M, 1, device="cuda"), torch.rand(N, 1, device="cuda")
    product(qa, ra, False, qb, rb, True, G.ROWWISE)
    product(qa, ra.flatten(), False, qb, torch.rand(N, 2, device="cuda")[:, :1], True, G.ROWWISE)
    kb = -(-K // 128)
    km, tiles = torch.rand(kb, M, device="cuda"), torch.rand(-(-N // 128), kb, device="cuda")
    product(qa, km.t(), False, qb, tiles, True, G.BLOCKWISE)
    product(qa, km.t().contiguous(), False, qb, tiles, True, G.BLOCKWISE)
    product(qa, km.t(), False, qb, tiles.t().contiguous().t(), True, G.BLOCKWISE)
    product(qa, km, False, qb, torch.rand(kb, N, device="cuda"), True, G.BLOCKWISE)
    tiles_t, bt = tiles.t().contiguous(), qb.t().contiguous()
    product(qa, km.t(), False, bt, tiles_t, False, G.BLOCKWISE)
    product(qa, km.t().contiguous(), False, bt, tiles_t, False, G.BLOCKWISE)
    _same("primus_turbo", "gemm_fp8_impl", qa, km.t(), False, bt, tiles, False, out_dtype, trans_c, G.BLOCKWISE.value, 1)  # (the wrong way round)
    if M and K % 32 == 0:
        wa, sa, _, _ = torch.ops.primus_turbo.quantize_mx(a, E4M3, True, True, 8, 8)
        wb, sb, _, _ = torch.ops.primus_turbo.quantize_mx(b, E4M3, True, True, 8, 8)
        product(wa, sa, False, wb, sb, True, G.MX_BLOCKWISE)
        wb, sb, _, _ = torch.ops.primus_turbo.quantize_mx(b, E4M3, True, True, 0, 0)
        product(wa, sa, False, wb, sb, True, G.MX_BLOCKWISE)
        fa, ga, _, _ = torch.ops.primus_turbo.quantize_mx(a, F4, True, True, 8, 8)
        fb, gb, _, _ = torch.ops.primus_turbo.quantize_mx(b, F4, True, True, 8, 8)
        product(fa, ga, False, fb, gb, True, G.MX_BLOCKWISE)
        for to in (E4M3, F4):  # row-major scales of both, which a user's own calls have
            ua, ta, _, _ = torch.ops.primus_turbo.quantize_mx(a, to, True, False, 0, 0)
            ub, tb, _, _ = torch.ops.primus_turbo.quantize_mx(b, to, True, False, 1, 0)
            product(ua, ta, False, ub, tb, True, G.MX_BLOCKWISE)


@pytest.mark.parametrize("bad", ["reduction", "scale shape", "scale type", "half operands", "3-D", "device"])
def test_refusals(bad):
    a, b = torch.zeros(32, 256, device="cuda").to(E4M3), torch.zeros(48, 256, device="cuda").to(E4M3)
    sa, sb = torch.ones(32, 1, device="cuda"), torch.ones(48, 1, device="cuda")
    if bad == "reduction":
        b = b[:, :128].contiguous()
    elif bad == "scale shape":
        sa = sa[:31]
    elif bad == "scale type":
        sb = sb.double()
    elif bad == "half operands":
        a = a.to(BF16)
    elif bad == "3-D":
        a = a[None]
    else:
        sb = sb.cpu()
    args = (a, sa, False, b, sb, True, BF16, False, G.ROWWISE.value, 1)
    assert isinstance(_run(torch.ops.primus_turbo.gemm_fp8_impl_general, args), str)
    _same("primus_turbo", "gemm_fp8_impl", *args)


# What the C library answers: every entry point returns `status` and counts the call, none launches anything.
_STUB = """
int status, calls;
const char *pt_last_error(void) { return "stub"; }
unsigned long pt_gemm_fp8_workspace_bytes(void) { return 0; }
unsigned long pt_gemm_mx_workspace_bytes(void) { return 0; }
unsigned long pt_quantize_fp8_rowwise_outer_workspace_bytes(void) { return 256; }
int pt_gemm_fp8_vec_in_place(void) { return 0; }
int pt_gemm_fp8_nn_in_place(void) { return 0; }
""" + "".join(f"int {n}(void) {{ ++calls; return status; }}\n" for n in (
    "pt_gemm_fp8", "pt_gemm_mx", "pt_quantize_fp8_tensorwise_static", "pt_quantize_fp8_tensorwise_t", "pt_dequantize_fp8_tensorwise",
    "pt_quantize_fp8_rowwise", "pt_quantize_fp8_rowwise_padded", "pt_quantize_fp8_rowwise_outer_ld",
    "pt_quantize_fp8_blockwise_kmajor", "pt_quantize_mx"))


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    import ctypes
    import subprocess

    d = tmp_path_factory.mktemp("stub")
    (d / "stub.c").write_text(_STUB)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(d / "stub.so"), str(d / "stub.c")], check=True)
    return ctypes.CDLL(str(d / "stub.so")), str(d / "stub.so")


@pytest.mark.parametrize("status", ["LAUNCH", "INVALID_ARGUMENT", "UNSUPPORTED", "WORKSPACE"])
def test_status_of_the_library(stub, status):
    """A call that the library refuses goes to the Python body. One whose launch failed raises and is not issued again:
    the error may be one that an earlier call left, found after a kernel that did run, and an accumulating product would
    add twice."""
    import ctypes

    from primus_turbo import _native as N

    x = bf16_randn((64, 256), seed=1).cuda()
    q, one = x.to(E4M3), torch.full((), 0.5, device="cuda")
    qt, s, qmx, smx = *torch.ops.primus_turbo.quant_fp8_rowwise_padded_impl(x, E4M3, 256), *torch.ops.primus_turbo.quantize_mx(x, E4M3, True, False, 8, 8)[:2]
    own, ext = torch.ops.primus_turbo, torch.ops.primus_turbo_cpp_extension
    product = (q, one, False, q, one, True)
    km, tiles, bt = torch.rand(2, 64, device="cuda"), torch.rand(1, 2, device="cuda"), q.t().contiguous()
    out = torch.zeros(64, 64, device="cuda")
    calls = {
        "gemm": lambda: own.gemm_fp8_impl(*product, F32, False, G.TENSORWISE.value, 1),
        "gemm mx": lambda: own.gemm_fp8_impl(qmx, smx, False, qmx, smx, True, F32, False, G.MX_BLOCKWISE.value, 1),
        "gemm block": lambda: own.gemm_fp8_impl(q, km.t(), False, q, tiles, True, F32, False, G.BLOCKWISE.value, 1),
        "gemm block, b [K, N]": lambda: own.gemm_fp8_impl(q, km.t(), False, bt, tiles.t().contiguous(), False, F32, False, G.BLOCKWISE.value, 1),
        "accumulating": lambda: own.gemm_fp8_accum_impl(*product, F32, False, G.TENSORWISE.value, out, 1),
        "accumulating mx": lambda: own.gemm_fp8_accum_impl(qmx, smx, False, qmx, smx, True, F32, False, G.MX_BLOCKWISE.value, out, 1),
        "tensorwise": lambda: ext.quantize_fp8_tensorwise(x, E4M3, None),
        "tensorwise t": lambda: own.quantize_fp8_tensorwise_t(x, E4M3, 256, 128),
        "dequantize": lambda: ext.dequantize_fp8_tensorwise(q, one, BF16),
        "rowwise": lambda: ext.quantize_fp8_rowwise(x, E4M3, -1, None),
        "rowwise padded": lambda: own.quant_fp8_rowwise_padded_impl(x, E4M3, 384),
        "rowwise t": lambda: own.quant_fp8_rowwise_t_impl(qt, s, BF16, E4M3, 128, None),
        "kmajor": lambda: own.quant_fp8_blockwise_kmajor_impl(x, E4M3, 128, True),
        "mx": lambda: own.quantize_mx(x, E4M3, True, True, 8, 8),
    }
    lib, path = stub
    code, counter = ctypes.c_int.in_dll(lib, "status"), ctypes.c_int.in_dll(lib, "calls")

    def results(call):
        out.zero_()
        r = call()
        r = out.clone() if r is None else r
        return [t.contiguous().flatten().view(torch.uint8) for t in (r if isinstance(r, (list, tuple)) else [r])]

    code.value, want = getattr(N, "PT_ERR_" + status), {name: results(call) for name, call in calls.items()}
    own._bind_native(path)
    try:
        for name, call in calls.items():
            counter.value = 0
            if status == "LAUNCH":
                with pytest.raises(RuntimeError, match="native error -4: stub"):
                    results(call)
                assert not out.any(), name  # (a second launch would have been the real library's)
            else:
                assert all(torch.equal(g, w) for g, w in zip(results(call), want[name])), name
            assert counter.value == 1, name
    finally:
        own._bind_native(str(N.LIB_PATH))
