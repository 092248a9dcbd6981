"""GPU parity of rowwise quantization along a non-contiguous axis vs the CPU oracle (bit-exact): codes in
place, codes transposed, and FP8 codes quantized again along their other axis."""

import numpy as np
import pytest
import torch

from helpers import FMT, bf16_randn, bits_np, codes_np, round_to, to_f32_np
from oracle import quantize as Q

pytestmark = pytest.mark.gpu

# edges of the 512-column strips, of the 128 x 128 tiles and of the eight-row runs; columns that are no
# multiple of eight take the one-column lanes
SHAPES = [(1, 8), (7, 8), (33, 9), (128, 128), (129, 136), (257, 520), (1000, 516), (3001, 264), (3, 65, 72), (2, 5, 130, 16)]
# a wavefront over several rows, with whole and with idle lanes, and with more rows than one round of a
# workgroup; rows for more than 64 chunks, whose maxima meet by atomics
SPLITS = [(300, 1), (300, 3), (4099, 16), (700, 24), (1000, 40), (70, 33, 24), (25000, 264), (66000, 33)]


@pytest.mark.parametrize("shape", SHAPES + SPLITS)
@pytest.mark.parametrize("src,dtype", [(torch.bfloat16, torch.float8_e4m3fn), (torch.float16, torch.float8_e5m2),
                                       (torch.float32, torch.float8_e4m3fn)])
def test_outer_axis(native_lib, shape, src, dtype):
    from primus_turbo.pytorch.kernels.quantization import quantization_impl as I

    x = bf16_randn(shape, seed=21, outlier_frac=0.01, dtype=src)
    axis = len(shape) - 2
    oq, osinv = Q.fp8_rowwise(to_f32_np(x), axis, FMT[dtype])
    q, sinv = I.quantize_fp8_rowwise_impl(x.cuda(), dtype, axis)
    assert np.array_equal(bits_np(sinv), osinv.view(np.uint32)) and np.array_equal(codes_np(q), oq)
    qt, sinv = I.quant_fp8_rowwise_t_impl(x.cuda(), None, src, dtype, 128)
    M = shape[-2]
    assert tuple(qt.shape) == (*shape[:-2], shape[-1], -(-M // 128) * 128)
    got = codes_np(qt)
    assert np.array_equal(bits_np(sinv), osinv.view(np.uint32))
    assert np.array_equal(got[..., :M], np.swapaxes(oq, -1, -2)) and not got[..., M:].any()


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("src,dtype", [(torch.bfloat16, torch.float8_e4m3fn), (torch.float16, torch.float8_e5m2),
                                       (torch.float32, torch.float8_e4m3fn)])
def test_codes_quantized_again(native_lib, shape, src, dtype):
    from primus_turbo.pytorch.kernels.quantization import quantization_impl as I

    x = bf16_randn(shape, seed=22, outlier_frac=0.01, dtype=src)
    q1, s1 = Q.fp8_rowwise(to_f32_np(x), len(shape) - 1, FMT[dtype])
    hp = round_to(Q.fp8_dequant(q1, s1, FMT[dtype]), src)
    oq, osinv = Q.fp8_rowwise(to_f32_np(hp), len(shape) - 2, FMT[dtype])
    codes = torch.from_numpy(q1).view(dtype).cuda()
    qt, sinv = I.quant_fp8_rowwise_t_impl(codes, torch.from_numpy(s1).cuda(), src, dtype, 16)
    M = shape[-2]
    got = codes_np(qt)
    assert np.array_equal(bits_np(sinv), osinv.view(np.uint32))
    assert np.array_equal(got[..., :M], np.swapaxes(oq, -1, -2)) and not got[..., M:].any()


@pytest.mark.parametrize("shape", SPLITS)
@pytest.mark.parametrize("src,dtype", [(torch.bfloat16, torch.float8_e4m3fn), (torch.float16, torch.float8_e5m2),
                                       (torch.float32, torch.float8_e4m3fn)])
def test_codes_quantized_again_is_three_steps(native_lib, shape, src, dtype):
    """The same bits as de-quantize, quantize, transpose. (Against those launches and not the oracle's rounding:
    over ten million fp16 elements a dozen de-quantized values differ from it in their last bit, the GPU
    rounding code times scale once where the oracle rounds to fp32 and then to fp16.)"""
    from primus_turbo.pytorch.kernels.quantization import quantization_impl as I

    nd, M = len(shape), shape[-2]
    codes, s1 = I.quantize_fp8_rowwise_impl(bf16_randn(shape, seed=22, outlier_frac=0.01, dtype=src).cuda(), dtype, nd - 1)
    want, sinv = I.quantize_fp8_rowwise_impl(I.dequantize_fp8_rowwise_impl(codes, src, nd - 1, s1), dtype, nd - 2)
    qt, sinv_t = I.quant_fp8_rowwise_t_impl(codes, s1, src, dtype, 16)
    qt = qt.view(torch.uint8)
    assert torch.equal(sinv_t, sinv) and torch.equal(qt[..., :M], want.view(torch.uint8).transpose(-1, -2))
    assert not qt[..., M:].any()


@pytest.mark.parametrize("shape", SHAPES + SPLITS)
@pytest.mark.parametrize("src,dtype", [(torch.bfloat16, torch.float8_e4m3fn), (torch.float16, torch.float8_e5m2),
                                       (torch.float32, torch.float8_e4m3fn)])
@pytest.mark.parametrize("scales", ["dynamic", "given", "given in place"])
def test_entry_without_workspace(native_lib, shape, src, dtype, scales):
    """pt_quantize_fp8_rowwise: scales from the columns' maxima, which meet in scale_inv's storage, or given by
    the caller in a buffer of their own or in scale_inv's."""
    from primus_turbo import _native as N

    x = bf16_randn(shape, seed=23, outlier_frac=0.01, dtype=src)
    axis = len(shape) - 2
    B, M, n = int(np.prod(shape[:-2])), shape[-2], shape[-1]
    scale = torch.rand(*shape[:-2], 1, n, generator=torch.Generator().manual_seed(5)) * 60 + 0.5
    oq, osinv = Q.fp8_rowwise(to_f32_np(x), axis, FMT[dtype], scale=None if scales == "dynamic" else scale.numpy())
    xd, sinv = x.cuda(), scale.cuda()
    given = {"dynamic": None, "given": sinv.clone(), "given in place": sinv if n > 1 else sinv.clone()}[scales]
    q = torch.empty(shape, dtype=dtype, device="cuda")
    N.check(native_lib.pt_quantize_fp8_rowwise(N.ptr(xd), N.dtype_code(xd.dtype), B, M, n, N.ptr(q), N.dtype_code(q.dtype),
                                               N.ptr(given), N.ptr(sinv), N.stream_of(xd)))
    assert np.array_equal(bits_np(sinv), osinv.view(np.uint32)) and np.array_equal(codes_np(q), oq)


def test_more_rows_than_a_grid_has_blocks_along_y(native_lib):
    """128 rows for each of 65535 blocks and a few more: the scales are the columns' maxima, the codes those of
    the same rows under given scales, and the transposed codes the same codes."""
    from primus_turbo.pytorch.kernels.quantization import quantization_impl as I

    M, n = 128 * 65535 + 200, 8
    x = torch.randn(M, n, generator=torch.Generator(device="cuda").manual_seed(7), device="cuda", dtype=torch.bfloat16)
    amax = to_f32_np(x.abs().amax(0, keepdim=True))
    _, osinv = Q.fp8_rowwise(amax, 0, "e4m3")
    scale = torch.from_numpy(np.float32(448) / amax).cuda()
    q, sinv = I.quantize_fp8_rowwise_impl(x, torch.float8_e4m3fn, 0)
    assert np.array_equal(bits_np(sinv), osinv.view(np.uint32))
    for m in (0, M // 2, M - 1000):
        part, _ = torch.ops.primus_turbo_cpp_extension.quantize_fp8_rowwise(x[m : m + 1000].contiguous(), torch.float8_e4m3fn, 0, scale)
        assert torch.equal(q[m : m + 1000].view(torch.uint8), part.view(torch.uint8))
    qt, sinv_t = I.quant_fp8_rowwise_t_impl(x, None, x.dtype, torch.float8_e4m3fn, 128)
    assert torch.equal(sinv_t, sinv) and torch.equal(qt[:, :M].view(torch.uint8), q.view(torch.uint8).t())
    assert not qt[:, M:].view(torch.uint8).any()
