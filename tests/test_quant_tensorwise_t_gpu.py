"""The tensorwise cast that emits the codes transposed as well: the same bytes as the cast and a transposition, at
the edges of its 128 x 128 tiles, beyond what its registers hold, with padded rows, and where it takes the steps one
by one; the rowwise casts with padded rows beside it."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pad", [False, True])
@pytest.mark.parametrize("R,C", [(1, 16), (130, 144), (3001, 1056), (16, 16), (16, 2048), (128, 128), (144, 272), (1040, 112), (4096, 4096), (8208, 4112), (40, 64), (64, 40)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("fp8", [torch.float8_e4m3fn, torch.float8_e5m2])
def test_same_bytes_as_two_steps(native_lib, R, C, dtype, fp8, pad):
    from primus_turbo.pytorch.kernels.quantization import quantization_impl as impl

    x = torch.randn(R, C, generator=torch.Generator(device="cuda").manual_seed(R + C), device="cuda", dtype=dtype)
    x[R // 2, C // 3] = 37.0  # the maximum, in one place
    q, scale_inv = impl._quantize_fp8_tensorwise(x, fp8)
    for mode in ("auto", "two_pass"):
        before = impl.set_tensorwise_mode(mode)
        try:
            got, got_t, got_scale = impl.quantize_fp8_tensorwise_t_impl(x, fp8, *((-(-n // 128) * 128 if pad else n) for n in (C, R)))
        finally:
            impl.set_tensorwise_mode(before)
        assert torch.equal(got_scale, scale_inv)
        assert torch.equal(got.view(torch.uint8)[:, :C], q.view(torch.uint8)) and not got.view(torch.uint8)[:, C:].any()
        assert torch.equal(got_t.view(torch.uint8)[:, :R], q.view(torch.uint8).t()) and not got_t.view(torch.uint8)[:, R:].any()


@pytest.mark.parametrize("M,N", [(1, 32), (33, 200), (5, 256), (257, 2880), (40, 9000)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rowwise_rows_are_padded(native_lib, M, N, dtype):
    from primus_turbo.pytorch.kernels.quantization import quantization_impl as impl

    x = torch.randn(M, N, generator=torch.Generator(device="cuda").manual_seed(M + N), device="cuda", dtype=dtype)
    q, s = impl._quantize_fp8_rowwise(x, torch.float8_e4m3fn, 1)
    width = -(-N // 128) * 128
    got, got_s = impl.quant_fp8_rowwise_padded_impl(x, torch.float8_e4m3fn, width)
    assert torch.equal(got.view(torch.uint8)[:, :N], q.view(torch.uint8)) and not got.view(torch.uint8)[:, N:].any()
    assert torch.equal(got_s, s)
    for codes, cols in ((q, None), (got, N)):  # quantized again along the other axis, from either
        t, ts = impl.quant_fp8_rowwise_t_impl(codes, s, dtype, torch.float8_e4m3fn, 128, cols)
        if cols is None:
            want, want_s = t, ts
    assert torch.equal(t.view(torch.uint8), want.view(torch.uint8)) and torch.equal(ts, want_s)


def test_one_launch_needs_an_aligned_tensor(native_lib):
    from primus_turbo.pytorch.kernels.quantization import quantization_impl as impl

    x = torch.randn(64 * 64 + 1, device="cuda", dtype=torch.bfloat16)[1:].view(64, 64)
    q, q_t, _ = impl.quantize_fp8_tensorwise_t_impl(x, torch.float8_e4m3fn, 64, 64)
    assert torch.equal(q.view(torch.uint8), impl._quantize_fp8_tensorwise(x, torch.float8_e4m3fn)[0].view(torch.uint8))
    assert torch.equal(q_t.view(torch.uint8), q.view(torch.uint8).t())


# 0, an infinity and a NaN, in one tile or alone, with rows and columns that are padded
@pytest.mark.parametrize("R,C", [(144, 272), (3001, 1056)])
@pytest.mark.parametrize("values", [(), (float("inf"),), (float("nan"),), (float("-inf"), float("nan"))])
@pytest.mark.parametrize("zeros", [False, True])
@pytest.mark.parametrize("fp8", [torch.float8_e4m3fn, torch.float8_e5m2])
def test_special_values(native_lib, R, C, values, zeros, fp8):
    from primus_turbo.pytorch.kernels.quantization import quantization_impl as impl

    x = torch.randn(R, C, generator=torch.Generator(device="cuda").manual_seed(R), device="cuda", dtype=torch.bfloat16) * (not zeros)
    for i, v in enumerate(values):
        x[R - 1 - i, C - 1 - i] = v
    u8 = lambda t: t.view(torch.uint8)  # noqa: E731
    q, scale_inv = impl._quantize_fp8_tensorwise(x, fp8)
    got, got_t, got_scale = impl.quantize_fp8_tensorwise_t_impl(x, fp8, *(-(-n // 128) * 128 for n in (C, R)))
    assert torch.equal(got_scale.view(torch.int32), scale_inv.view(torch.int32))
    assert torch.equal(u8(got)[:, :C], u8(q)) and not u8(got)[:, C:].any()
    assert torch.equal(u8(got_t)[:, :R], u8(q).t()) and not u8(got_t)[:, R:].any()
    q, s = impl._quantize_fp8_rowwise(x[:, : C - 8].contiguous(), fp8, 1)
    got, got_s = impl.quant_fp8_rowwise_padded_impl(x[:, : C - 8].contiguous(), fp8, -(-C // 128) * 128)
    assert torch.equal(got_s.view(torch.int32), s.view(torch.int32))
    assert torch.equal(u8(got)[:, : C - 8], u8(q)) and not u8(got)[:, C - 8 :].any()
