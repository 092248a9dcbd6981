"""Operators registered by ``native_op`` without a GPU: what autograd, tracing and transforms see of them."""

import pytest
import torch

import primus_turbo.pytorch as turbo
from primus_turbo.pytorch.core import native_op as no
from primus_turbo.pytorch.core.low_precision import ScalingGranularity as G

NO_FORMULA = "no autograd formula was registered"
HP = torch.bfloat16


def _meta(*shape, dtype=HP, grad=True):
    return torch.empty(shape, device="meta", dtype=dtype).requires_grad_(grad)


def _codes(*shape):
    return torch.empty(shape, device="meta", dtype=turbo.float8_e4m3)


def _bytes(*shape):
    return torch.empty(shape, device="meta", dtype=torch.uint8)


def _public_calls():
    """name -> () -> (the tensor that asks for a gradient, a floating-point output of the call)"""
    from primus_turbo.pytorch.kernels.quantization import quantization_impl as Q

    f8, x = turbo.float8_e4m3, lambda: _meta(256, 512)

    def of(make, fn):
        def run():
            t = make()
            out = fn(t)
            return t, out[0] if isinstance(out, (tuple, list)) else out

        return run

    scale = lambda *shape: (lambda: _meta(*shape, dtype=torch.float32))  # noqa: E731
    return {
        "quantize blockwise": of(x, lambda t: turbo.ops.quantize_fp8(t, f8, G.BLOCKWISE, block_size=128, axis=1)),
        "quantize blockwise, both directions": of(
            x, lambda t: turbo.ops.quantize_fp8_with_trans(t, f8, G.BLOCKWISE, block_size=128)),
        "quantize blockwise weight": of(x, lambda t: Q.quant_fp8_blockwise_for_weight_impl(t, f8, 128)),
        "quantize MXFP8": of(x, lambda t: turbo.ops.quantize_fp8(t, f8, G.MX_BLOCKWISE, block_size=32, axis=1)),
        "quantize MXFP8, both directions": of(
            x, lambda t: turbo.ops.quantize_fp8_with_trans(t, f8, G.MX_BLOCKWISE, block_size=32)),
        "dequantize blockwise": of(scale(256, 4), lambda s: turbo.ops.dequantize_fp8(
            _codes(256, 512), HP, G.BLOCKWISE, block_size=128, axis=1, scale_inv=s)),
        "quantize rowwise, transposed": of(x, lambda t: Q.quant_fp8_rowwise_t_impl(t, None, HP, f8, 128)),
        "quantize tensorwise, transposed": of(x, lambda t: Q.quantize_fp8_tensorwise_t_impl(t, f8, 512, 256)),
    }


@pytest.mark.parametrize("name", sorted(_public_calls()))
def test_backward_raises_instead_of_losing_a_path(name):
    t, out = _public_calls()[name]()
    assert out.requires_grad
    with pytest.raises(RuntimeError, match=NO_FORMULA):
        (out.float().sum() + t.float().sum()).backward()
    with torch.no_grad():
        assert not _public_calls()[name]()[1].requires_grad


def _dummy(name):
    @no.native_op(f"primus_turbo::{name}")
    def fill(x: torch.Tensor, value: int, other: torch.Tensor) -> torch.Tensor:
        return torch.empty_like(x).fill_(value)

    @fill.register_fake
    def _fake(x, value, other):
        return torch.empty_like(x)

    return fill


_fill = _dummy("host_test_fill")


@pytest.fixture(params=["call", "operator"])
def fill(request, monkeypatch):
    """The returned function and the operator behind it, on CPU tensors."""
    monkeypatch.setattr(no, "_AUTOGRAD", torch._C.DispatchKey.AutogradCPU)
    return _fill if request.param == "call" else torch.ops.primus_turbo.host_test_fill


def test_autograd_of_a_native_op(fill):
    x, y = torch.ones(3, requires_grad=True), torch.ones(3)
    out = fill(x, 2, y)
    assert out.requires_grad and torch.equal(out.detach(), torch.full((3,), 2.0))
    with pytest.raises(RuntimeError, match=NO_FORMULA):
        (out + x).sum().backward()
    for wanted in ((lambda: fill(y, 2, x)), (lambda: fill(x=x, value=2, other=y)), (lambda: fill(y, value=2, other=x))):
        with pytest.raises(RuntimeError, match=NO_FORMULA):
            wanted().sum().backward()
    assert not fill(y, 2, y).requires_grad
    with torch.no_grad():
        assert not fill(x, 2, x).requires_grad
    with torch.inference_mode():
        assert fill(y, 2, y).is_inference()
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: fill(t, 2, y).sum())(y)
    # the state that a call sets is gone after it, also after one that failed
    with pytest.raises(Exception):
        fill(y, "two", y)
    assert (y.clone().requires_grad_(True) * 2).requires_grad


def test_native_op_within_an_autograd_function(fill):
    class Layer(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return fill(x, 2, x)

        @staticmethod
        def backward(ctx, g):
            return fill(g, 3, g)

    for run in (Layer.apply, torch.compile(Layer.apply, backend="aot_eager", fullgraph=True)):
        x = torch.ones(3, requires_grad=True)
        run(x).sum().backward()
        assert torch.equal(x.grad, torch.full((3,), 3.0))


def test_native_op_traced_and_batched(fill):
    x = torch.ones(2, 3)
    assert torch.equal(torch.compile(lambda t: fill(t, 2, t) + 1, backend="aot_eager", fullgraph=True)(x), x + 2)
    assert torch.vmap(lambda t: fill(t, 2, t))(x).shape == (2, 3)
    from torch._subclasses import FakeTensorMode

    with FakeTensorMode():
        assert fill(torch.ones(3), 2, torch.ones(3)).shape == (3,)


@pytest.mark.parametrize("pinned", [0, 3])
def test_product_with_a_pinned_tile(pinned, monkeypatch):
    """The operator behind ``gemm_fp8_impl`` while a tile is pinned is traced and refuses a backward pass as the other."""
    from primus_turbo.pytorch.kernels.gemm import gemm_fp8_impl as impl

    monkeypatch.setattr(impl, "TILE_CFG", pinned)
    scale = _meta(1, dtype=torch.float32)
    args = (_codes(48, 256), scale, False, _codes(32, 256), _meta(1, dtype=torch.float32, grad=False), True, HP, True, G.TENSORWISE.value, 1)
    out = impl.gemm_fp8_impl(*args)
    assert out.shape == (32, 48) and out.dtype == HP
    with pytest.raises(RuntimeError, match=NO_FORMULA):
        (out.float().sum() + scale.sum()).backward()
    torch._dynamo.reset()
    with torch.no_grad():
        assert torch.compile(impl.gemm_fp8_impl, backend="aot_eager", fullgraph=True)(*args).shape == (32, 48)
