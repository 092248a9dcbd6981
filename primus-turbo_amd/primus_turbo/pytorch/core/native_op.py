"""Registration of the operators that launch the native library's kernels."""

from __future__ import annotations

from typing import Callable, Optional

import torch

from primus_turbo import _native

if _native.TORCH_LIB_PATH.exists():
    _native.load_torch_ops()

_lib = torch.library.Library("primus_turbo", "FRAGMENT")
_below_autograd = torch._C._AutoDispatchBelowAutograd
_is_compiling = torch.compiler.is_compiling
# The same for CUDA tensors by hand: 0.9 us a call instead of 1.4, the context manager's own construction being most of it
_AUTOGRAD = torch._C.DispatchKey.AutogradCUDA
_is_excluded, _set_excluded = torch._C._dispatch_tls_is_dispatch_key_excluded, torch._C._dispatch_tls_set_dispatch_key_excluded


class _NoBackward(torch.autograd.Function):
    """An operator's results for a caller that wants gradients: they come out as parts of the graph, and a
    backward pass that reaches them raises instead of leaving this path out of the sum."""

    @staticmethod
    def forward(ctx, qualname, op, kwargs, *args):
        ctx.qualname = qualname
        with _below_autograd():
            return op(*args, **kwargs)

    @staticmethod
    def backward(ctx, *grads):
        raise RuntimeError(f"Trying to backward through {ctx.qualname} but no autograd formula was registered: "
                           "use the layers of primus_turbo.pytorch.ops, which have one")


def _wants_gradient(args, kwargs) -> bool:
    return torch.is_grad_enabled() and torch._C._any_requires_grad(*args, **kwargs)


def _autograd_kernel(name: str) -> Callable:
    op, qualname = getattr(torch.ops.primus_turbo, name).default, f"primus_turbo::{name}"

    def kernel(*args, **kwargs):
        if _wants_gradient(args, kwargs):
            return _NoBackward.apply(qualname, op, kwargs, *args)
        with _below_autograd():
            return op(*args, **kwargs)

    return kernel


def native_op(qualname: str, device_types: Optional[str] = None, cpp: bool = False) -> Callable:
    """``torch.library.custom_op(qualname, mutates_args=(), device_types=...)`` for functions that allocate
    their results, launch on the current stream and return: the same operator for tracing (schema from the
    annotations, ``register_fake`` on the returned function) and for autograd (a backward pass through it raises),
    without the wrappers that ``custom_op`` runs around the body on every call -- an autograd kernel written in
    Python, a check of the results' storages, a guard against being traced into. They cost 5 to 8 us a call (a 16 x
    512 x 512 product 18.9 -> 14.1 us of host time), and a training step makes nine calls. The layers' autograd
    functions call these operators with gradients off: the returned function sees that and steps over the
    autograd kernel (0.9 us), which everything else that reaches the operator passes through. Results are fresh tensors,
    and a tracer sees the operator through its fake. Operators that write into an argument stay with ``custom_op``,
    which advances that tensor's version.

    ``cpp``: the operator's CUDA kernel is in csrc/torch_ops.cpp; the function is the body for every other
    device and, as the operator ``<name>_general`` (with the same fake and the same autograd), for the forms which that kernel does
    not handle itself."""
    namespace, name = qualname.split("::")
    assert namespace == "primus_turbo"

    def wrap(fn: Callable) -> Callable:
        schema, key = torch.library.infer_schema(fn, mutates_args=()), "CUDA" if device_types == "cuda" else "CompositeExplicitAutograd"
        names = [name, name + "_general"] if cpp else [name]
        for n in names:
            _lib.define(n + schema, tags=(torch.Tag.pt2_compliant_tag,))
            if not cpp or n != name or key != "CUDA":
                _lib.impl(n, fn, key)
            _lib.impl(n, _autograd_kernel(n), "Autograd")
        op = getattr(torch.ops.primus_turbo, name).default

        def call(*args, **kwargs):
            if _is_compiling() or _wants_gradient(args, kwargs) or _is_excluded(_AUTOGRAD):
                return op(*args, **kwargs)
            _set_excluded(_AUTOGRAD, True)
            try:
                return op(*args, **kwargs)
            finally:
                _set_excluded(_AUTOGRAD, False)

        call.__name__, call.__doc__, call.__module__ = fn.__name__, fn.__doc__, fn.__module__
        call.register_fake = lambda fake: [torch.library.register_fake(f"{namespace}::{n}", fake, lib=_lib) for n in names]
        return call

    return wrap
