"""Registration of the operators that launch the native library's kernels."""

from __future__ import annotations

from typing import Callable, Optional

import torch

_lib = torch.library.Library("primus_turbo", "FRAGMENT")


def native_op(qualname: str, device_types: Optional[str] = None) -> Callable:
    """``torch.library.custom_op(qualname, mutates_args=(), device_types=...)`` for functions that allocate
    their results, launch on the current stream and return: the same operator for tracing (schema from the
    annotations, ``register_fake`` on the returned function) without the wrappers that ``custom_op`` runs around
    the body on every call -- an autograd kernel written in Python, a check of the results' storages, a guard
    against being traced into. They cost 5 to 8 us a call (a 16 x 512 x 512 product 18.9 -> 14.1 us of host time),
    and a training step makes nine calls. None of them has anything to do here: gradients come from the autograd
    functions around these operators, results are fresh tensors, and a tracer sees the operator through its
    fake. Operators that write into an argument stay with ``custom_op``, which advances that tensor's version."""
    namespace, name = qualname.split("::")
    assert namespace == "primus_turbo"

    def wrap(fn: Callable) -> Callable:
        _lib.define(name + torch.library.infer_schema(fn, mutates_args=()), tags=(torch.Tag.pt2_compliant_tag,))
        _lib.impl(name, fn, "CUDA" if device_types == "cuda" else "CompositeExplicitAutograd")
        op = getattr(torch.ops.primus_turbo, name).default

        def call(*args, **kwargs):
            return op(*args, **kwargs)

        call.__name__, call.__doc__, call.__module__ = fn.__name__, fn.__doc__, fn.__module__
        call.register_fake = lambda fake: torch.library.register_fake(qualname, fake, lib=_lib)
        return call

    return wrap
