"""Operands that the layers refuse before their casts run: reduction lengths that differ (the casts pad them to a common
length), expert counts away from the GPU (the rows' cast of serving does not read them)."""

import pytest
import torch

import primus_turbo.pytorch as turbo
from primus_turbo.pytorch.core.low_precision import Float8QuantConfig
from primus_turbo.pytorch.core.low_precision import ScalingGranularity as G


@pytest.fixture(autouse=True)
def _no_hardware_check(native_lib, monkeypatch):
    import primus_turbo.pytorch.core.low_precision as LP

    monkeypatch.setattr(LP, "_needs", lambda *a: (True, ""))


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("granularity", [G.TENSORWISE, G.ROWWISE])
@pytest.mark.parametrize("k_a, k_b", [(112, 128), (128, 112), (112, 96), (96, 112), (240, 256), (272, 384), (256, 512)])
def test_reduction_lengths_that_differ_are_refused(granularity, k_a, k_b, train):
    a = torch.empty(64, k_a, device="meta", dtype=torch.bfloat16).requires_grad_(train)
    b = torch.empty(48, k_b, device="meta", dtype=torch.bfloat16).requires_grad_(train)
    with pytest.raises(AssertionError, match=f"reduction dims differ: {k_a} vs {k_b}"):
        turbo.ops.gemm_fp8(a, b, trans_b=True, config=Float8QuantConfig(granularity=granularity))


@pytest.mark.parametrize("away", ["group_lens", "group_offs"])
def test_serving_refuses_group_counts_on_another_device(away):
    a = torch.empty(64, 256, device="meta", dtype=torch.bfloat16)
    b = torch.empty(2, 384, 256, device="meta", dtype=torch.bfloat16)
    where = lambda name: "cpu" if name == away else "meta"  # noqa: E731
    lens = torch.full((2,), 32, dtype=torch.int64, device=where("group_lens"))
    offs = torch.zeros(3, dtype=torch.int64, device=where("group_offs"))
    with pytest.raises(RuntimeError, match="on the device of a"):
        turbo.ops.grouped_gemm_fp8(a, b, lens, offs, trans_b=True, config=Float8QuantConfig(granularity=G.BLOCKWISE, block_size=128))
