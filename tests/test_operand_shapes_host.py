"""Operands whose reduction lengths differ are refused before the casts pad them to a common length."""

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
