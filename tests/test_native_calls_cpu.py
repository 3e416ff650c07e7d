"""The one-call form of the Python API (native *_call functions) takes only
ordinary calls: anything else returns None, so that the long way raises its
errors or sees its modes."""

from __future__ import annotations

import pytest
import torch

from custom_cuda_kernals_amd import kernels
from custom_cuda_kernals_amd._lib import native

X = torch.zeros(4, 16)
IDS = torch.zeros(4, 2, dtype=torch.int64)
CALLS = {
    "rmsnorm_residual_call": (X, X, X[0], 1e-6),
    "rmsnorm_residual_fp8_call": (X, X, X[0], 1e-6, "e4m3", None),
    "swiglu_call": (X, X),
    "swiglu_fp8_call": (X, X, "e4m3", None),
    "rope_call": (X.view(1, 2, 2, 16), X.view(1, 2, 2, 16), X[:2, :8].contiguous(), X[:2, :8].contiguous(), False),
    "fp8_quant_call": (X, "e4m3", "token", None),
    "token_gather_call": (X, IDS[:, 0].contiguous()),
    "token_combine_call": (X, IDS, X[:, :2].contiguous()),
    "compute_permutation_call": (IDS, 8),
    "moe_router_call": (X, 2, True),
}


@pytest.mark.parametrize("name", CALLS)
def test_other_arguments_return_none(name):
    call, args = getattr(native, name), CALLS[name]
    assert call(*args) is None  # CPU tensors
    assert call() is None and call(*args, None) is None
    for i in range(len(args)):
        for other in (None, object(), 3, 2.5, "e4m3", 1 << 80, [1], X.numpy()):
            assert call(*args[:i], other, *args[i + 1:]) is None


def test_the_long_way_raises():
    for call in (lambda: kernels.rmsnorm_residual(X, X, X[0]), lambda: kernels.swiglu_fp8(X, X),
                 lambda: kernels.fp8_quant(X), lambda: kernels.moe_router(X, 2),
                 lambda: kernels.compute_permutation(IDS, 8)):
        with pytest.raises(ValueError, match="must be a CUDA tensor, got device type 'cpu'"):
            call()
