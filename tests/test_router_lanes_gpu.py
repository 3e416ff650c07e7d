"""The router's 16- and 8-lane forms at the edges of their stripe counts and
of the token counts that choose between them and the wave form: weights bit for
bit, selections equal up to exact ties, with tied, masked (-inf) and NaN rows."""

from __future__ import annotations

import pytest
import torch

from custom_cuda_kernals_amd.kernels import moe_router
from oracle import inputs, moe
from tests.test_moe_router_gpu import _check

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("e", [17, 32, 33, 48, 49, 64, 65, 96, 97, 129, 161, 192, 193, 255, 256])
def test_stripe_edges(e, dtype):
    for t, k in ((1, 1), (5, min(e, 17)), (67, 8), (2047, 2), (2048, 6)):
        logits = inputs.router_inputs(t, e, dtype, seed=t + e)
        logits[::3] = torch.round(logits[::3])  # many exact ties
        logits[1::5, : e // 2] = float("-inf")
        _check(logits, min(k, e), k != 8)


@pytest.mark.parametrize("e,t", [(32, 8191), (32, 8192), (64, 16383), (64, 16384), (17, 8193), (40, 16390)])
def test_token_count_edges(e, t):
    _check(inputs.router_inputs(t, e, torch.bfloat16, seed=t), 6, True)


@pytest.mark.parametrize("e", [12, 20, 64, 200])
def test_nan_rows_keep_their_neighbours(e):
    logits = inputs.router_inputs(9, e, torch.float32, seed=e)
    logits[4, e // 2] = float("nan")
    w, i = moe_router(logits.cuda(), 4)
    ref, _ = moe.moe_router_avx512(logits, 4, True)
    keep = torch.arange(9) != 4
    assert torch.equal(w.cpu()[keep].view(torch.int32), ref[keep].view(torch.int32))
    assert bool(torch.isnan(w.cpu()[4]).all())
