"""Ragged rows whose workgroups take more than one: every row against the oracle,
where the register-resident ragged kernels refill their registers after the partial
vector was moved in place, alternate their reduction buffers, and loop on grids of
the workgroups the device holds at once; and rows with NaN and infinities."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from custom_cuda_kernals_amd import _native as native
from oracle import eager, inputs
from oracle import fp8 as ofp8
from tests._parity import assert_codes_equal, assert_f32_bits_equal, bits_equal, codes_np
from tests._routes import kernels_of

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32
F8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
CAP = 65536  # workgroups of a row kernel's grid at most


def _norm(rows, cols, dtype, static):
    """Plain (static is False), per-token (None) or static-scale; every row."""
    x, r, w = inputs.rmsnorm_inputs(rows, cols, dtype, seed=rows + cols)
    d = [t.cuda() for t in (x, r, w)]
    ro = torch.empty_like(d[0])
    if static is False:
        y = torch.empty_like(d[0])
        native.rmsnorm_residual_fwd(*d, y, ro, 1e-5)
        y_ref, ro_ref = eager.rmsnorm_residual(x, r, w, 1e-5)
        assert bits_equal(y, y_ref).all()
    else:
        q = torch.empty(rows, cols, dtype=F8["e4m3"], device="cuda")
        s = torch.empty(rows, device="cuda") if static is None else None
        native.rmsnorm_residual_fp8_fwd(*d, q, s, ro, 1e-5, "e4m3", static)
        codes, s_ref, ro_ref, _ = eager.rmsnorm_residual_fp8(x, r, w, 1e-5, "e4m3", static)
        assert_codes_equal(q, codes)
        if static is None:
            assert_f32_bits_equal(s, s_ref)
    assert bits_equal(ro, ro_ref).all()


@pytest.mark.parametrize("rows,cols,dtype,static", [
    (1200, 12283, BF16, None), (900, 24571, BF16, None), (900, 24571, BF16, 0.05), (900, 8190, F32, None),
    (900, 12281, F32, 0.05), (CAP + 37, 9, BF16, False), (CAP + 37, 13, BF16, None), (CAP + 37, 17, F16, 0.05),
    (CAP + 37, 7, F32, False), (CAP + 37, 5, F32, None)])
def test_rmsnorm(rows, cols, dtype, static):
    _norm(rows, cols, dtype, static)


@pytest.mark.parametrize("cols,dtype", [(9, BF16), (33, F16), (5, F32)])
def test_fp8_token(cols, dtype):
    x = inputs.randn((CAP + 37, cols), dtype, seed=cols)
    xd, s = x.cuda(), torch.empty(CAP + 37, device="cuda")
    q = torch.empty(x.shape, dtype=F8["e4m3"], device="cuda")
    native.fp8_quant_token_fwd(xd, q, s, "e4m3")
    codes, s_ref = ofp8.quant_token(x.float().numpy(), "e4m3")
    assert_codes_equal(q, codes)
    assert_f32_bits_equal(s, s_ref)


@pytest.mark.parametrize("cols,dtype", [(9, BF16), (17, F16), (5, F32)])
def test_swiglu_fp8(cols, dtype):
    g, u = inputs.swiglu_inputs(CAP + 37, cols, dtype, seed=cols)
    q, s = torch.empty(g.shape, dtype=F8["e5m2"], device="cuda"), torch.empty(CAP + 37, device="cuda")
    native.swiglu_fp8_fwd(g.cuda(), u.cuda(), q, s, "e5m2", None)
    codes, s_ref, _ = eager.swiglu_fp8(g, u, "e5m2", None)
    assert_codes_equal(q, codes)
    assert_f32_bits_equal(s, s_ref)


def test_gather():
    """More destination rows than one grid of the ragged and of the sliced form
    takes at once (four a workgroup)."""
    for h, kernel in ((129, "token_gather_slicesILb1E"), (1024, "token_gather_slicesILb0E")):
        src = inputs.randn((3000, h), BF16, seed=h)
        idx = torch.randint(-1, 3001, (4 * CAP + 7,), generator=torch.Generator().manual_seed(h))
        sd, idx_d = src.cuda(), idx.cuda()
        dst = torch.empty(4 * CAP + 7, h, dtype=BF16, device="cuda")
        (name, _), = kernels_of(lambda: native.token_gather_fwd(sd, idx_d, dst))
        assert kernel in name
        ok = (idx_d >= 0) & (idx_d < 3000)
        ref = torch.where(ok[:, None], sd[torch.where(ok, idx_d, 0)], 0.0)
        assert torch.equal(dst.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("hq,hkv,d,kernel", [(2, 1, 128, "RopePolicyE1E"), (2, 1, 48, "RopePolicyE2E"),
                                             (2, 2, 64, "RopePolicyE1E")])
def test_rope(hq, hkv, d, kernel):
    """More tokens than workgroups, on chip (8 and 4 chunks) and split (3)."""
    q, k, cos, sin = inputs.rope_inputs(1, CAP + 37, hq, hkv, d, dtype=BF16, seed=d, theta=10000.0)
    t = [v.cuda() for v in (q, k, cos, sin)]
    qo, ko = torch.empty_like(t[0]), torch.empty_like(t[1])
    (name, _), = kernels_of(lambda: native.rope_fwd(*t, qo, ko))
    assert "rope_heads" in name and kernel in name, name
    q_ref, k_ref = eager.rope(q, k, cos, sin)
    assert bits_equal(qo, q_ref).all() and bits_equal(ko, k_ref).all()


NAN, INF = float("nan"), float("inf")
# Every class of row: NaN and infinities in whole vectors, in the partial one, in
# the element before it (loaded with it and dropped), zeros, and plain rows between.
SPECIALS = [(1, 0, NAN), (2, 3, INF), (3, -1, NAN), (4, -1, -INF), (5, -9, NAN), (6, -2, INF)]


def _special(rows, cols, dtype, seed):
    x = inputs.randn((rows, cols), dtype, seed=seed)
    for row, col, value in SPECIALS:
        x[row, col] = value
    x[7] = 0.0
    return x


def _codes_or_nan(q, codes, fmt):
    """Codes equal; where the oracle has a NaN, any NaN code."""
    got = codes_np(q).reshape(codes.shape)
    is_nan = (lambda c: (c & 0x7F) == 0x7F) if fmt == "e4m3" else (lambda c: (c & 0x7F) > 0x7C)
    assert np.array_equal(is_nan(got), is_nan(codes))
    assert np.array_equal(got[~is_nan(codes)], codes[~is_nan(codes)])


@pytest.mark.parametrize("dtype", [BF16, F16, F32], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
@pytest.mark.parametrize("cols", [1003, 4099])
def test_nan_and_inf_rows(cols, fmt, dtype):
    x = _special(9, cols, dtype, cols)
    q, s = torch.empty(x.shape, dtype=F8[fmt], device="cuda"), torch.empty(9, device="cuda")
    native.fp8_quant_token_fwd(x.cuda(), q, s, fmt)
    codes, s_ref = ofp8.quant_token(x.float().numpy(), fmt)
    _codes_or_nan(q, codes, fmt)
    assert_f32_bits_equal(s, s_ref)

    g, u = _special(9, cols, dtype, cols + 1), inputs.randn((9, cols), dtype, seed=cols + 2)
    native.swiglu_fp8_fwd(g.cuda(), u.cuda(), q, s, fmt, None)
    codes, s_ref, _ = eager.swiglu_fp8(g, u, fmt, None)
    _codes_or_nan(q, codes, fmt)
    assert_f32_bits_equal(s, s_ref)


@pytest.mark.parametrize("dtype", [BF16, F16, F32], ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
def test_nan_and_inf_tiles(fmt, dtype):
    """Block scales: special values in the partial vector's tile must not reach
    the tile on its left, whose elements it loads, nor the other way round."""
    for n in (257, 261, 384 + 3):
        for col, value in ((n - 1, NAN), (255, NAN), (n - 1, INF), (255, -INF), (0, NAN)):
            x = inputs.randn((130, n), dtype, seed=n)
            x[5, col] = value
            q = torch.empty(x.shape, dtype=F8[fmt], device="cuda")
            s = torch.empty(2, (n + 127) // 128, device="cuda")
            native.fp8_quant_block_fwd(x.cuda(), q, s, fmt)
            codes, s_ref = ofp8.quant_block(x.float().numpy(), fmt)
            _codes_or_nan(q, codes, fmt)
            assert_f32_bits_equal(s, s_ref)
