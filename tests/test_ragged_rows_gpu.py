"""Rows whose length is no multiple of a 16-byte vector, or whose buffers start
off a 16-byte boundary, through the register-resident row kernels: bit for bit
against the oracle at the edges of the row shapes (one vector, one element
either side of a shape's capacity, the widest shapes and past them), with the
memory around every output untouched.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from custom_cuda_kernals_amd import _native as native
from oracle import eager, inputs, moe
from oracle import fp8 as ofp8
from tests._parity import assert_codes_equal, assert_f32_bits_equal, bits_equal

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]
F8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
# Row capacities of the shapes, in vectors; a row is one element short of one,
# or one element longer, so its last vector is partial on either side.
CAPACITIES = [1, 64, 128, 256, 320, 384, 512, 768, 1024, 1536, 2048, 3072, 4096]


class Guarded:
    """A device tensor `offset` elements into a buffer whose other bytes must
    keep a pattern."""

    def __init__(self, shape, dtype, offset: int) -> None:
        n = int(np.prod(shape))
        self.flat = torch.full(((n + offset + 64) * dtype.itemsize,), 0xA5, dtype=torch.uint8, device="cuda")
        self.lo, self.hi = offset * dtype.itemsize, (n + offset) * dtype.itemsize
        self.t = self.flat[self.lo:self.hi].view(dtype).view(shape)

    def check(self) -> None:
        rest = torch.cat([self.flat[:self.lo], self.flat[self.hi:]])
        assert bool((rest == 0xA5).all()), "written outside the output"


def _off(t: torch.Tensor, offset: int) -> torch.Tensor:
    view = torch.empty(t.numel() + offset, dtype=t.dtype, device="cuda")[offset:].view(t.shape)
    view.copy_(t.cuda())
    return view


def _lengths(vec: int) -> list[int]:
    return [c * vec + d for c in CAPACITIES for d in (-1, 1) if c * vec + d >= 1]


def _check_norm(x, r, w, static, offset=0):
    """Plain (static is False), per-token (None) or static-scale RMSNorm."""
    ro = Guarded(x.shape, x.dtype, offset)
    xd, rd, wd = _off(x, offset), _off(r, offset), _off(w, offset)
    if static is False:
        y = Guarded(x.shape, x.dtype, offset)
        native.rmsnorm_residual_fwd(xd, rd, wd, y.t, ro.t, 1e-5)
        y_ref, ro_ref = eager.rmsnorm_residual(x, r, w, 1e-5)
        assert bits_equal(y.t, y_ref).all()
        y.check()
    else:
        q = Guarded(x.shape, F8["e4m3"], offset)
        s = torch.empty(x.shape[0], dtype=torch.float32, device="cuda") if static is None else None
        native.rmsnorm_residual_fp8_fwd(xd, rd, wd, q.t, s, ro.t, 1e-5, "e4m3", static)
        codes, s_ref, ro_ref, _ = eager.rmsnorm_residual_fp8(x, r, w, 1e-5, "e4m3", static)
        assert_codes_equal(q.t, codes)
        if static is None:
            assert_f32_bits_equal(s, s_ref)
        q.check()
    assert bits_equal(ro.t, ro_ref).all()
    ro.check()


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("static", [False, None, 0.05], ids=["plain", "token", "static"])
def test_rmsnorm(dtype, static):
    vec = 16 // dtype.itemsize
    for cols in _lengths(vec):
        x, r, w = inputs.rmsnorm_inputs(5, cols, dtype, seed=cols)
        _check_norm(x, r, w, static, offset=cols % 3)
    # Whole vectors from an unaligned start, and every remainder after whole vectors.
    for cols in [256 * vec, *range(600 * vec, 601 * vec)]:
        x, r, w = inputs.rmsnorm_inputs(3, cols, dtype, seed=cols + 1)
        _check_norm(x, r, w, static, offset=1)


def test_rmsnorm_absent_elements_stay_out_of_the_amax():
    """Rows whose variance underflows at eps = 0: 1 / sqrt(0) is infinite, so
    present elements give infinities (a zero element NaN) and an infinite
    scale; the partial vector's absent elements must not add a NaN."""
    x = torch.full((3, 1003), 1e-30, dtype=torch.float32).to(torch.bfloat16)
    x[1, 5] = 0.0
    x[2] = 1.0
    r, w = torch.zeros_like(x), torch.ones(1003, dtype=torch.bfloat16)
    q = torch.empty(x.shape, dtype=F8["e4m3"], device="cuda")
    s = torch.empty(3, dtype=torch.float32, device="cuda")
    native.rmsnorm_residual_fp8_fwd(x.cuda(), r.cuda(), w.cuda(), q, s, torch.empty_like(x, device="cuda"), 0.0,
                                    "e4m3", None)
    codes, s_ref, _, _ = eager.rmsnorm_residual_fp8(x, r, w, 0.0, "e4m3", None)
    assert_f32_bits_equal(s, s_ref)
    assert np.isinf(s_ref.reshape(-1)[0]) and np.isnan(s_ref.reshape(-1)[1])
    got = q.view(torch.uint8).cpu().numpy()
    nan = (codes & 0x7F) == 0x7F
    assert np.array_equal((got & 0x7F) == 0x7F, nan) and np.array_equal(got[~nan], codes[~nan])


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_swiglu_fp8_token(dtype):
    """Per-token SwiGLU + FP8: the last vector overlaps its neighbour, on every
    shape, on parked rows (more rows than resident workgroups) and past the
    widest shape."""
    vec = 16 // dtype.itemsize
    shapes = [(5, c) for c in _lengths(vec) + [256 * vec, 6144 * vec - 1, 6144 * vec + 1]]
    if dtype == torch.bfloat16:
        shapes += [(600, 17001), (300, 28665)]
    for rows, cols in shapes:
        g, u = inputs.swiglu_inputs(rows, cols, dtype, seed=cols)
        offset = cols % 3
        q = Guarded(g.shape, F8["e5m2"], offset)
        s = torch.empty(rows, dtype=torch.float32, device="cuda")
        native.swiglu_fp8_fwd(_off(g, offset), _off(u, offset), q.t, s, "e5m2", None)
        codes, s_ref, _ = eager.swiglu_fp8(g, u, "e5m2", None)
        assert_codes_equal(q.t, codes)
        assert_f32_bits_equal(s, s_ref)
        q.check()


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_fp8_token(dtype):
    vec = 16 // dtype.itemsize
    for cols in _lengths(vec) + [256 * vec, 6144 * vec - 1, 8192 * vec - 1, 8192 * vec + 1]:
        x = inputs.randn((5, cols), dtype, seed=cols)
        q = Guarded(x.shape, F8["e4m3"], cols % 3)
        s = torch.empty(5, dtype=torch.float32, device="cuda")
        native.fp8_quant_token_fwd(_off(x, cols % 3), q.t, s, "e4m3")
        codes, s_ref = ofp8.quant_token(x.float().numpy(), "e4m3")
        assert_codes_equal(q.t, codes)
        assert_f32_bits_equal(s, s_ref)
        q.check()


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_fp8_block(dtype):
    """128 x 128 tiles of ragged rows: the partial vector first in its tile
    (its loaded neighbours belong to the tile on the left), every remainder,
    one row, and matrices of barely one vector."""
    vec = 16 // dtype.itemsize
    shapes = [(1, vec), (1, vec + 1), (129, vec - 1), (127, 128 + 1), (257, 513), (130, 256 - 1), (128, 128)]
    shapes += [(131, 384 + d) for d in range(1, vec)]
    for m, n in shapes:
        x = inputs.randn((m, n), dtype, seed=m + n)
        x[:, n // 2:] *= 1000.0  # neighbouring tiles of other levels
        offset = 1 + n % 2
        q = Guarded(x.shape, F8["e4m3"], offset)
        s = torch.empty((m + 127) // 128, (n + 127) // 128, dtype=torch.float32, device="cuda")
        native.fp8_quant_block_fwd(_off(x, offset), q.t, s, "e4m3")
        codes, s_ref = ofp8.quant_block(x.float().numpy(), "e4m3")
        assert_codes_equal(q.t, codes)
        assert_f32_bits_equal(s, s_ref)
        q.check()


@pytest.mark.parametrize("dtype", DTYPES + [F8["e4m3"]], ids=lambda d: str(d).split(".")[-1])
def test_gather(dtype):
    """Ragged rows and, with more than two destinations a source row, sliced whole
    ones: one vector and less, both sides of every slice count, a last slice of
    few vectors, indices out of range, one destination row."""
    es = dtype.itemsize
    nbytes = [15, 17, 250, 254, 256, 258, 262, 1000, 1023, 1024, 2047, 2048, 2064, 4096, 4080, 8191, 8192, 8208, 11008, 16384]
    for rb in nbytes:
        h = max(1, rb // es)
        for n_dst in (1, 7, 4 * 19 + 1):
            src = torch.randint(0, 256, (19, h * es), dtype=torch.uint8, generator=torch.Generator().manual_seed(rb))
            idx = torch.randint(0, 19, (n_dst,), generator=torch.Generator().manual_seed(rb + n_dst))
            bad = torch.zeros(n_dst, dtype=torch.bool)
            if n_dst > 5:
                idx[3], idx[5] = 19, -2
                bad[3] = bad[5] = True
            offset = rb % 2
            dst = Guarded((n_dst, h), dtype, offset)
            native.token_gather_fwd(_off(src.view(dtype), offset), idx.cuda(), dst.t)
            ref = torch.where(bad[:, None], torch.zeros((), dtype=torch.uint8), src[torch.where(bad, 0, idx)])
            assert torch.equal(dst.t.view(torch.uint8).cpu(), ref), (rb, n_dst)
            dst.check()


@pytest.mark.parametrize("k", [1, 3, 4, 8, 16, 17])
@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_combine(dtype, k):
    """Main columns by unaligned vectors with the scalar columns beside them in
    one launch (a launch of their own past top 16): row lengths around the
    32-column boundaries, one token, terms out of range, unaligned buffers."""
    for h in (127, 128, 129, 159, 160, 1000, 4100, 4127, 8200):
        for t in (1, 9):
            eo, ui, w = inputs.combine_inputs(t, k, h, dtype, seed=h + k)
            ui_ref, w_ref = ui.clone(), w.clone()
            if t > 1:
                ui[2, k - 1], ui_ref[2, k - 1], w_ref[2, k - 1] = t * k, 0, 0.0
                ui[4, 0], ui_ref[4, 0], w_ref[4, 0] = -1, 0, 0.0
            offset = h % 2
            out = Guarded((t, h), dtype, offset)
            native.token_combine_fwd(_off(eo, offset), ui.cuda(), w.cuda(), out.t)
            assert bits_equal(out.t, moe.token_combine_aten(eo, ui_ref, w_ref)).all(), (t, h)
            out.check()


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_flat_swiglu_tails(dtype):
    """The elements past the last vector, plain and static-scale FP8: every
    remainder after one vector, after one workgroup's vectors and in the
    SiLU-table stream."""
    vec = 16 // dtype.itemsize
    for n in [vec + d for d in range(vec)] + [1024 * vec + d for d in (1, vec - 1)] + [(1 << 17) * vec + 3]:
        g, u = inputs.swiglu_inputs(1, n, dtype, seed=n)
        y, q = Guarded(g.shape, dtype, 0), Guarded(g.shape, F8["e4m3"], 0)
        s = torch.empty(1, dtype=torch.float32, device="cuda")
        native.swiglu_fwd(g.cuda(), u.cuda(), y.t)
        native.swiglu_fp8_fwd(g.cuda(), u.cuda(), q.t, s, "e4m3", 0.05)
        y_ref = eager.swiglu(g, u)
        assert bits_equal(y.t, y_ref).all(), n
        assert_codes_equal(q.t, ofp8.quant_static(y_ref.float().numpy(), 0.05, "e4m3"))
        y.check()
        q.check()


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
def test_fp8_tensor_one_workgroup_edge(dtype):
    """Per-tensor FP8 either side of what one workgroup takes whole."""
    vec = 16 // dtype.itemsize
    for nvec in (2048, 2049, 4096, 4097, 6144, 6145):
        x = inputs.randn((nvec, vec), dtype, seed=nvec)
        q = Guarded(x.shape, F8["e5m2"], 0)
        s = torch.empty(1, dtype=torch.float32, device="cuda")
        native.fp8_quant_tensor_fwd(x.cuda(), q.t, s, None, "e5m2")
        codes, s_ref = ofp8.quant_tensor(x.float().numpy(), "e5m2")
        assert_codes_equal(q.t, codes)
        assert_f32_bits_equal(s, np.asarray(s_ref).reshape(1))
        q.check()
