"""Either side of the lines that a measurement drew between two kernels of one
op: the call takes the kernel that was the faster one there, and its results are
the oracle's bits."""

from __future__ import annotations

import pytest
import torch

from custom_cuda_kernals_amd import _native as native
from oracle import eager, inputs, moe
from oracle import fp8 as ofp8
from tests._parity import assert_codes_equal, assert_f32_bits_equal, bits_equal
from tests._routes import kernels_of
from tests.test_moe_router_gpu import _check as check_router

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16


def _takes(call, kernel: str, threads: int | None = None) -> None:
    name, block = kernels_of(call)[0]
    assert kernel in name and threads in (None, block), (name, block)


# (tokens, top k, columns, kernel, threads)
COMBINES = [(1024, 1, 287, "token_combine_elems", 256), (1024, 1, 289, "token_combine_vec", None),
            (1025, 1, 287, "token_combine_vec", None), (1024, 2, 159, "token_combine_elems", 256),
            (1024, 2, 161, "token_combine_vec", None), (1025, 4, 129, "token_combine_vec", None),
            (256, 17, 599, "token_combine_elems", 256), (256, 17, 601, "token_combine_vec", None),
            (257, 17, 399, "token_combine_elems", 256), (257, 17, 401, "token_combine_vec", None),
            (1537, 17, 159, "token_combine_elems", 256), (1537, 17, 161, "token_combine_vec", None),
            (3073, 17, 129, "token_combine_vec", None),
            (5, 2, 8, "token_combine_elems", 64), (5, 17, 24, "token_combine_elems", 64),
            (7, 17, 72, "token_combine_vecINS_9CodecBF16ELi64ELi1ELi2ELb1ELb0E", 64),
            (7, 17, 4104, "token_combine_vecINS_9CodecBF16ELi512ELi1ELi2ELb1ELb1E", 512),
            (7, 16, 72, "token_combine_vecINS_9CodecBF16ELi64ELi2ELi2ELb0ELb1E", 64)]


@pytest.mark.parametrize("t,k,h,kernel,threads", COMBINES)
def test_combine(t, k, h, kernel, threads):
    eo, ui, w = inputs.combine_inputs(t, k, h, BF16, seed=h + k)
    ui_ref, w_ref = ui.clone(), w.clone()
    for row, j, bad in ((0, 0, -1), (t // 2, k - 1, t * k)):
        ui[row, j], ui_ref[row, j], w_ref[row, j] = bad, 0, 0.0
    d = [v.cuda() for v in (eo, ui, w)]
    out = torch.empty(t, h, dtype=BF16, device="cuda")
    _takes(lambda: native.token_combine_fwd(*d, out), kernel, threads)
    assert bits_equal(out, moe.token_combine_aten(eo, ui_ref, w_ref)).all()


@pytest.mark.parametrize("k", [1, 7, 8, 9, 15, 16])
@pytest.mark.parametrize("h", [1003, 1000])
def test_combine_of_no_rows_and_of_infinite_weights(h, k):
    """The other columns' loads stand under no branch: with no expert rows, and
    with weights that would make NaNs of a dropped term, dropped terms add nothing."""
    eo, ui, w = inputs.combine_inputs(6, k, h, BF16, seed=k)
    out = torch.empty(6, h, dtype=BF16, device="cuda")
    native.token_combine_fwd(eo[:0].cuda(), ui.cuda(), torch.full_like(w, float("inf")).cuda(), out)
    assert bits_equal(out, torch.zeros(6, h, dtype=BF16)).all()
    bad = ui.clone()
    bad[::2, k // 2] = 6 * k
    w_bad, ui_ref, w_ref = w.clone(), ui.clone(), w.clone()
    w_bad[::2, k // 2], ui_ref[::2, k // 2], w_ref[::2, k // 2] = float("nan"), 0, 0.0
    native.token_combine_fwd(eo.cuda(), bad.cuda(), w_bad.cuda(), out)
    assert bits_equal(out, moe.token_combine_aten(eo, ui_ref, w_ref)).all()


PLAIN, RAGGED, CACHED = (f"token_gather_slicesILb{a}ELb{c}E" for a, c in ((0, 0), (1, 0), (1, 1)))
# (source rows, destination rows, columns, kernel)
GATHERS = [(8, 33, 1016, "token_gather_rows"), (8, 33, 1280, PLAIN), (8, 32, 1280, "token_gather_rows"),
           (8, 25, 1024, PLAIN), (8, 24, 1024, "token_gather_rows"), (8, 17, 4096, PLAIN),
           (8, 16, 4096, "token_gather_rows"),
           (300, 901, 5120, PLAIN), (300, 900, 5120, "token_gather_flat"), (8, 25, 2880, PLAIN), (40, 189, 8320, "token_gather_flat"), (40, 190, 8320, PLAIN),
           (200, 585, 7168, "token_gather_flat"), (200, 586, 7168, PLAIN), (0, 3, 1024, PLAIN),
           (7, 9, 127, "token_gather_elems"), (7, 9, 129, CACHED), (0, 9, 1001, CACHED), (500, 2095, 1001, CACHED),
           (500, 2096, 1001, RAGGED), (40, 300, 8321, RAGGED)]


@pytest.mark.parametrize("ns,nd,h,kernel", GATHERS)
def test_gather(ns, nd, h, kernel):
    """(A source of no rows: every index is out of range, and nothing is read.)"""
    src = inputs.randn((max(ns, 1), h), BF16, seed=h)
    idx = torch.randint(-1, ns + 1, (nd,), generator=torch.Generator().manual_seed(nd))
    dst = torch.empty(nd, h, dtype=BF16, device="cuda")
    d = src[:ns].cuda(), idx.cuda()
    _takes(lambda: native.token_gather_fwd(*d, dst), kernel)
    ok = (idx >= 0) & (idx < ns)
    assert bits_equal(dst, torch.where(ok[:, None], src[torch.where(ok, idx, 0)], 0.0)).all()


WAVES = "moe_router_waves"
F32 = torch.float32
# (dtype, tokens, experts, top k, kernel)
ROUTERS = [(BF16, 2, 129, 8, WAVES), (BF16, 3, 129, 3, "ELi16ELi10E"), (BF16, 3, 129, 2, WAVES),
           (BF16, 1024, 160, 2, WAVES), (BF16, 1025, 160, 2, "ELi16ELi10E"), (BF16, 2, 128, 2, "ELi16ELi8E"),
           (BF16, 3072, 161, 1, WAVES), (BF16, 3073, 161, 1, "ELi16ELi12E"), (BF16, 5, 176, 6, WAVES), (BF16, 5, 176, 7, "ELi16ELi12E"), (BF16, 5, 177, 4, WAVES),
           (BF16, 5, 177, 5, "ELi16ELi12E"), (BF16, 2048, 193, 8, WAVES), (BF16, 2049, 193, 8, "ELi16ELi16E"),
           (BF16, 2049, 193, 4, WAVES), (BF16, 3073, 193, 4, "ELi16ELi16E"),
           (F32, 2, 160, 8, WAVES), (F32, 3, 160, 1, "ELi16ELi10E"), (F32, 4, 256, 8, WAVES),
           (F32, 5, 256, 8, "ELi16ELi16E"), (F32, 64, 256, 6, WAVES), (F32, 65, 256, 6, "ELi16ELi16E"),
           (F32, 1024, 200, 5, WAVES), (F32, 1025, 200, 5, "ELi16ELi16E"),
           (BF16, 24576, 32, 2, "ELi8ELi2E"), (F32, 24577, 32, 2, "ELi4ELi2E"), (BF16, 24577, 17, 9, "ELi4ELi2E"),
           (BF16, 24577, 33, 2, "ELi8ELi4E")]


@pytest.mark.parametrize("dtype,t,e,k,kernel", ROUTERS)
def test_router(dtype, t, e, k, kernel):
    logits = inputs.router_inputs(t, e, dtype, seed=t + e)
    logits[::3] = torch.round(logits[::3])  # many exact ties
    logits[1::5, : e // 2] = float("-inf")
    d = logits.cuda()
    w, i = torch.empty(t, k, device="cuda"), torch.empty(t, k, dtype=torch.int64, device="cuda")
    _takes(lambda: native.moe_router_fwd(d, w, i, True), kernel)
    check_router(logits, k, True)


def _ragged(rows: int, cols: int, seed: int, dtype=BF16) -> torch.Tensor:
    return inputs.randn((rows, cols), dtype, seed=seed)


# (rows, columns, kernel): the last template arguments are RAGGED, CACHED.
TOKENS = [(300, 9, "ELi64ELi1ELb1ELb1E"), (4056, 259, "ELi64ELi1ELb1ELb0E"), (4000, 259, "ELi64ELi1ELb1ELb1E"),
          (5, 511, "ELi64ELi1ELb1ELb1E"), (5, 513, "ELi64ELi2ELb1ELb0E"), (5, 8, "ELi64ELi1ELb0ELb0E")]


@pytest.mark.parametrize("m,n,kernel", TOKENS)
def test_fp8_token(m, n, kernel):
    x = _ragged(m, n, m + n)
    xd, q, s = x.cuda(), torch.empty(m, n, dtype=torch.float8_e4m3fn, device="cuda"), torch.empty(m, device="cuda")
    _takes(lambda: native.fp8_quant_token_fwd(xd, q, s, "e4m3"), kernel)
    codes, s_ref = ofp8.quant_token(x.float().numpy(), "e4m3")
    assert_codes_equal(q, codes)
    assert_f32_bits_equal(s, s_ref)


# (rows, columns, kernel): RAGGED, CACHED as above, after TAB, STATIC and LDSY.
GATED = [(300, 9, "ELb0ELb0ELb0ELb1ELb1E"), (4056, 259, "ELb0ELb0ELb0ELb1ELb0E"), (4000, 259, "ELb0ELb0ELb0ELb1ELb1E"),
         (5, 513, "ELi64ELi2ELi4ELb0ELb0ELb0ELb1ELb0E")]


@pytest.mark.parametrize("m,n,kernel", GATED)
def test_swiglu_fp8_token(m, n, kernel):
    g, u = inputs.swiglu_inputs(m, n, BF16, seed=n)
    gd, ud = g.cuda(), u.cuda()
    q, s = torch.empty(m, n, dtype=torch.float8_e5m2, device="cuda"), torch.empty(m, device="cuda")
    _takes(lambda: native.swiglu_fp8_fwd(gd, ud, q, s, "e5m2", None), kernel)
    codes, s_ref, _ = eager.swiglu_fp8(g, u, "e5m2", None)
    assert_codes_equal(q, codes)
    assert_f32_bits_equal(s, s_ref)


BLOCK, SCALAR = "fp8_block_resident", "fp8_block_generic"
# (dtype, rows, columns, kernel)
BLOCKS = [(BF16, 1, 4101, SCALAR), (BF16, 2, 129, SCALAR), (BF16, 3, 129, BLOCK), (BF16, 28, 9, SCALAR),
          (BF16, 29, 9, BLOCK), (BF16, 500, 7, SCALAR), (F32, 4, 129, SCALAR), (F32, 5, 129, BLOCK),
          (F32, 102, 5, SCALAR), (F32, 103, 5, BLOCK), (BF16, 1, 4096, BLOCK)]


@pytest.mark.parametrize("dtype,m,n,kernel", BLOCKS)
def test_fp8_block(dtype, m, n, kernel):
    x = _ragged(m, n, m + n, dtype)
    xd, q = x.cuda(), torch.empty(m, n, dtype=torch.float8_e4m3fn, device="cuda")
    s = torch.empty((m + 127) // 128, (n + 127) // 128, device="cuda")
    _takes(lambda: native.fp8_quant_block_fwd(xd, q, s, "e4m3"), kernel)
    codes, s_ref = ofp8.quant_block(x.float().numpy(), "e4m3")
    assert_codes_equal(q, codes)
    assert_f32_bits_equal(s, s_ref)


@pytest.mark.parametrize("dtype", [BF16, torch.float16, F32], ids=lambda d: str(d).split(".")[-1])
def test_swiglu_streams_of_whole_vectors_have_no_tail(dtype):
    vec = 16 // dtype.itemsize
    for n, tail in ((64 * vec, "Lb0EE"), (64 * vec + 1, "Lb1EE"), ((1 << 17) * vec, "Lb0EE"), ((1 << 17) * vec + 1, "Lb1EE")):
        g, u = inputs.swiglu_inputs(1, n, dtype, seed=n)
        gd, ud, y = g.cuda(), u.cuda(), torch.empty(1, n, dtype=dtype, device="cuda")
        q, s = torch.empty(1, n, dtype=torch.float8_e4m3fn, device="cuda"), torch.empty(1, device="cuda")
        for call in (lambda: native.swiglu_fwd(gd, ud, y), lambda: native.swiglu_fp8_fwd(gd, ud, q, s, "e4m3", 0.05)):
            (name, _), = kernels_of(call)
            assert "_flat" in name and tail in name, name
        y_ref = eager.swiglu(g, u)
        assert bits_equal(y, y_ref).all()
        assert_codes_equal(q, ofp8.quant_static(y_ref.float().numpy(), 0.05, "e4m3"))


# rope_heads streaming, with cached loads, with cached loads and stores; SPREAD last
STREAM, ONCHIP, SPLIT = (f"RopePolicyE{p}EL" for p in (0, 1, 2))
# (dtype, tokens, q heads, kv heads, head dim, kernel)
ROPES = [(BF16, 128, 40, 40, 96, SPLIT + "b1E"), (BF16, 129, 40, 40, 96, SPLIT + "b0E"), (BF16, 1, 32, 8, 96, SPLIT + "b0E"),
         (F32, 3, 8, 8, 512, ONCHIP + "b1E"), (F32, 300, 32, 8, 96, ONCHIP + "b0E"), (BF16, 3, 128, 8, 128, ONCHIP + "b1E"),
         (BF16, 2048, 32, 8, 128, ONCHIP + "b0E"), (F32, 1100, 32, 8, 128, "rope_tokens"),
         (F32, 3000, 12, 12, 64, STREAM + "b0E"), (F32, 100, 64, 8, 128, STREAM + "b1E"),
         (F32, 300, 64, 8, 128, STREAM + "b0E"), (F32, 3000, 16, 16, 64, "rope_tokens")]


@pytest.mark.parametrize("dtype,s,hq,hkv,d,kernel", ROPES)
def test_rope(dtype, s, hq, hkv, d, kernel):
    q, k, cos, sin = inputs.rope_inputs(1, s, hq, hkv, d, dtype=dtype, seed=s + d, theta=10000.0)
    t = [v.cuda() for v in (q, k, cos, sin)]
    qo, ko = torch.empty_like(t[0]), torch.empty_like(t[1])
    _takes(lambda: native.rope_fwd(*t, qo, ko), kernel)
    q_ref, k_ref = eager.rope(q, k, cos, sin)
    assert bits_equal(qo, q_ref).all() and bits_equal(ko, k_ref).all()
    native.rope_fwd(*t, t[0], t[1])
    assert bits_equal(t[0], q_ref).all() and bits_equal(t[1], k_ref).all()
