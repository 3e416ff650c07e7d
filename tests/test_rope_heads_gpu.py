"""RoPE of head dims whose half is any number of 16-byte chunks, bit for bit
against the oracle, out of place and in place: chunk counts that are no power
of two, tokens of more than 1024 (head, chunk) pairs, more pairs than the
chunk split is exact for (the scalar kernel), and both sides of the input
size from which the accesses stream."""

from __future__ import annotations

import pytest
import torch

from custom_cuda_kernals_amd.kernels import rope
from oracle import eager, inputs
from tests._parity import bits_equal

pytestmark = pytest.mark.gpu

# (batch, seq, q heads, kv heads, chunks of the half dimension)
CASES = [(2, 9, 3, 1, 3), (1, 7, 32, 8, 5), (2, 5, 32, 32, 6), (1, 3, 1, 1, 7), (1, 5, 9, 3, 12), (1, 4, 40, 30, 15),
         (1, 2, 3, 2, 33), (1, 2, 1, 1, 32), (1, 1, 5000, 461, 12), (1, 1, 5000, 462, 12), (3, 1100, 5, 0, 3),
         (1, 1100, 33, 8, 8), (1, 1100, 17, 16, 16), (2, 1100, 24, 8, 4)]
DTYPES = [torch.float32, torch.float16, torch.bfloat16]


def _check(b, s, hq, hkv, d, dtype, inplace):
    q, k, cos, sin = inputs.rope_inputs(b, s, hq, hkv, d, dtype=dtype, seed=s + hq + d, theta=10000.0)
    qo, ko = rope(q.cuda(), k.cuda(), cos.cuda(), sin.cuda(), inplace=inplace)
    q_ref, k_ref = eager.rope(q, k, cos, sin)
    assert bits_equal(qo, q_ref).all() and bits_equal(ko, k_ref).all()


@pytest.mark.parametrize("inplace", [False, True])
@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d).split(".")[-1])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_any_chunk_count(case, dtype, inplace):
    b, s, hq, hkv, chunks = case
    _check(b, s, hq, hkv, 2 * chunks * 16 // dtype.itemsize, dtype, inplace)


@pytest.mark.parametrize("seq", [2730, 2731, 2900])  # 64 MiB of q and k: 2730.67 tokens of 64 heads of 192
def test_streaming_line(seq):
    _check(1, seq, 48, 16, 192, torch.bfloat16, True)
