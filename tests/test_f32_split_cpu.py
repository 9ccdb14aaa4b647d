"""The FP32 forward's split of operands into BF16 parts, emulated in float64 on the CPU: the bound
that tests/test_f32_forward_gpu.py holds the kernels to passes the six products they sum and
fails for every five of them, so a kernel that lost one would not pass."""

import math

import pytest
import torch

REL = 1e-6  # relative error in the 2-norm, for N(0, 1) inputs

SIX = [(2, 0), (0, 2), (1, 1), (1, 0), (0, 1), (0, 0)]


def _parts(x):
    """x as three values of 8 significant bits, each the rest cut to a float's upper 16 bits."""
    parts = []
    for _ in range(3):
        cut = (x.contiguous().view(torch.int32) & -65536).view(torch.float32)
        parts.append(cut.double())
        x = x - cut
    assert not x.any()
    return parts


def _product(a, b, products):
    a, b = _parts(a), _parts(b)
    return sum(a[i] @ b[j] for i, j in products)


def _error(seq_len, dim, score_products, value_products):
    gen = torch.Generator().manual_seed(seq_len + dim)
    q, k, v = (torch.randn(2, seq_len, dim, generator=gen) for _ in range(3))
    scores = _product(q, k.transpose(-1, -2), score_products) / math.sqrt(dim)
    p = (scores - scores.amax(-1, keepdim=True)).exp().float()
    out = _product(p, v, value_products) / p.double().sum(-1, keepdim=True)
    exact = torch.softmax(q.double() @ k.double().transpose(-1, -2) / math.sqrt(dim), dim=-1) @ v.double()
    return ((out - exact).norm() / exact.norm()).item()


@pytest.mark.parametrize("seq_len, dim", [(31, 64), (129, 128), (520, 64)])
def test_bound_sees_every_product(seq_len, dim):
    assert _error(seq_len, dim, SIX, SIX) < REL / 2
    for lost in range(6):
        five = SIX[:lost] + SIX[lost + 1:]
        assert _error(seq_len, dim, five, SIX) > 2 * REL
        assert _error(seq_len, dim, SIX, five) > 2 * REL


def test_bound_sees_a_lost_part_of_a_single_value():
    """At one key the result is V itself."""
    assert _error(1, 64, SIX, SIX) < REL / 2
    assert _error(1, 64, SIX, SIX[:1] + SIX[2:]) > 2 * REL
