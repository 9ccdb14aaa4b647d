"""The FP32 forward kernels at the edges of their tiles, on 4-byte aligned views, and with
NaN and infinite inputs, against FP64 on the CPU."""

import math

import pytest
import torch

from flash_attention_2_lab_amd import capi

pytestmark = pytest.mark.gpu

# Worst case of a score: two FP32 sums of D/2 products and their sum, (D/2 + 2) roundings of
# at most 2^-24 * sum |q_d k_d| / sqrt(D), about 5 for N(0, 1) inputs at D = 64 and 7 at
# D = 128: at most 2.8e-5, a relative error of the probability. Outputs are averages of
# values below 5, with their own sums' rounding far below that.
ATOL = 5 * 2.8e-5

# Relative error in the 2-norm against FP64: the kernels show 2e-7 to 4e-7 (FP32's rounding of the
# scores, the probabilities and the sums), and one that lost one of the six products of the
# split operands 7e-6 or more (tests/test_f32_split_cpu.py).
REL = 1e-6


def _inputs(batch_heads, seq_len, dim, seed=0, offset=0):
    """N(0, 1) tensors whose storage starts `offset` floats past a 16-byte boundary."""
    gen = torch.Generator().manual_seed(seed)
    size = batch_heads * seq_len * dim
    flat = [torch.randn(size + offset, generator=gen).cuda()[offset:] for _ in range(3)]
    return [t.view(1, batch_heads, seq_len, dim) for t in flat]


def _exact(q, k, v):
    q, k, v = (t.double().cpu() for t in (q, k, v))
    return torch.softmax(q @ k.transpose(-1, -2) / math.sqrt(q.shape[-1]), dim=-1) @ v


# 16-query kernel, 32-query kernel with 8 and with 4 waves: at most 128, at most 256 and more
# blocks of 32 queries. Lengths around one tile, one tile per wave and the next, with and
# without a partial last tile.
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("batch_heads, seq_len", [
    (1, 1), (2, 15), (2, 17), (1, 127), (1, 129), (1, 257), (1, 1040), (4, 1024),
    (129, 1), (129, 31), (65, 33), (43, 95), (33, 128), (26, 161), (5, 1025), (9, 520),
    (130, 40), (257, 1), (260, 31), (129, 64), (65, 129), (52, 161), (9, 1025)])
def test_f32_forward_edges(batch_heads, seq_len, dim, offset):
    q, k, v = _inputs(batch_heads, seq_len, dim, offset=offset)
    out = capi.attention_forward_f32(q, k, v).double().cpu()
    expected = _exact(q, k, v)
    torch.testing.assert_close(out, expected, atol=ATOL, rtol=0)
    assert (out - expected).norm() <= REL * expected.norm()


HEADS = [1, 24, 40]  # 16-query kernel, 32-query kernel with 8 and with 4 waves


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("batch_heads", HEADS)
def test_f32_forward_nan_and_infinity(batch_heads, dim):
    """NaN and infinities reach exactly the outputs the formula gives them."""
    q, k, v = _inputs(batch_heads, 197, dim, seed=3)
    q[0, 0, 3, 5] = math.nan
    q[0, 0, 9, 7] = math.inf
    k[0, 0, 20, 2] = math.inf     # scores of +inf, -inf: rows of NaN, and rows without key 20
    v[0, 0, 60, 11] = math.inf
    v[0, 0, 61, 12] = math.nan
    v[0, 0, 62, 13] = -math.inf
    # Another head: -inf scores hide two whole key tiles.
    head = batch_heads - 1
    if head:
        k[0, head, :64] = 0.0
        k[0, head, :64, 0] = -math.inf
        q[0, head, :, 0] = q[0, head, :, 0].abs() + 0.1
        v[0, 1, 196, 3] = math.inf
        k[0, 2, 0, dim - 1] = -math.inf
    out = capi.attention_forward_f32(q, k, v).double().cpu()
    torch.testing.assert_close(out, _exact(q, k, v), atol=ATOL, rtol=0, equal_nan=True)


@pytest.mark.parametrize("batch_heads", HEADS)
def test_f32_forward_keeps_subnormals(batch_heads):
    """Values below the smallest normal number are averaged, not flushed."""
    q, k, _ = _inputs(batch_heads, 197, 64, seed=4)
    v = torch.full_like(q, 2.0 ** -140)
    out = capi.attention_forward_f32(q, k, v)
    assert (out.double() / 2.0 ** -140 - 1).abs().max().item() <= 2.0 ** -5


# Values at either end of the exponent range keep all their bits: scaled dimensions of Q and
# K whose products are of ordinary size, and scaled columns of V.
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("batch_heads", HEADS)
@pytest.mark.parametrize("exponent", [-110, 110])
def test_f32_forward_keeps_small_and_large_values(batch_heads, dim, exponent):
    q, k, v = _inputs(batch_heads, 130, dim, seed=6)
    q[0, 0, :, 3] *= 2.0 ** exponent
    k[0, 0, :, 3] *= 2.0 ** -exponent
    q[0, -1] *= 2.0 ** -exponent
    k[0, -1] *= 2.0 ** exponent
    v[0, 0, :, 5] *= 2.0 ** exponent
    v[0, -1, :, 6] *= 2.0 ** -exponent
    out = capi.attention_forward_f32(q, k, v).double().cpu()
    expected = _exact(q, k, v)
    scale = v.double().cpu().abs().amax(dim=-2, keepdim=True) / 5.0
    assert ((out - expected).abs() <= ATOL * scale).all()
    # Every column by itself: the scaled ones keep as many bits as the others.
    assert ((out - expected).norm(dim=-2) <= REL * expected.norm(dim=-2)).all()


# Scores of 2^40 and more, whose product with log2(e) rounds by more than a float's exponents
# span: each row is its largest score's value row. The scores' own errors, 2^-20 of them at most,
# stay far below the gaps between them.
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("batch_heads", HEADS)
def test_f32_forward_huge_scores(batch_heads, dim):
    q, k, v = _inputs(batch_heads, 197, dim, seed=8)
    q[0, 0] *= 2.0 ** 20
    k[0, 0] *= 2.0 ** 20
    # Growing along the keys, so that the running max passes from ordinary to huge values.
    k[0, -1] *= torch.logspace(0, 50, 197, base=2.0, device="cuda").unsqueeze(-1)
    out = capi.attention_forward_f32(q, k, v).double().cpu()
    torch.testing.assert_close(out, _exact(q, k, v), atol=ATOL, rtol=0)


@pytest.mark.parametrize("batch_heads", HEADS)
def test_f32_forward_huge_negative_scores(batch_heads):
    """Every score of every row below -2^38, from one product each: the smallest one wins."""
    q, k, v = _inputs(batch_heads, 197, 64, seed=9)
    q[..., 1:], k[..., 1:] = 0.0, 0.0
    q[..., 0] = (q[..., 0].abs() + 1.0) * 2.0 ** 20
    k[..., 0] = -(k[..., 0].abs() + 1.0) * 2.0 ** 21
    out = capi.attention_forward_f32(q, k, v).double().cpu()
    torch.testing.assert_close(out, _exact(q, k, v), atol=ATOL, rtol=0)


# A score of one product is exact, so a probability of 2^-122 is off by the rounding of its
# exponent, 122 * 2^-24, and what exp2 and the sums add: 1.5e-5 in all.
@pytest.mark.parametrize("case", ["zero_value", "large_values", "small_value"])
@pytest.mark.parametrize("batch_heads", HEADS)
def test_f32_forward_keeps_small_weights(batch_heads, case):
    """What a probability near the smallest float, or a value below it, gives keeps its bits
    when it is what the result consists of."""
    q, k, v = _inputs(batch_heads, 197, 64, seed=10)
    gen = torch.Generator().manual_seed(11)
    low, high = (-200.0, -190.0) if case == "small_value" else (-85.0, -83.0)
    q.zero_()
    k.zero_()
    q[..., 0] = 8.0
    k[..., 0] = (low + (high - low) * torch.rand(batch_heads, 197, generator=gen)).cuda()
    k[..., 100, 0] = 0.0  # every row sees key 100 with probability 1
    v = v.abs() + 0.5
    if case == "zero_value":
        v[..., 100, :] = 0.0
    elif case == "large_values":
        v *= 2.0 ** 122
        v[..., 100, :] *= 2.0 ** -122
    else:
        v[..., 100, :] *= 2.0 ** -121
    out = capi.attention_forward_f32(q, k, v).double().cpu()
    torch.testing.assert_close(out, _exact(q, k, v), atol=0, rtol=2e-5)


# Scores: 64 x 64 blocks of 32 x 32, dimensions in chunks of 64; 4-byte fetches when the
# head dimension is not a multiple of 4 or the storage is 4-byte aligned.
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("seq_len", [1, 31, 33, 63, 65, 130])
@pytest.mark.parametrize("dim", [1, 3, 4, 60, 64, 68, 130, 256])
def test_scores_edges(seq_len, dim, offset):
    q, k, _ = _inputs(3, seq_len, dim, seed=dim, offset=offset)
    out = capi.attention_scores_f32(q, k).double().cpu()
    exact_q, exact_k = q.double().cpu(), k.double().cpu()
    expected = exact_q @ exact_k.transpose(-1, -2) / math.sqrt(dim)
    # Two sums of dim/2 products, each rounding at most 2^-24 of sum |q_d k_d|.
    bound = (dim / 2 + 3) * 2.0 ** -24 * (exact_q.abs() @ exact_k.abs().transpose(-1, -2)) / math.sqrt(dim)
    assert ((out - expected).abs() <= bound).all()


def _blocks_and_ranges(batch_heads, seq_len):
    """64-column blocks of a row of blocks, and the workgroups they are dealt to: four workgroups
    per CU in all, and at most eight blocks each."""
    blocks = -(-seq_len // 64)
    return blocks, min(blocks, max(-(-blocks // 8), -(-1024 // (batch_heads * blocks))))


# Workgroups of several blocks: the next block's operands land in the other ring slot while a
# block is multiplied and stored. Two blocks each, one or two, five, six or seven, and eight; one,
# two, three and four chunks of dimensions a block.
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("batch_heads, seq_len", [(8, 1024), (8, 1000), (40, 333), (64, 600), (20, 2100), (128, 512)])
@pytest.mark.parametrize("dim", [3, 60, 64, 68, 130, 200])
def test_scores_of_several_blocks(batch_heads, seq_len, dim, offset):
    blocks, ranges = _blocks_and_ranges(batch_heads, seq_len)
    assert ranges < blocks
    q, k, _ = _inputs(batch_heads, seq_len, dim, seed=dim, offset=offset)
    out = capi.attention_scores_f32(q, k)
    for head in range(batch_heads):
        # On the GPU: FP64 products of a plain matrix and a transposed copy.
        exact_q, exact_k = q[0, head].double(), k[0, head].double().t().contiguous()
        expected = exact_q @ exact_k / math.sqrt(dim)
        bound = (dim / 2 + 3) * 2.0 ** -24 * (exact_q.abs() @ exact_k.abs()) / math.sqrt(dim)
        assert ((out[0, head].double() - expected).abs() <= bound).all()


# The narrow fetch: up to 16 dimensions, four rows an instruction; its edges in dimensions and rows,
# from one block to ranges of several, beside the fetches that take over above 16 dimensions and,
# for 16-byte aligned rows of whole chunks, above 16 rows.
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("batch_heads, seq_len", [(3, 1), (2, 4), (2, 5), (2, 16), (2, 17), (2, 62), (2, 97), (70, 300)])
@pytest.mark.parametrize("dim", [1, 2, 5, 8, 9, 15, 16, 17])
def test_scores_narrow_fetch(batch_heads, seq_len, dim, offset):
    q, k, _ = _inputs(batch_heads, seq_len, dim, seed=dim, offset=offset)
    out = capi.attention_scores_f32(q, k).double().cpu()
    exact_q, exact_k = q.double().cpu(), k.double().cpu()
    expected = exact_q @ exact_k.transpose(-1, -2) / math.sqrt(dim)
    bound = (dim / 2 + 3) * 2.0 ** -24 * (exact_q.abs() @ exact_k.abs().transpose(-1, -2)) / math.sqrt(dim)
    assert ((out - expected).abs() <= bound).all()


# The one-row fetch past 64 dimensions stops at the last row of units of up to 24 rows and fetches 32
# of larger ones; lengths on both sides, in the first and in the second unit of a block.
@pytest.mark.parametrize("batch_heads, seq_len", [(3, 1), (2, 24), (2, 25), (2, 32), (2, 56), (2, 57), (2, 88), (40, 345)])
@pytest.mark.parametrize("dim", [65, 129])
def test_scores_few_rows(batch_heads, seq_len, dim):
    q, k, _ = _inputs(batch_heads, seq_len, dim, seed=dim, offset=1)
    out = capi.attention_scores_f32(q, k).double().cpu()
    exact_q, exact_k = q.double().cpu(), k.double().cpu()
    expected = exact_q @ exact_k.transpose(-1, -2) / math.sqrt(dim)
    bound = (dim / 2 + 3) * 2.0 ** -24 * (exact_q.abs() @ exact_k.abs().transpose(-1, -2)) / math.sqrt(dim)
    assert ((out - expected).abs() <= bound).all()


def test_scores_nan_and_infinity():
    q, k, _ = _inputs(2, 70, 64, seed=5)
    q[0, 0, 3, 5], q[0, 1, 65, 63], k[0, 0, 40, 2], k[0, 1, 1, 0] = math.nan, math.inf, -math.inf, math.inf
    out = capi.attention_scores_f32(q, k).double().cpu()
    expected = q.double().cpu() @ k.double().cpu().transpose(-1, -2) / 8.0
    torch.testing.assert_close(out, expected, atol=1e-4, rtol=0, equal_nan=True)
