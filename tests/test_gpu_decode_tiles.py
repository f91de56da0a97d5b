"""GPU parity of decode attention for query groups on the matrix cores.

Groups of three or more query heads per kv head at head_dim 64 and 128 run in
tiles of up to 4 or 8 heads (several tiles above 8, the last one partly
filled).  Cases sit at the tiles' edges: group sizes around 4 and 8, contexts
around one wave iteration (16 or 32 tokens) and one page, pages that do and
do not hold whole iterations, whole sequences, split-K and the balanced walk.
Tolerance: the decode gate against the fp32 oracle."""

import pytest
import torch

from gpu_cases import decode_inputs
from mini_engine_hip.kernels.data import write_kv_cache_batch
from mini_engine_hip.kernels.paged import paged_attention, paged_attention_decode_write
from oracle import paged_oracle

pytestmark = pytest.mark.gpu
DEV = "cuda"
GATE = {torch.float16: 2e-3, torch.bfloat16: 1.6e-2}


def oracle(args):
    return paged_oracle.fp32_oracle(dict(zip(paged_oracle.TENSOR_NAMES, args[:5])), args[5])


def check(args, dtype, partition):
    dev = [a.to(DEV) if isinstance(a, torch.Tensor) else a for a in args]
    actual = paged_attention(*dev, partition_tokens=partition).float().cpu()
    assert (actual - oracle(args)).abs().max().item() <= GATE[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("group", [3, 4, 5, 7, 8, 9, 12, 16, 17])
def test_group_sizes_around_the_tiles(dtype, dim, group):
    lengths = (1, 15, 16, 17, 33, 130, 257, 700)
    args = decode_inputs(dtype, head_dim=dim, lengths=lengths, heads=2 * group, kv_heads=2, seed=100 * dim + group)
    for partition in (0, 64, 192, -1):
        check(args, dtype, partition)


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("group", [3, 5, 6, 8, 12, 17])
@pytest.mark.parametrize("block,lengths", [(16, (33, 1, 18)), (24, (70, 24)), (256, (5,)), (16, (2500,))])
def test_groups_of_small_calls(block, lengths, group, dim):
    """Calls of few tokens split groups into tiles of 1, 2 or 4 heads: whole
    sequences, split-K and the walk."""
    dtype = torch.float16
    args = decode_inputs(dtype, head_dim=dim, block_size=block, lengths=lengths, heads=group, kv_heads=1,
                         seed=block + group)
    for partition in (0, 64, -1):
        check(args, dtype, partition)


@pytest.mark.parametrize("block,lengths,partition", [
    (7, (50, 13, 1), 0), (24, (500, 24, 25), 128), (5, (333, 40), -1),     # per-token page lookups
    (16, (4097,), 0), (256, (2048, 1, 700), 0), (256, (5000, 4100), 0),    # plan's walk and split-K
    (16, tuple([200] * 40), 0), (16, tuple(range(1, 161, 4)), 0),           # whole sequences
])
@pytest.mark.parametrize("dim,group", [(64, 7), (128, 4), (128, 7)])
def test_pages_and_modes(block, lengths, partition, dim, group):
    dtype = torch.bfloat16
    args = decode_inputs(dtype, head_dim=dim, block_size=block, lengths=lengths, heads=4 * group, kv_heads=4,
                         seed=block + len(lengths))
    check(args, dtype, partition)


@pytest.mark.parametrize("dim,group", [(64, 8), (128, 4), (128, 8)])
def test_scores_that_keep_rising_and_stale_rows(dim, group):
    """Scores rise by several binary orders along the context, so that the
    running reference is raised again and again (and late keys carry nearly
    all of the weight); rows past a context's end hold NaN and infinities."""
    dtype = torch.float16
    args = list(decode_inputs(dtype, head_dim=dim, lengths=(601, 250), heads=2 * group, kv_heads=2, seed=dim))
    q, key, value, table, lens, block = args
    q.fill_(0.5)
    for b in range(2):
        for i, page in enumerate(table[b].tolist()):
            key[page] = 0.02 * key[page] + 0.004 * i * (128 / dim)
    last = table[1, 250 // block]
    key[last, 250 % block:] = float("nan")
    value[last, 250 % block:] = float("inf")
    dev = [a.to(DEV) if isinstance(a, torch.Tensor) else a for a in args]
    clean = [a.clone() if isinstance(a, torch.Tensor) else a for a in args]
    clean[1][last, 250 % block:] = 0
    clean[2][last, 250 % block:] = 0
    for partition in (0, 64, -1):
        actual = paged_attention(*dev, partition_tokens=partition, validate=False).float().cpu()
        assert (actual - oracle(clean)).abs().max().item() <= GATE[dtype]


@pytest.mark.parametrize("dim,group", [(64, 4), (64, 8), (128, 2), (128, 4), (128, 7)])
def test_one_score_for_all_of_a_tokens_lanes(dim, group):
    """Scores near 2^13 binary orders that differ by a few: a lane that rounded its
    token's score otherwise than its neighbours gives the dims it holds other weights
    than the sum has, 2^-10 apart.  With V all 1 every output is the weights' sum over
    itself, 1 to the few fp32 roundings by which the two sums' orders differ."""
    gen = torch.Generator().manual_seed(dim + group)
    args = list(decode_inputs(torch.float16, head_dim=dim, lengths=(5, 11, 20, 30, 48, 100, 200, 300) * 4,
                              heads=8 * group, kv_heads=8))
    q, key, value = args[:3]
    sign = torch.randint(0, 2, (8, dim), generator=gen) * 2.0 - 1
    scale = 40 * (128 / dim) ** 0.5
    q.copy_((sign * scale).repeat_interleave(group, 0) * (1 + 0.01 * torch.randn(q.shape, generator=gen)))
    key.copy_(20 * sign + 0.03 * key.float())
    value.fill_(1.0)
    dev = [a.to(DEV) if isinstance(a, torch.Tensor) else a for a in args]
    for partition in (0, 64, -1):
        out = paged_attention(*dev, partition_tokens=partition)
        assert torch.equal(out, torch.ones_like(out))


def test_absent_pages_and_lengths_count_as_nothing():
    """Trusted calls with pages and lengths out of range: those tokens are
    absent, a sequence without any gives zeros."""
    args = list(decode_inputs(torch.bfloat16, lengths=(300, 90, 64), heads=28, kv_heads=4))
    q, key, value, table, lens, block = [a.to(DEV) if isinstance(a, torch.Tensor) else a for a in args]
    table = table.clone()
    table[0, 3] = 1 << 40
    table[1, :] = -1
    lens = torch.tensor([300, 90, 1 << 40], device=DEV)
    keep = [t for t in range(300) if t // block != 3]
    flat_k = key[table[0].clamp(0, key.shape[0] - 1)].flatten(0, 1)[keep].float()
    flat_v = value[table[0].clamp(0, key.shape[0] - 1)].flatten(0, 1)[keep].float()
    score = torch.stack([flat_k[:, h // 7] @ q[0, h].float() for h in range(28)]) * 128 ** -0.5
    want = torch.stack([score[h].softmax(0) @ flat_v[:, h // 7] for h in range(28)])
    for partition in (0, 64, -1):
        out = paged_attention(q, key, value, table, lens, block, validate=False, partition_tokens=partition).float()
        assert (out[0] - want).abs().max().item() <= GATE[torch.bfloat16]
        assert out[1].abs().max().item() == 0 and out[2].abs().max().item() == 0


@pytest.mark.parametrize("lengths,kv_heads", [
    ((2048,), 1), ((3000,), 4), ((1, 2500, 64, 65, 129, 2), 4), (tuple([2300] * 20), 4),
    ((2730,) * 12, 1), ((2730,) * 11 + (2739,), 1),  # 32760 and 32769 tokens: parts of 128 and of 256
    (tuple(1 + 37 * i for i in range(64)), 3), (tuple(2600 - 40 * i for i in range(59)), 4),
])
@pytest.mark.parametrize("group", [7, 8, 12])
def test_partitions_decided_by_the_lengths(lengths, kv_heads, group):
    """8-head tiles over tables of 2048 tokens and more: the partition length
    follows from the lengths (one sequence, 64 of them, equal, one token,
    two tiles per group), also when they change under the same tables, with
    an empty sequence, and with the step's row written by the launch."""
    dtype = torch.bfloat16
    args = decode_inputs(dtype, lengths=lengths, heads=group * kv_heads, kv_heads=kv_heads, seed=len(lengths))
    check(args, dtype, 0)
    q, key, value, table, lens, block = [a.to(DEV) if isinstance(a, torch.Tensor) else a for a in args]
    shorter = torch.clamp(lens // 3, min=1)
    got = paged_attention(q, key, value, table, shorter, block, validate=False).float().cpu()
    want = oracle(list(args[:4]) + [shorter.cpu(), block])
    assert (got - want).abs().max().item() <= GATE[dtype]
    empty = lens.clone()
    empty[0] = 0
    out = paged_attention(q, key, value, table, empty, block, validate=False)
    assert out[0].abs().max().item() == 0
    new_k, new_v = (torch.randn(len(lengths), kv_heads, 128, device=DEV).to(dtype) for _ in range(2))
    k2, v2 = key.clone(), value.clone()
    fused = paged_attention_decode_write(q, key, value, table, lens, block, new_k, new_v, validate=False)
    write_kv_cache_batch(k2, v2, table, lens - 1, new_k, new_v, block, validate=False)
    assert torch.equal(key, k2) and torch.equal(value, v2)
    assert torch.equal(fused, paged_attention(q, k2, v2, table, lens, block, validate=False))


@pytest.mark.parametrize("block", [8, 16, 24, 32, 48, 17])
@pytest.mark.parametrize("dim,group", [(64, 2), (64, 4), (64, 8), (128, 4)])
def test_runs_of_pages(block, dim, group):
    """Iterations of 32 tokens at 64 dims cover two runs of 16, each in a page
    of its own; contexts end inside the first and the second run, and absent
    pages lie under either."""
    dtype = torch.float16
    args = list(decode_inputs(dtype, head_dim=dim, block_size=block, lengths=(1, 16, 17, 31, 32, 33, 49, 300, 530),
                              heads=2 * group, kv_heads=2, seed=block + dim))
    for partition in (0, 128, -1):
        check(args, dtype, partition)
    q, k, v, table, lens, _ = [a.to(DEV) if isinstance(a, torch.Tensor) else a for a in args]
    for bad, hole in ((-1, 0), (k.shape[0], 1), (1 << 33, 2)):
        holed = table.clone()
        holed[7, hole] = bad
        out = paged_attention(q, k, v, holed, lens, block, validate=False).float().cpu()
        rows = torch.arange(300).div(block, rounding_mode="floor") != hole
        pages = args[3][7].repeat_interleave(block)[:300][rows]
        offsets = (torch.arange(300) % block)[rows]
        keys, values = args[1][pages, offsets].float(), args[2][pages, offsets].float()
        query = args[0][7].float().view(2, group, dim)
        scores = torch.einsum("hgd,thd->hgt", query, keys) / dim ** 0.5
        want = torch.einsum("hgt,thd->hgd", scores.softmax(-1), values).reshape(2 * group, dim)
        assert (out[7] - want).abs().max().item() <= GATE[dtype]


@pytest.mark.parametrize("dim", [16, 64])
@pytest.mark.parametrize("block,length", [(3, 1048575), (5, 1048575), (1000, 1048000), (524287, 1048574), (174763, 174764)])
def test_pages_of_no_power_of_two(block, length, dim):
    """Page lookups up to the largest capacity, 2^20 tokens, by a product instead of
    a division: every key's row holds the key's position, spread over the pages by a
    permutation, and the query picks out single positions, the last one and those
    around page ends among them."""
    width = -(-length // block)
    gen = torch.Generator(device=DEV).manual_seed(block)
    table = torch.randperm(width, generator=gen, device=DEV)
    spots = [t for t in {length - 1, length - length % block, block - 1, block, 2 * block - 1, length // 2, 0} if 0 <= t < length][:8]
    key = torch.zeros(width, block, 1, dim, dtype=torch.float16, device=DEV)
    value = torch.zeros_like(key)
    q = torch.zeros(1, 4, dim, dtype=torch.float16, device=DEV)
    q[0, :, 0] = 240.0
    for heads in (spots[:4], spots[4:]):
        key.zero_()
        for h, t in enumerate(heads):
            q[0, h] = 0
            q[0, h, h] = 240.0
            key[table[t // block], t % block, 0, h] = 240.0
            value[table[t // block], t % block, 0] = 1.0 + h
        lens = torch.tensor([length], device=DEV)
        out = paged_attention(q, key, value, table[None], lens, block)
        want = torch.tensor([1.0 + h for h in range(len(heads))], device=DEV).half()
        assert torch.equal(out[0, :len(heads)], want[:, None].expand(-1, dim))
        value.zero_()
