"""GPU parity of the pipelined prefill loop over pages smaller than a key
tile (8, 16 and 32 tokens) and in dense mode, and of the order of query
blocks across sequences."""

import math

import pytest
import torch

from mini_engine_hip.kernels.prefill import (paged_prefill_attention, paged_prefill_workspace_bytes,
                                              prefill_attention)
from oracle import paged_oracle

pytestmark = pytest.mark.gpu
DEV = "cuda"
GATE = {torch.float16: 2e-3, torch.bfloat16: 1.6e-2}


def paged_case(new, prior, block, heads, kv_heads, dtype, seed, dim=128):
    gen = torch.Generator().manual_seed(seed)
    cu = torch.tensor([0] + torch.tensor(new).cumsum(0).tolist())
    starts = torch.tensor(prior)
    lens = starts + torch.tensor(new)
    width = max(1, -(-int(lens.max()) // block))
    pages = len(new) * width + 3
    kc = torch.randn(pages, block, kv_heads, dim, generator=gen).to(dtype)
    vc = torch.randn(pages, block, kv_heads, dim, generator=gen).to(dtype)
    tables = torch.randperm(pages, generator=gen)[:len(new) * width].view(len(new), width)
    q = torch.randn(int(cu[-1]), heads, dim, generator=gen).to(dtype)
    return [q, kc, vc, cu, starts, tables, lens]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("block", [8, 16, 32])
@pytest.mark.parametrize("new,prior,chunk", [
    ([64, 1, 130], [0, 63, 64], 0),          # whole tiles, one key past a tile, one before
    ([40], [4400], 0), ([40], [4400], 8192),  # more than a window of 64 tiles, split and not
    ([300, 77], [1200, 41], 256),            # walks over key chunks
])
def test_small_pages_match_the_oracle(dtype, block, new, prior, chunk):
    args = paged_case(new, prior, block, 8, 4, dtype, seed=block + sum(new))
    actual = paged_prefill_attention(*[a.to(DEV) for a in args], block, chunk_tokens=chunk).float().cpu()
    expected = paged_oracle.paged_prefill_attention(*args, block, cast=False)
    assert (actual - expected).abs().max().item() <= GATE[dtype]


@pytest.mark.parametrize("block", [8, 16, 32, 64])
def test_absent_pages_inside_a_tile(block):
    """Trusted calls: a page out of range in the middle of a whole tile; its
    keys are absent for every wave, the tile's other keys are not."""
    dtype = torch.bfloat16
    args = paged_case([50, 200], [400, 0], block, 8, 4, dtype, seed=block)
    q, kc, vc, cu, starts, tables, lens = args
    hole = 192 // block  # keys 192 .. 192 + block of sequence 0
    tables[0, hole] = kc.shape[0] + 5
    out = paged_prefill_attention(*[a.to(DEV) for a in args], block, validate=False).float().cpu()
    keep = [k for k in range(450) if k // block != hole]
    key = kc[tables[0].clamp(max=kc.shape[0] - 1)].flatten(0, 1).float()
    value = vc[tables[0].clamp(max=kc.shape[0] - 1)].flatten(0, 1).float()
    for row in (0, 49):
        seen = [k for k in keep if k <= 400 + row]
        for h in (0, 7):
            p = (key[seen, h // 2] @ q[row, h].float() * 128 ** -0.5).softmax(0)
            assert (out[row, h] - p @ value[seen, h // 2]).abs().max().item() <= GATE[dtype]


@pytest.mark.parametrize("seqs,heads,kv_heads", [(40, 16, 8), (64, 8, 8), (65, 16, 8)])
def test_query_blocks_of_many_sequences(seqs, heads, kv_heads):
    """Enough ragged sequences that keys are not split: the work-groups take
    the query blocks by falling key end across sequences (up to 64 of them;
    65 keep the order of the batch), empty sequences among them.  Every
    block has to be computed exactly once: the outputs start as NaN where a
    block is missed, and every row is compared."""
    dtype, block = torch.bfloat16, 16
    gen = torch.Generator().manual_seed(seqs)
    new = torch.randint(0, 400, (seqs,), generator=gen).tolist()
    new[3] = 0
    prior = torch.randint(0, 900, (seqs,), generator=gen).tolist()
    prior[5] = 0
    args = paged_case(new, prior, block, heads, kv_heads, dtype, seed=seqs)
    dev = [a.to(DEV) for a in args]
    # Keys are not split: nothing to merge.
    assert paged_prefill_workspace_bytes(seqs, sum(new), heads, kv_heads, 128, block, args[5].shape[1], dtype) == 0
    torch.full_like(dev[0], float("nan"))  # freed at once: the output's storage
    actual = paged_prefill_attention(*dev, block, validate=False).float().cpu()
    expected = paged_oracle.paged_prefill_attention(*args, block, cast=False)
    assert (actual - expected).abs().max().item() <= GATE[dtype]


@pytest.mark.parametrize("dim", [64, 128, 256])
@pytest.mark.parametrize("lengths", ["alike", "ragged"])
def test_query_blocks_over_short_tables(lengths, dim):
    """Tables of at most 512 tokens: longest blocks first where the sequences are
    alike, in turn otherwise, an empty one among them."""
    dtype, block, seqs = torch.bfloat16, 16, 40
    gen = torch.Generator().manual_seed(dim)
    new = [290] * seqs if lengths == "alike" else torch.randint(60, 450, (seqs,), generator=gen).tolist()
    prior = [0] * seqs if lengths == "alike" else torch.randint(0, 60, (seqs,), generator=gen).tolist()
    if lengths == "ragged":
        new[7] = 0
    args = paged_case(new, prior, block, 8, 4, dtype, seed=seqs, dim=dim)
    dev = [a.to(DEV) for a in args]
    assert paged_prefill_workspace_bytes(seqs, sum(new), 8, 4, dim, block, args[5].shape[1], dtype) == 0
    torch.full_like(dev[0], float("nan"))  # freed at once: the output's storage
    actual = paged_prefill_attention(*dev, block, validate=False).float().cpu()
    expected = paged_oracle.paged_prefill_attention(*args, block, cast=False)
    assert (actual - expected).abs().max().item() <= GATE[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tokens,start", [(64, 0), (65, 0), (1, 128), (130, 4300), (700, 33)])
def test_dense_tiles_and_windows(dtype, tokens, start):
    gen = torch.Generator().manual_seed(tokens + start)
    q = torch.randn(1, 8, tokens, 128, generator=gen).to(dtype)
    k = torch.randn(1, 4, start + tokens + 9, 128, generator=gen).to(dtype)
    v = torch.randn(1, 4, start + tokens + 9, 128, generator=gen).to(dtype)
    actual = prefill_attention(q.to(DEV), k.to(DEV), v.to(DEV), query_start=start).float().cpu()
    expected = paged_oracle.prefill_attention(q, k, v, query_start=start, cast=False)
    assert (actual - expected).abs().max().item() <= GATE[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("block", [4, 8, 16, 64, 256])
@pytest.mark.parametrize("new,prior,chunk,heads", [
    ([64, 1, 130], [0, 63, 64], 0, 14), ([40], [4400], 8192, 8), ([300, 77], [1200, 41], 256, 4),
])
def test_head_dim_64_tiles(dtype, block, new, prior, chunk, heads):
    """The 64-dim tile shape: whole and partial tiles, windows, key chunks,
    pages smaller and larger than a tile (4-token pages keep the padded
    shape), groups of 7, 4 and 2."""
    args = paged_case(new, prior, block, heads, 2, dtype, seed=block + sum(new), dim=64)
    actual = paged_prefill_attention(*[a.to(DEV) for a in args], block, chunk_tokens=chunk).float().cpu()
    expected = paged_oracle.paged_prefill_attention(*args, block, cast=False)
    assert (actual - expected).abs().max().item() <= GATE[dtype]


@pytest.mark.parametrize("batch,tokens,start,view", [(1, 130, 0, True), (2, 65, 4300, True), (1, 700, 33, False)])
def test_head_dim_64_dense(batch, tokens, start, view):
    dtype, gen = torch.bfloat16, torch.Generator().manual_seed(tokens)
    make = lambda n, h: torch.randn(batch, n, h, 64, generator=gen).to(dtype)  # noqa: E731
    q, k, v = make(tokens, 14), make(start + tokens, 2), make(start + tokens, 2)
    dev = [t.to(DEV).transpose(1, 2) for t in (q, k, v)]
    if not view:
        dev = [t.contiguous() for t in dev]
    actual = prefill_attention(*dev, query_start=start).float().cpu()
    expected = paged_oracle.prefill_attention(*[t.transpose(1, 2) for t in (q, k, v)], query_start=start, cast=False)
    assert (actual - expected).abs().max().item() <= GATE[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("mode", [8, 16, 32, 64, "dense"])
def test_scores_that_keep_rising(mode, dim, dtype):
    """Scores rise by 12 binary orders per tile of 64 keys, so that every tile exceeds
    the reference by more than 2^8: the sums and the output so far are rescaled again
    and again, and the last keys carry nearly all of the weight."""
    new, prior, heads, kv_heads, block = 200, 437, 4, 2, mode if mode != "dense" else 16
    q, kc, vc, cu, starts, tables, lens = paged_case([new], [prior], block, heads, kv_heads, dtype, seed=dim, dim=dim)
    q.copy_(0.5 + 0.02 * q.float())
    slope = 12 / 64 / (0.5 * dim ** 0.5 * math.log2(math.e))
    for i, page in enumerate(tables[0].tolist()):
        rows = (i * block + torch.arange(block)).float()[:, None, None]
        kc[page] = (0.02 * kc[page].float() + slope * rows).to(dtype)
    if mode == "dense":
        k, v = (c[tables[0]].flatten(0, 1)[:new + prior].transpose(0, 1).unsqueeze(0) for c in (kc, vc))
        views = (q.transpose(0, 1).unsqueeze(0), k, v)
        actual = prefill_attention(*[t.to(DEV) for t in views], query_start=prior).float().cpu()
        expected = paged_oracle.prefill_attention(*views, query_start=prior, cast=False)
    else:
        args = [q, kc, vc, cu, starts, tables, lens]
        actual = paged_prefill_attention(*[a.to(DEV) for a in args], block, chunk_tokens=1024).float().cpu()
        expected = paged_oracle.paged_prefill_attention(*args, block, cast=False)
    assert (actual - expected).abs().max().item() <= GATE[dtype]


def peaked_row(keys, dim):
    """One query whose first key has probability ~1 and the others 2^-25.2 each, below
    half of fp16's smallest number; V is 1 at the first key and 0 elsewhere.  Returns
    q [dim], K, V [keys, dim] and the exact output."""
    q, k, v = torch.zeros(dim), torch.zeros(keys, dim), torch.zeros(keys, dim)
    q[0], k[0, 0], v[0] = 16.0, 25.2 * math.log(2) * dim ** 0.5 / 16, 1.0
    q, k, v = q.half(), k.half(), v.half()
    exact = 1 / (1 + (keys - 1) * math.exp(-float(q[0]) * float(k[0, 0]) / dim ** 0.5))
    return q, k, v, exact


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("mode", [8, 32, "dense"])
def test_row_sums_hold_tiny_probabilities(mode, dim):
    """65535 keys of probability 2^-25.2 are 0.17 % of the row's sum, 3.5 spacings of
    fp16 below 1: sums of probabilities rounded to fp16 lose all of it.  The bound is
    half a spacing of the output and 1e-5 for the sum's own fp32 roundings."""
    keys = 65536
    q, k, v, exact = peaked_row(keys, dim)
    if mode == "dense":
        # 384 rows of work, so that keys are not split; every row reads the same keys.
        wide = [t.to(DEV)[None, None].expand(48, 8, keys, dim) for t in (k, v)]
        out = prefill_attention(q.to(DEV).expand(48, 8, 1, dim).contiguous(), *wide, query_start=keys - 1)
    else:
        pages = [t.to(DEV).view(keys // mode, mode, 1, dim) for t in (k, v)]
        meta = [[0, 1], [keys - 1], [list(range(keys // mode))], [keys]]
        out = paged_prefill_attention(q.to(DEV)[None, None], *pages, *[torch.tensor(m).to(DEV) for m in meta], mode,
                                      chunk_tokens=keys)
    assert (out.double() - exact).abs().max().item() <= 2.0 ** -12 + 1e-5
