"""Which decode calls the plan gives the balanced walk, and what it computes
there: unit counts around the CUs' number and its multiples, capacities on
both sides of each line, and workspaces that do not hold the walk's partials.
Tolerance: the decode gate against the fp32 oracle."""

import pytest
import torch

from gpu_cases import decode_inputs
from mini_engine_hip.kernels import hip_extension as ext
from mini_engine_hip.kernels.paged import paged_attention
from oracle import paged_oracle

DEV = "cuda"
GATE = 1.6e-2


def walk_bytes(gtile, dim=128):
    return 256 * 2 * gtile * (dim + 2) * 4 + 256 * 32


@pytest.mark.parametrize("batch,walks_from", [
    (8, 4096), (12, 2560), (29, 2560), (30, 2560), (32, 2560), (33, 1024), (40, 1024), (41, 2048), (48, 2048),
    (49, 3072), (60, 3072), (61, None), (64, None),
])
def test_lines_of_the_walk(batch, walks_from):
    lib = ext.load_hip_extension()
    size = lambda cap, part=0: lib.workspace_size(batch, 16, 8, 128, 16, cap // 16, part)
    walk = size(4096, -1)
    assert walk == size(64, -1) > 0
    if walks_from is None:
        assert size(1 << 20) != walk
        return
    assert size(walks_from) == walk and size(walks_from * 2) == walk
    assert size(walks_from - 16) != walk


@pytest.mark.parametrize("heads,kv_heads,batch,walks_from", [
    (8, 8, 34, 1024), (32, 8, 34, 1024), (40, 8, 32, 3072), (40, 8, 40, 4096), (40, 8, 49, None), (28, 4, 62, 3072),
])
def test_lines_of_the_walk_by_group(heads, kv_heads, batch, walks_from):
    lib = ext.load_hip_extension()
    size = lambda cap, part=0: lib.workspace_size(batch, heads, kv_heads, 128, 16, cap // 16, part)
    walk = size(4096, -1)
    if walks_from is None:
        assert size(1 << 19) != walk
    else:
        assert size(walks_from) == walk and size(walks_from - 16) != walk


def test_other_head_dims_keep_their_lines():
    lib = ext.load_hip_extension()
    for dim in (64, 256):
        size = lambda batch, cap: lib.workspace_size(batch, 16, 8, dim, 16, cap // 16, 0)
        line = (2 << 20) // (4 * dim)
        assert size(32, line - 16) == 0 < size(32, line)
        assert size(33, line) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("batch,cap", [(33, 1024), (40, 1040), (48, 2048), (12, 2560), (32, 2576)])
def test_walk_with_more_units_than_shares(batch, cap):
    gen = torch.Generator().manual_seed(batch)
    lengths = torch.randint(0, 200, (batch,), generator=gen).tolist()
    lengths[batch // 2], lengths[0], lengths[-1] = cap, 1, cap - 1
    print(f"walk: {batch} sequences, capacity {cap}", flush=True)
    args = decode_inputs(torch.bfloat16, lengths=lengths, seed=cap)
    q, k, v, table, lens, block = [a.to(DEV) if isinstance(a, torch.Tensor) else a for a in args]
    lib = ext.load_hip_extension()
    shape = (batch, 16, 8, 128, block, table.shape[1], 0)
    need = lib.workspace_size(*shape)
    assert need == lib.workspace_size(*shape[:-1], -1)
    expected = paged_oracle.fp32_oracle(dict(zip(paged_oracle.TENSOR_NAMES, args[:5])), block)
    actual = paged_attention(q, k, v, table, lens, block)
    assert (actual.float().cpu() - expected).abs().max().item() <= GATE
    assert torch.equal(actual, paged_attention(q, k, v, table, lens, block, partition_tokens=-1))

    # A workspace of the right size off a 16-byte boundary, and none: the
    # plan without the walk (split-K for 12 sequences, which needs its own).
    room = torch.empty(need + (8 << 20), dtype=torch.uint8, device=DEV)
    for pointer, size in ((room.data_ptr() + 4, room.numel() - 4), (None, 0)):
        out = torch.full_like(q, float("nan"))
        call = lambda: lib.call("mvme_paged_attention", out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                table.data_ptr(), lens.data_ptr(), batch, 16, 8, 128, k.shape[0], block,
                                table.shape[1], 0, ext.BF16, pointer, size, ext.current_stream(q.device))
        if batch == 12 and size == 0:
            with pytest.raises(Exception, match="workspace"):
                call()
            continue
        call()
        assert (out.float().cpu() - expected).abs().max().item() <= GATE
