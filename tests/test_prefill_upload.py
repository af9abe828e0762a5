"""``PackedPrefill.upload`` (one host-built upload per group) against the container built from its
parts: same positions, slots, offsets and claims, and the same refusals."""

from __future__ import annotations

import pytest
import torch

from miattn import PackedPrefill, PagedPool, PagedWriteSink


def _parts(pool, prompts, tables):
    cu = [0]
    for p in prompts:
        cu.append(cu[-1] + len(p))
    return PackedPrefill(cu_seqlens=cu, positions=torch.cat([torch.arange(len(p)) for p in prompts]),
                         sinks=[PagedWriteSink(pool, t, len(p)) for t, p in zip(tables, prompts)])


@pytest.mark.parametrize("lengths", [[1], [16], [17, 1, 33], [5, 48, 16, 15]])
def test_upload_equals_the_parts(lengths):
    pool = PagedPool(2, 32, 16, 2, 8)
    perm = torch.randperm(32, generator=torch.Generator().manual_seed(1)).tolist()
    prompts = [tuple(range(100 * i, 100 * i + n)) for i, n in enumerate(lengths)]
    tables = [[perm.pop() for _ in range(-(-n // 16) + 1)] for n in lengths]
    got, tokens = PackedPrefill.upload(prompts, pool, tables, torch.device("cpu"))
    want = _parts(pool, prompts, tables)
    assert tokens.tolist() == [t for p in prompts for t in p] and tokens.dtype == torch.int64
    for name in ("positions", "last_token_index", "group_slots"):
        a, b = getattr(got, name), getattr(want, name)
        assert torch.equal(a, b) and a.dtype == b.dtype, name
    for name in ("cu_seqlens", "total_tokens", "n_seqs", "max_seqlen", "rope_len"):
        assert getattr(got, name) == getattr(want, name), name
    assert all(torch.equal(a.slots, b.slots) and a.block_table == b.block_table for a, b in zip(got.sinks, want.sinks))
    k, v = torch.randn(2, 1, sum(lengths), 2, 8)
    got.write(1, k, v)
    with pytest.raises(RuntimeError, match="already written"):
        got.write(1, k, v)


def test_upload_refuses_what_the_parts_refuse():
    pool = PagedPool(1, 4, 16, 2, 8)
    dev = torch.device("cpu")
    for prompts, tables, error in (([[1, 2]], [[9]], IndexError), ([[1] * 17], [[0]], IndexError),
                                   ([[1], [2]], [[0]], ValueError), ([[1], []], [[0], [1]], ValueError),
                                   ([], [], ValueError), ([[1]], [[True]], ValueError),
                                   ([["1", "2"]], [[0]], ValueError), (["12"], [[0]], ValueError)):
        with pytest.raises(error):
            PackedPrefill.upload(prompts, pool, tables, dev)


@pytest.mark.parametrize("prompts", [[[[5]]], [[[5], [6]]], [[[5, 6]]]])
def test_upload_refuses_nested_tokens(prompts):
    """Refused by the packed tensor's shape before, one token or several."""
    with pytest.raises(ValueError):
        PackedPrefill.upload(prompts, PagedPool(1, 4, 16, 2, 8), [[0]], torch.device("cpu"))
