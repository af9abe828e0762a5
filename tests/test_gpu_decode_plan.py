"""The decode's device-side split plan at the sizes where it changes its mind: the batch's
token total around the point from which splits have a floor, rows around 32 batches, ragged
batches whose partial splits overflow the workgroups aimed for (the split size is then fitted),
64 and 65 rows (fitted or not), head layouts with one or several workgroup columns and with 4
query heads per lane around 96-token splits, and rows short enough for the one-launch kernel.

Each result is held to the fp32 gather oracle within 2e-2 and, beyond its own 16-bit rounding
(2^-8 relative for bf16), within 1e-3, the bars of ``test_gpu_decode.py``: a plan that drops,
repeats or misplaces a split misses them by orders of magnitude. The plan must not depend on
anything but the row lengths, and the one-launch kernel is the two launches' equal bit for bit:
the same rows through a wider table give the same bits.
"""

from __future__ import annotations

import pytest
import torch

from miattn import _lib, paged_decode, paged_decode_plan
from oracle.decode import reference_paged_decode

pytestmark = pytest.mark.gpu

BS = 16


def _build(lengths, H, H_kv, D, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    pages = [-(-n // BS) for n in lengths]
    n_blocks = sum(pages) + 3
    k, v = (torch.randn(n_blocks, BS, H_kv, D, generator=g).to(dtype) for _ in range(2))
    q = torch.randn(len(lengths), H, D, generator=g).to(dtype)
    perm = torch.randperm(n_blocks, generator=g).to(torch.int32)
    table = torch.zeros(len(lengths), max(max(pages), 1), dtype=torch.int32)
    at = 0
    for r, n in enumerate(pages):
        table[r, :n] = perm[at:at + n]
        at += n
    return q, k, v, table, torch.tensor(lengths, dtype=torch.int32)


def _ragged(n, lo, hi, seed):
    return torch.randint(lo, hi + 1, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


QWEN3 = (16, 8, 128)
CASES = [
    pytest.param([1023], QWEN3, id="one-row-1023"),
    pytest.param([1024], QWEN3, id="one-row-1024"),
    pytest.param([1025], QWEN3, id="one-row-1025"),
    pytest.param([256, 100], QWEN3, id="32-batches"),
    pytest.param([257, 100], QWEN3, id="past-32-batches"),
    pytest.param([512, 500, 12], QWEN3, id="total-1024"),
    pytest.param([512, 501, 12], QWEN3, id="total-1025"),
    pytest.param(_ragged(32, 128, 2048, 5), QWEN3, id="ragged-32"),
    pytest.param(_ragged(64, 1, 700, 6), QWEN3, id="ragged-64"),
    pytest.param(_ragged(65, 1, 700, 7), QWEN3, id="ragged-65"),
    pytest.param([0] * 20 + [1] * 40 + [3000, 0, 2500, 1], QWEN3, id="mostly-short"),
    pytest.param([8192] + [17] * 31, QWEN3, id="one-long"),
    pytest.param(_ragged(33, 1, 900, 8), (32, 16, 128), id="two-columns"),
    pytest.param(_ragged(16, 100, 1500, 9), (32, 4, 128), id="head-chunks"),
    pytest.param(_ragged(30, 1, 1200, 10), (16, 16, 64), id="d64"),
    pytest.param([2048] * 12, (8, 2, 256), id="4-heads-96-tokens"),
    pytest.param([2048] * 12 + [9], (8, 2, 256), id="4-heads-past-96-tokens"),
    pytest.param(_ragged(16, 128, 2048, 11), (8, 2, 256), id="4-heads-ragged"),
    pytest.param(_ragged(9, 1, 300, 12), (10, 5, 128), id="five-columns"),
    # short rows: one launch (table width at most 32 batches)
    pytest.param([1], QWEN3, id="short-1"),
    pytest.param([8, 9, 0, 7, 16, 17], QWEN3, id="short-batch-edges"),
    pytest.param([256, 255, 249, 248, 241, 1], QWEN3, id="short-all-32-splits"),
    pytest.param(_ragged(32, 0, 256, 13), QWEN3, id="short-32-rows"),
    pytest.param([250] * 32, QWEN3, id="short-longer-splits"),
    pytest.param(_ragged(33, 1, 200, 14), QWEN3, id="short-too-many-rows"),
    pytest.param(_ragged(5, 1, 256, 15), (8, 8, 128), id="short-mha"),
    pytest.param(_ragged(20, 1, 256, 16), (16, 16, 64), id="short-d64"),
    pytest.param(_ragged(20, 1, 128, 17), (32, 16, 128), id="short-one-token-loads"),
    pytest.param(_ragged(3, 1, 128, 18), (32, 32, 64), id="short-d64-one-token-loads"),
    pytest.param(_ragged(6, 1, 250, 19), (48, 8, 128), id="short-head-chunks"),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("lengths,heads", CASES)
def test_split_plan_edges(lengths, heads, dtype, cuda):
    H, H_kv, D = heads
    q, k, v, table, seqlen = _build(lengths, H, H_kv, D, dtype, seed=len(lengths))
    want = reference_paged_decode(q, k, v, table, seqlen, out_dtype=torch.float32)
    dev = [t.to(cuda) for t in (q, k, v, table, seqlen)]
    got = paged_decode(*dev)
    # past the short-row kernel's table width: the same rows through the split and merge launches
    wide = torch.cat([dev[3], torch.full((len(lengths), 17), -999, dtype=torch.int32, device=cuda)], 1)
    again = paged_decode(dev[0], dev[1], dev[2], wide, dev[4])
    torch.cuda.synchronize()
    assert torch.equal(got, again)
    diff = (got.cpu().float() - want).abs()
    assert diff.max().item() <= 2e-2
    assert (diff - want.abs() * 2.0 ** -8).max().item() <= 1e-3
    assert not got[seqlen == 0].any()


@pytest.mark.parametrize("lengths", [
    pytest.param([13, 16, 17], id="2-3-splits"),
    pytest.param([120, 121, 128, 129], id="15-17-splits"),
    pytest.param([256, 249], id="32-splits"),
    pytest.param([257, 511], id="17-32-splits-of-16"),
    pytest.param([528, 8], id="33-splits"),
    pytest.param([1, 0, 9, 500], id="mixed"),
])
@pytest.mark.parametrize("heads", [QWEN3, (16, 16, 64), (8, 2, 256), (4, 2, 32)], ids=["d128", "d64", "d256", "d32"])
def test_merge_of_few_and_many_splits(lengths, heads, cuda):
    """Rows whose split counts lie around the widths that the merge folds at once (16, 32), through
    a table wide enough that the one-launch kernel does not take them."""
    H, H_kv, D = heads
    q, k, v, table, seqlen = _build(lengths, H, H_kv, D, torch.bfloat16, seed=sum(lengths))
    want = reference_paged_decode(q, k, v, table, seqlen, out_dtype=torch.float32)
    wide = torch.cat([table, torch.full((len(lengths), 17), -999, dtype=torch.int32)], 1)
    got = paged_decode(*(t.to(cuda) for t in (q, k, v, wide, seqlen))).cpu()
    diff = (got.float() - want).abs()
    assert diff.max().item() <= 2e-2
    assert (diff - want.abs() * 2.0 ** -8).max().item() <= 1e-3
    assert not got[seqlen == 0].any()


def _split_counts(lengths, heads, width=None):
    """Splits per row, from the (first slot, split count) records that the split launch leaves for the
    merge at the start of the workspace. Every table entry names one of a few pages, so that long
    batches cost no memory."""
    H, H_kv, D = heads
    B, width = len(lengths), width or -(-max(lengths) // BS)
    g = torch.Generator().manual_seed(B)
    k, v = (torch.randn(4, BS, H_kv, D, generator=g).bfloat16().cuda() for _ in range(2))
    q = torch.randn(B, H, D, generator=g).bfloat16().cuda()
    table = torch.randint(0, 4, (B, width), generator=g, dtype=torch.int32).cuda()
    seqlen = torch.tensor(lengths, dtype=torch.int32, device="cuda")
    out = torch.empty_like(q)
    code = _lib.dtype_code(q.dtype)
    n = _lib.lib.mi_paged_decode_workspace_size(B, H, H_kv, D, BS, width, code)
    ws = torch.full((n,), 0xff, dtype=torch.uint8, device="cuda")
    rc = _lib.lib.mi_paged_decode(q.data_ptr(), k.data_ptr(), v.data_ptr(), table.data_ptr(), seqlen.data_ptr(),
                                  out.data_ptr(), B, H, H_kv, D, BS, width,
                                  _lib.int64_array((*q.stride(), *k.stride(), *v.stride(), *out.stride(), width)),
                                  D ** -0.5, code, ws.data_ptr(), n, _lib.current_stream(q.device))
    _lib.check(rc, "mi_paged_decode")
    torch.cuda.synchronize()
    some = [0, B // 2, B - 1]
    want = reference_paged_decode(q[some].cpu(), k.cpu(), v.cpu(), table[some].cpu(), seqlen[some].cpu(),
                                  out_dtype=torch.float32)
    assert (out[some].cpu().float() - want).abs().max().item() <= 2e-2
    return ws[: 8 * B].view(torch.int32).view(B, 2).cpu()


@pytest.mark.parametrize("heads,most", [(QWEN3, 256), ((16, 16, 64), 256), ((32, 4, 128), 256), ((8, 2, 256), 512)],
                         ids=["d128", "d64", "head-chunks", "d256"])
@pytest.mark.parametrize("lengths", [
    pytest.param([8192] * 44, id="44x8192"), pytest.param([4096] * 52, id="52x4096"),
    pytest.param([8192] * 64, id="64x8192"), pytest.param(_ragged(64, 4096, 8192, 20), id="64-ragged"),
    pytest.param(_ragged(60, 4096, 8192, 21), id="60-ragged"), pytest.param(_ragged(33, 1, 8192, 22), id="33-ragged"),
    pytest.param([30000] + [5000] * 20, id="one-long"),
])
def test_splits_of_long_batches_fit_the_workgroups(lengths, heads, most, cuda):
    """However long the rows of up to 64 requests are, their splits fit the workgroups aimed for: one
    workgroup too many puts a second one on a CU that the whole launch then waits for."""
    first, count = _split_counts(lengths, heads).unbind(1)
    assert count.sum().item() <= most
    assert torch.equal(first, count.cumsum(0).int() - count) and count.min().item() >= 1


@pytest.mark.parametrize("lengths,heads,one_launch", [
    pytest.param([192], QWEN3, True, id="192"), pytest.param([193], QWEN3, False, id="193"),
    pytest.param([256, 40, 7, 250, 99, 1, 80, 200], QWEN3, False, id="8-of-256"),
    pytest.param([192] * 32, QWEN3, True, id="32-of-192"), pytest.param([100] * 33, QWEN3, False, id="too-many-rows"),
    pytest.param([256], (16, 16, 64), True, id="d64-256"), pytest.param([257], (16, 16, 64), False, id="d64-257"),
    pytest.param([128], (32, 16, 128), True, id="4-token-batches-128"),
    pytest.param([129], (32, 16, 128), False, id="4-token-batches-129"),
    pytest.param([160] * 2, (40, 8, 128), True, id="5-chunks-160"),
    pytest.param([161] * 2, (40, 8, 128), False, id="5-chunks-161"),
])
def test_one_launch_only_where_it_is_the_faster(lengths, heads, one_launch, cuda):
    """The one-launch kernel leaves no records in the workspace; past its range (tables of more than
    24576 K elements per row) the two launches run."""
    records = _split_counts(lengths, heads)
    assert (records == -1).all().item() if one_launch else (records >= 0).all().item()


@pytest.mark.parametrize("heads,lengths,least,most", [
    # two workgroup columns: all of the workgroups, fitted
    pytest.param((32, 32, 128), [2048] * 8, 256, 256, id="2-groups"),
    pytest.param((32, 32, 128), _ragged(20, 1000, 4000, 30), 200, 256, id="2-groups-ragged"),
    pytest.param((16, 16, 256), [300] * 12, 180, 256, id="2-groups-d256"),
    # more: as they come, 512 / columns of them and a partial split per row
    pytest.param((12, 12, 128), [2048] * 8, 140, 178, id="3-groups"),
    pytest.param((40, 8, 128), [400] * 8, 104, 104, id="5-chunks"),
    pytest.param((10, 5, 128), [1000] * 10, 80, 80, id="5-groups"),
    # half the workgroups up to fitted splits of so many batches, all of them past it: four heads per
    # lane at D 256 (12 of 8 tokens) and at D 128 (24 of 4 tokens), page ids per lane (8 of 32; 3 of 32)
    pytest.param((8, 2, 256), [1536] * 16, 256, 256, id="d256-12-batches"),
    pytest.param((8, 2, 256), [2048] * 12, 400, 512, id="d256-fitted-past-12"),
    pytest.param((32, 8, 128), [768] * 32, 256, 256, id="gqa4-24-batches"),
    pytest.param((32, 8, 128), [800] * 32, 400, 512, id="gqa4-past-24"),
    pytest.param((4, 1, 128), [2048] * 32, 256, 256, id="one-kv-head-8-batches"),
    pytest.param((4, 1, 128), [2100] * 32, 400, 512, id="one-kv-head-past-8"),
    pytest.param((2, 2, 128), [1536] * 16, 256, 256, id="two-kv-heads-3-batches"),
    pytest.param((2, 2, 128), [1600] * 16, 400, 512, id="two-kv-heads-past-3"),
])
def test_workgroups_aimed_for(heads, lengths, least, most, cuda):
    """How many of the workgroups a batch's splits are shared out over, by the columns of workgroups
    that its heads need."""
    assert least <= _split_counts(lengths, heads)[:, 1].sum().item() <= most


@pytest.mark.parametrize("heads,lengths,splits", [
    # 8-token batches: rows of up to 32 of them are cut by the workgroups alone
    pytest.param(QWEN3, [256] * 8, [32] * 8, id="32-batches"),
    pytest.param(QWEN3, [256] * 7 + [257], [11] * 8, id="past-32-batches"),
    pytest.param(QWEN3, [300], [19], id="tiny"), pytest.param(QWEN3, [1024], [64], id="tiny-edge"),
    pytest.param(QWEN3, [1025], [43], id="past-tiny"),
    pytest.param((8, 2, 256), [200] * 6, [25] * 6, id="4-heads"), pytest.param((8, 2, 256), [400] * 3, [17] * 3, id="4-heads-long"),
    # 4-token batches: floors of two and three of them
    pytest.param((32, 16, 128), [200], [25], id="4-token-batches"),
    pytest.param((32, 16, 128), [160] * 7, [14] * 7, id="4-token-batches-past-tiny"),
    pytest.param((32, 16, 128), [120] * 10, [15] * 10, id="4-token-batches-short"),
    pytest.param((32, 8, 128), [130, 100], [17, 13], id="4-token-batches-4-heads"),
    pytest.param((8, 1, 128), [16], [1], id="one-batch"),
])
def test_split_floors(heads, lengths, splits, cuda):
    """Splits per row around the lines of the floors (a table wide enough for the two launches)."""
    width = max(33, -(-max(lengths) // BS))
    assert _split_counts(lengths, heads, width)[:, 1].tolist() == splits


def _other_pools(k, v, table, seqlen, block, head_major):
    """The same rows over pools of another page size, each page's tokens moved, and of another layout."""
    lengths, H_kv, D = seqlen.tolist(), k.shape[2], k.shape[3]
    need = [max(1, -(-n // block)) for n in lengths]
    n_blocks = sum(need) + 2
    k2, v2 = (torch.full((n_blocks, block, H_kv, D), 7.0, dtype=k.dtype) for _ in range(2))
    table2 = torch.zeros(len(lengths), max(need), dtype=torch.int32)
    ids = torch.randperm(n_blocks, generator=torch.Generator().manual_seed(block)).tolist()
    for r, n in enumerate(lengths):
        for page in range(need[r]):
            table2[r, page] = ids.pop()
        for old, new in ((k, k2), (v, v2)):
            row = old[table[r].long()].reshape(-1, H_kv, D)[:n]
            for page in range(-(-n // block)):
                part = row[page * block:(page + 1) * block]
                new[int(table2[r, page]), : len(part)] = part
    if head_major:
        k2, v2 = (t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) for t in (k2, v2))
    return k2.cuda(), v2.cuda(), table2.cuda()


@pytest.mark.parametrize("head_major", [False, True], ids=["token-major", "head-major"])
@pytest.mark.parametrize("block", [1, 4, 16, 32, 64])
@pytest.mark.parametrize("heads,lengths", [
    pytest.param(QWEN3, [1, 0, 150, 64, 33, 97, 128], id="d128"),
    pytest.param((16, 16, 64), [1, 150, 190, 64, 0, 65], id="d64"),
    pytest.param((32, 16, 128), [1, 100, 64, 0, 128], id="4-token-batches"),
    pytest.param((48, 8, 128), [128, 5, 77], id="head-chunks"),
])
def test_one_launch_of_other_pages_and_layouts(heads, lengths, block, head_major, cuda):
    H, H_kv, D = heads
    q, k, v, table, seqlen = _build(lengths, H, H_kv, D, torch.bfloat16, seed=sum(lengths))
    ref = paged_decode(*(t.cuda() for t in (q, k, v)), torch.cat(
        [table, torch.full((len(lengths), 17), -999, dtype=torch.int32)], 1).cuda(), seqlen.cuda())  # two launches
    k2, v2, table2 = _other_pools(k, v, table, seqlen, block, head_major)
    assert block * table2.shape[1] * D <= 24576
    got = paged_decode(q.cuda(), k2, v2, table2, seqlen.cuda())
    torch.cuda.synchronize()
    assert torch.equal(got, ref)
    want = reference_paged_decode(q, k, v, table, seqlen, out_dtype=torch.float32)
    assert (got.cpu().float() - want).abs().max().item() <= 2e-2


def test_one_launch_in_a_graph_whose_rows_grow(cuda):
    """A captured call reads the row lengths at each replay: rows grow, start and end between replays."""
    H, H_kv, D = QWEN3
    q, k, v, table, _ = _build([192] * 6, H, H_kv, D, torch.bfloat16, seed=5)
    q, k, v, table = (t.cuda() for t in (q, k, v, table))
    wide = torch.cat([table, torch.full((6, 17), -999, dtype=torch.int32, device=cuda)], 1)
    seqlen = torch.tensor([1, 8, 0, 100, 16, 191], dtype=torch.int32, device=cuda)
    plan = paged_decode_plan(q, [k], [v], table, seqlen)
    plan.run(0, q)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = plan.run(0, q)
    for step, lengths in enumerate([[1, 8, 0, 100, 16, 191], [2, 9, 1, 101, 17, 192], [8, 16, 64, 128, 24, 0],
                                    [0, 0, 0, 0, 0, 0], [192] * 6, [192, 1, 1, 1, 1, 1]]):
        seqlen.copy_(torch.tensor(lengths, dtype=torch.int32))
        out.fill_(9.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, paged_decode(q, k, v, wide, seqlen)), step
        assert not out[seqlen == 0].any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("lengths,heads", [
    pytest.param([192, 191, 185, 184, 177, 1], QWEN3, id="24-splits"),
    pytest.param([190] * 32, QWEN3, id="32-rows-longer-splits"), pytest.param(_ragged(32, 0, 192, 40), QWEN3, id="32-ragged"),
    pytest.param([256, 255, 249, 1], (16, 16, 64), id="d64-32-splits"),
    pytest.param([128, 127, 125, 124, 1], (32, 16, 128), id="4-token-batches-32-splits"),
    pytest.param([160, 33], (40, 8, 128), id="5-chunks"), pytest.param(_ragged(7, 1, 192, 41), (8, 8, 128), id="one-head"),
])
def test_one_launch_up_to_its_widest_table(lengths, heads, dtype, cuda):
    test_split_plan_edges(lengths, heads, dtype, cuda)
