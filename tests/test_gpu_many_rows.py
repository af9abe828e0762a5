"""The 16-byte kernels that the token ops of a packed group run on (many rows) against the
kernels that small batches run on: the same op on the same rows, once as one call and once in
calls of a few rows each, must give the same bits. The small calls are pinned to the
reference's tensor ops in ``test_gpu_epilogue.py``; every op here is row by row, so equality
is the whole contract. Rows of zeros, negative zeros and large values are among the inputs.
"""

from __future__ import annotations

import pytest
import torch

from miattn import PagedPool
from miattn.qwen3 import add_rms_norm, rope_table, silu_mul

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.view(torch.int16)


def _values(g, *shape, dtype, scale=1.0):
    t = (torch.randn(*shape, generator=g) * scale).to(dtype)
    flat = t.view(-1)
    flat[::97] = 0.0
    flat[5::193] = -0.0
    t[shape[0] // 2] = 0.0   # a whole row of zeros
    t[-1] *= 200.0
    return t.cuda()


# rows x heads x D from 2^20 values on take the 16-byte kernel; 1024 rows on, one workgroup per row
@pytest.mark.parametrize("rows,heads,rotary", [
    (260, (16, 8, 128), 128), (1025, (16, 8, 128), 64), (1030, (8, 2, 256), 64), (342, (8, 2, 256), 256),
    (1100, (4, 2, 256), 128), (900, (7, 7, 64), 64), (1300, (12, 3, 64), 64),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("zero_centred", [False, True], ids=["qwen3-norm", "qwen35-norm"])
def test_epilogue_of_many_rows_is_the_small_batches(rows, heads, rotary, dtype, zero_centred):
    H, H_kv, D = heads
    g = torch.Generator().manual_seed(rows)
    width = (H + 2 * H_kv) * D
    assert rows * width >= 1 << 20
    pad = 8 if rotary == 64 else 0  # a longer row stride, still 16-byte rows
    qkv = _values(g, rows, width + pad, dtype=dtype, scale=2.0)[:, :width]
    qn, kn = ((1.0 + 0.1 * torch.randn(D, generator=g)).to(dtype).cuda() for _ in range(2))
    cos, sin = rope_table(rotary, 1e6, 2048, "cuda", dtype)
    pos = torch.randint(0, 2048, (rows,), generator=g).cuda()
    n_blocks = rows // 16 + 2
    slots = torch.randperm(n_blocks * 16, generator=g)[:rows].to(torch.int32 if pad else torch.int64).cuda()
    slots[3] = -1                 # nothing to write
    slots[rows - 2] = n_blocks * 16  # refused: past the pool
    pos[7] = 2048                 # refused: past the RoPE table
    got, want = {}, {}
    for out, step in ((got, rows), (want, 50)):
        assert step == rows or step * width < 1 << 20
        pool = PagedPool(1, n_blocks, 16, H_kv, D, dtype=dtype, device="cuda", n_head=H)
        k, v = (torch.full((rows, H_kv, D), 9.0, dtype=dtype, device="cuda") for _ in range(2))
        q = []
        for a in range(0, rows, step):
            b = min(rows, a + step)
            q.append(pool.write_qk_norm_rope(0, slots[a:b], qkv[a:b], qn, kn, cos, sin, pos[a:b], 1e-6, k_out=k[a:b],
                                             v_out=v[a:b], rotary_dim=rotary, zero_centred_norm=zero_centred))
        torch.cuda.synchronize()
        out.update(q=torch.cat(q), k=k, v=v, keys=pool.keys[0], values=pool.values[0])
        with pytest.raises(IndexError):
            pool.check_writes()
    for name in got:
        assert torch.equal(_bits(got[name]), _bits(want[name])), name
    assert not got["q"][[3, 7, rows - 2]].any() and not got["k"][[3, 7, rows - 2]].any()


@pytest.mark.parametrize("rows,cols", [(256, 512), (259, 1024), (1001, 1536), (300, 2560), (257, 4096)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("with_delta", [True, False])
def test_add_rms_norm_of_many_rows_is_the_small_batches(rows, cols, dtype, with_delta):
    g = torch.Generator().manual_seed(rows + cols)
    x = _values(g, rows, cols, dtype=dtype)
    d = _values(g, rows, cols, dtype=dtype, scale=0.5) if with_delta else None
    w = (1.0 + 0.1 * torch.randn(cols, generator=g)).to(dtype).cuda()
    for eps in (1e-6, 0.0):  # eps 0: a row of zeros divides by zero, NaN in both
        xa, xb = x.clone(), x.clone()
        _, ha = add_rms_norm(xa, d, w, eps)
        hb = torch.cat([add_rms_norm(xb[a:a + 100], None if d is None else d[a:a + 100], w, eps)[1]
                        for a in range(0, rows, 100)])
        torch.cuda.synchronize()
        nan = torch.isnan(hb)
        assert torch.equal(_bits(xa), _bits(xb)) and torch.equal(nan, torch.isnan(ha))
        assert torch.equal(_bits(ha)[~nan], _bits(hb)[~nan]) and nan.any().item() == (eps == 0.0)


@pytest.mark.parametrize("rows,inter", [(512, 1024), (1001, 3072), (700, 1000), (600, 1004), (65537 // 8, 72)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_silu_mul_of_many_rows_is_the_small_batches(rows, inter, dtype):
    g = torch.Generator().manual_seed(rows)
    assert rows * inter >= 1 << 19
    gu = _values(g, rows, 2 * inter, dtype=dtype, scale=3.0)
    gu[0, :6] = torch.tensor([float("inf"), -float("inf"), -88.0, -90.0, 90.0, -100.0], dtype=dtype)
    a = silu_mul(gu)
    step = max(1, (1 << 18) // inter)
    b = torch.cat([silu_mul(gu[i:i + step]) for i in range(0, rows, step)])
    torch.cuda.synchronize()
    nan = torch.isnan(b)
    assert torch.equal(nan, torch.isnan(a)) and torch.equal(_bits(a)[~nan], _bits(b)[~nan])


BF16, FP16 = torch.bfloat16, torch.float16


def _epilogue_equals_small_batches(rows, heads, rotary, dtype, zero_centred, pad=None, shift=0):
    H, H_kv, D = heads
    g = torch.Generator().manual_seed(rows)
    width = (H + 2 * H_kv) * D
    assert rows * width >= 1 << 20
    if pad is None:
        pad = 8 if rotary == 64 else 0  # a longer row stride, still 16-byte rows
    qkv = _values(g, rows, width + pad, dtype=dtype, scale=2.0)[:, shift: shift + width]
    qn, kn = ((1.0 + 0.1 * torch.randn(D, generator=g)).to(dtype).cuda() for _ in range(2))
    cos, sin = rope_table(rotary, 1e6, 2048, "cuda", dtype)
    pos = torch.randint(0, 2048, (rows,), generator=g).cuda()
    n_blocks = rows // 16 + 2
    slots = torch.randperm(n_blocks * 16, generator=g)[:rows].to(torch.int32 if pad else torch.int64).cuda()
    slots[3] = -1                 # nothing to write
    slots[rows - 2] = n_blocks * 16  # refused: past the pool
    pos[7] = 2048                 # refused: past the RoPE table
    got, want = {}, {}
    for out, step in ((got, rows), (want, 50)):
        assert step == rows or step * width < 1 << 20
        pool = PagedPool(1, n_blocks, 16, H_kv, D, dtype=dtype, device="cuda", n_head=H)
        k, v = (torch.full((rows, H_kv, D), 9.0, dtype=dtype, device="cuda") for _ in range(2))
        q = []
        for a in range(0, rows, step):
            b = min(rows, a + step)
            q.append(pool.write_qk_norm_rope(0, slots[a:b], qkv[a:b], qn, kn, cos, sin, pos[a:b], 1e-6, k_out=k[a:b],
                                             v_out=v[a:b], rotary_dim=rotary, zero_centred_norm=zero_centred))
        torch.cuda.synchronize()
        out.update(q=torch.cat(q), k=k, v=v, keys=pool.keys[0], values=pool.values[0])
        with pytest.raises(IndexError):
            pool.check_writes()
    for name in got:
        assert torch.equal(_bits(got[name]), _bits(want[name])), name
    assert not got["q"][[3, 7, rows - 2]].any() and not got["k"][[3, 7, rows - 2]].any()


@pytest.mark.parametrize("rows,heads,rotary,dtype,zero_centred", [
    # just past the line of each head_dim, type and norm: the 16-byte kernel
    pytest.param(513, (16, 8, 128), 128, FP16, False, id="d128-fp16"),
    pytest.param(1040, (16, 8, 128), 64, FP16, True, id="d128-fp16-rows"),
    pytest.param(343, (16, 16, 64), 64, FP16, True, id="d64-fp16"),
    pytest.param(2049, (4, 2, 64), 64, BF16, False, id="d64-8-heads"),
    pytest.param(1025, (8, 2, 256), 64, BF16, False, id="d256"),
    pytest.param(5462, (8, 2, 256), 64, BF16, True, id="d256-qwen35-norm"),
    pytest.param(5500, (8, 2, 256), 256, BF16, True, id="d256-qwen35-norm-rot256"),
    pytest.param(10924, (8, 2, 256), 128, FP16, False, id="d256-fp16"),
    pytest.param(8193, (16, 8, 256), 64, FP16, True, id="d256-fp16-qwen35-norm"),
    # just below it, and too few heads: the older kernel in one call and in many
    pytest.param(511, (16, 8, 128), 128, FP16, False, id="d128-fp16-below"),
    pytest.param(5461, (8, 2, 256), 64, BF16, True, id="d256-qwen35-norm-below"),
    pytest.param(2100, (4, 2, 256), 64, BF16, False, id="d256-8-heads"),
    pytest.param(5500, (1, 1, 64), 64, BF16, False, id="d64-3-heads"),
])
def test_epilogue_around_each_line(rows, heads, rotary, dtype, zero_centred):
    _epilogue_equals_small_batches(rows, heads, rotary, dtype, zero_centred)


@pytest.mark.parametrize("pad,shift", [(8, 1), (4, 0), (1, 1), (16, 8)], ids=["pointer", "stride", "both", "aligned"])
@pytest.mark.parametrize("dtype", [BF16, FP16], ids=["bf16", "fp16"])
def test_epilogue_of_rows_off_16_bytes(pad, shift, dtype):
    """A projection whose pointer or row stride is no multiple of 16 bytes goes to the older kernel."""
    _epilogue_equals_small_batches(530, (16, 8, 128), 128, dtype, False, pad=pad, shift=shift)


def _shifted(t, shift):
    """``t`` in storage that begins ``shift`` elements past a 16-byte boundary."""
    flat = torch.empty(t.numel() + shift, dtype=t.dtype, device=t.device)[shift:]
    return flat.copy_(t.reshape(-1)).view(t.shape)


def _add_norm_equals_small_batches(rows, cols, dtype, with_delta, shifts=(0, 0, 0)):
    g = torch.Generator().manual_seed(rows + cols)
    x = _values(g, rows, cols, dtype=dtype)
    d = _shifted(_values(g, rows, cols, dtype=dtype, scale=0.5), shifts[1]) if with_delta else None
    w = _shifted((1.0 + 0.1 * torch.randn(cols, generator=g)).to(dtype).cuda(), shifts[2])
    xa, xb = _shifted(x, shifts[0]), x.clone()
    _, ha = add_rms_norm(xa, d, w, 1e-6)
    hb = torch.cat([add_rms_norm(xb[a:a + 100], None if d is None else d[a:a + 100], w, 1e-6)[1]
                    for a in range(0, rows, 100)])
    torch.cuda.synchronize()
    assert torch.equal(_bits(xa), _bits(xb)) and torch.equal(_bits(ha), _bits(hb))


@pytest.mark.parametrize("rows,cols,dtype,with_delta", [
    (1024, 512, FP16, True), (1027, 1024, FP16, True), (1025, 1536, FP16, True), (1030, 2048, FP16, True),
    (1025, 2560, FP16, False), (1024, 3072, FP16, False), (1024, 4096, FP16, False), (1027, 3584, FP16, False),
    (1030, 2560, FP16, True), (1023, 1024, FP16, True),                        # the older kernel
    (321, 2048, BF16, False), (257, 2048, BF16, True), (258, 3072, BF16, True), (259, 3584, BF16, True),
    (300, 1000, BF16, True), (400, 2568, BF16, True), (2000, 1000, FP16, True),  # no multiple of 512
])
def test_add_rms_norm_around_each_line(rows, cols, dtype, with_delta):
    _add_norm_equals_small_batches(rows, cols, dtype, with_delta)


@pytest.mark.parametrize("shifts", [(1, 0, 0), (0, 1, 0), (0, 0, 1), (4, 4, 4), (8, 8, 8)])
@pytest.mark.parametrize("dtype", [BF16, FP16], ids=["bf16", "fp16"])
def test_add_rms_norm_off_16_bytes(shifts, dtype):
    _add_norm_equals_small_batches(1030, 1024, dtype, True, shifts)


@pytest.mark.parametrize("rows,inter,shift", [
    (2100, 1024, 0), (1001, 3072, 0), (820, 2560, 0), (5500, 384, 0), (260, 8200, 0), (2731, 776, 0), (1366, 1544, 0),
    (5700, 376, 0), (2100, 1004, 0),                       # narrow, or no multiple of 8
    (2100, 1024, 1), (2100, 1024, 4), (2100, 1024, 8),     # off 16 bytes, and on them again
])
@pytest.mark.parametrize("dtype", [BF16, FP16], ids=["bf16", "fp16"])
def test_silu_mul_around_each_line(rows, inter, shift, dtype):
    g = torch.Generator().manual_seed(rows)
    assert rows * inter >= 1 << 21
    gu = _shifted(_values(g, rows, 2 * inter, dtype=dtype, scale=3.0), shift)
    step = max(1, (1 << 18) // inter)
    a, b = silu_mul(gu), torch.cat([silu_mul(gu[i:i + step].clone()) for i in range(0, rows, step)])
    torch.cuda.synchronize()
    assert torch.equal(_bits(a), _bits(b))
