"""The work that a user of this package has it do, as cases that can be timed and compared.

Every case is one pass through public entry points of ``miattn``, at sizes taken from the
package's own workload configurations (``miattn/workloads.py``), tests and benchmark, or
generic ones. ``listed()`` names the cases, ``draw(rng)`` gives one more of the same ranges,
``prepare`` / ``run`` / ``work`` / ``tolerance`` / ``exact`` say what a case holds, does, cannot
do without, may differ by, and computes in 64 bits.

Kinds of case:

* ``decode``   -- one decode step's paged attention, every layer of it: ``PagedDecodePlan.run``
  per layer, called one by one or replayed from a HIP graph that the program captured once;
* ``prefill``  -- packed causal prefill attention of a group of prompts, a few layer calls of
  ``backend_for(device).prefill_varlen``;
* ``write``    -- a packed group's K and V scattered into the paged pool, ``PagedPool.write_slots``
  per layer;
* ``tokenops`` -- what one block of a packed prefill does beside its projections and its attention:
  input norm, q/k norm + RoPE + K/V write, residual add + norm twice, SiLU(gate) * up;
* ``seats``    -- one greedy decode step of a whole model, every seat of a serving batch, replayed
  from its captured graph (``SeatDecoder``);
* ``model``    -- a whole model's packed prefill of a group of prompts, to its logits (``Qwen3.prefill``).
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "llm-serving_amd"))  # the package's folder below the repository's root

from miattn import PagedPool, backend_for, paged_decode_plan  # noqa: E402
from miattn.qwen3 import Qwen3, Qwen3Config, add_rms_norm, rope_table, silu_mul  # noqa: E402
from miattn.serve import SeatDecoder  # noqa: E402

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
EPS = 1e-6
BLOCK = 16

# 8 prompts, lognormal(median 512, sigma 0.6) clipped to [64, 2048]: the lengths that the benchmark's
# packed group has
GROUP = "1742,110,658,364,390,450,152,445"


def listed():
    qwen3 = {"H": 16, "H_kv": 8, "D": 128}
    wide = {"H": 8, "H_kv": 2, "D": 256}
    return [
        # one user's chat: a single short row, the smallest step, where latency is all there is
        {"name": "decode_one_row", "kind": "decode", "B": 1, "lo": 300, "hi": 300, "block": 16, "layers": 28,
         "dtype": "bf16", "graph": False, **qwen3},
        # a few users at an even length (8 rows of 512 tokens), the step replayed from a graph
        {"name": "decode_small_batch", "kind": "decode", "B": 8, "lo": 512, "hi": 512, "block": 16, "layers": 28,
         "dtype": "bf16", "graph": True, **qwen3},
        # the ordinary serving batch: 32 ragged rows of 128 to 2048 tokens
        {"name": "decode_ragged_batch", "kind": "decode", "B": 32, "lo": 128, "hi": 2048, "block": 16, "layers": 28,
         "dtype": "bf16", "graph": True, **qwen3},
        # long documents: 32 rows of 8192 tokens, the most bytes a step here reads
        {"name": "decode_long_rows", "kind": "decode", "B": 32, "lo": 8192, "hi": 8192, "block": 16, "layers": 4,
         "dtype": "bf16", "graph": False, **qwen3},
        # the other attention shape in use (four query heads per KV head, head_dim 256), fp16, pages of 32
        {"name": "decode_wide_heads", "kind": "decode", "B": 16, "lo": 128, "hi": 2048, "block": 32, "layers": 28,
         "dtype": "fp16", "graph": True, **wide},
        # attention of an admitted group of ragged prompts
        {"name": "prefill_group", "kind": "prefill", "lengths": GROUP, "layers": 4, "dtype": "bf16", **qwen3},
        {"name": "prefill_group_wide_heads", "kind": "prefill", "lengths": GROUP, "layers": 4, "dtype": "bf16", **wide},
        # attention of one long prompt
        {"name": "prefill_long_prompt", "kind": "prefill", "lengths": "8192", "layers": 2, "dtype": "bf16", **qwen3},
        # the same group's K and V into the pool
        {"name": "write_group", "kind": "write", "lengths": GROUP, "layers": 8, "dtype": "bf16", "pages": 4096, **qwen3},
        # the block's other ops over a group that fills the server's prefill budget (8192 tokens)
        {"name": "tokenops_full_group", "kind": "tokenops", "lengths": "3001,1700,2048,903,540", "dtype": "bf16",
         "hidden": 1024, "inter": 3072, **qwen3},
        # the whole greedy step of 32 seats near 2048 tokens of context, at 8 layers: 16-bit roundings,
        # op by op, travel through every layer, and after 14 of them the residual stream is already
        # 3.4e-2 from its 64-bit value, too far to be compared
        {"name": "seats_step", "kind": "seats", "S": 32, "lo": 1920, "hi": 2047, "layers": 8},
        # the whole prefill of an admitted group
        {"name": "model_prefill_group", "kind": "model", "lengths": GROUP, "layers": 28},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _some_lengths(rng, most_prompts, hi, most_tokens):
    n = rng.randint(1, most_prompts)
    got = []
    for _ in range(n):
        k = _log_int(rng, 1 if rng.random() < 0.15 else 24, hi)
        if sum(got) + k > most_tokens:
            break
        got.append(k)
    return ",".join(str(k) for k in got or [hi])


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "write", "tokenops", "seats", "model"])
    heads = rng.choice([{"H": 16, "H_kv": 8, "D": 128}, {"H": 16, "H_kv": 8, "D": 128}, {"H": 8, "H_kv": 2, "D": 256},
                        {"H": 32, "H_kv": 4, "D": 128}, {"H": 16, "H_kv": 16, "D": 64}])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "decode":
        B, hi = _log_int(rng, 1, 64), _log_int(rng, 20, 8192)
        lo = max(1, int(hi * rng.choice([0.06, 0.5, 1.0])))
        while B * hi > 32 * 8192:
            B = max(1, B // 2)
        if rng.random() < 0.15:
            dtype = "fp32"
        # K and V of all layers stay below 4 GiB, so that three states fit the card with room
        token = 2 * heads["H_kv"] * heads["D"] * (4 if dtype == "fp32" else 2)
        layers = max(1, min(rng.choice([2, 8, 28]), (4 << 30) // (B * (hi + 64) * token)))
        return {"kind": kind, "B": B, "lo": lo, "hi": hi, "block": rng.choice([16, 16, 32]), "layers": layers,
                "dtype": dtype, "graph": rng.random() < 0.6, **heads}
    if kind == "prefill":
        return {"kind": kind, "lengths": _some_lengths(rng, 12, rng.choice([600, 2048, 6000]), 8192),
                "layers": rng.randint(1, 4), "dtype": dtype, **heads}
    if kind == "write":
        lengths = _some_lengths(rng, 12, 2048, 8192)
        need = sum(-(-int(n) // BLOCK) for n in lengths.split(","))
        if rng.random() < 0.2:
            dtype = "fp32"
        return {"kind": kind, "lengths": lengths, "layers": rng.randint(1, 8), "dtype": dtype,
                "pages": need + rng.randint(1, 400), **heads}
    if kind == "tokenops":
        if heads["D"] == 64:
            heads = {"H": 16, "H_kv": 8, "D": 128}
        return {"kind": kind, "lengths": _some_lengths(rng, 10, 2048, 8192), "dtype": dtype,
                "hidden": rng.choice([1024, 1024, 2048, 2560]), "inter": rng.choice([3072, 3072, 6144, 1000]), **heads}
    if kind == "seats":
        hi = _log_int(rng, 24, 2040)
        return {"kind": kind, "S": rng.randint(1, 32), "lo": max(1, int(hi * rng.choice([0.1, 0.9]))), "hi": hi,
                "layers": rng.choice([2, 8])}
    return {"kind": kind, "lengths": _some_lengths(rng, 10, 1500, 6000), "layers": rng.choice([4, 28])}


# ------------------------------------------------------------------------------- inputs
def _gen(seed, device="cpu"):
    return torch.Generator(device=device).manual_seed(int(seed))


def _normal(g, *shape, dtype, scale=1.0):
    """N(0, scale) on the card, drawn in fp32 and cast, in slabs that need no second large copy."""
    out = torch.empty(shape, dtype=dtype, device=DEV)
    flat = out.view(-1)
    for at in range(0, flat.numel(), 1 << 26):
        n = min(1 << 26, flat.numel() - at)
        flat[at: at + n] = torch.randn(n, generator=g, device=DEV) * scale if scale != 1.0 else torch.randn(n, generator=g, device=DEV)
    return out


def _tables(lengths, block, n_pages, g):
    """Disjoint pages for each row from one permutation of the pool."""
    perm = torch.randperm(n_pages, generator=g).tolist()
    got, at = [], 0
    for n in lengths:
        need = max(1, -(-n // block))
        got.append(perm[at: at + need])
        at += need
    return got


def _pages(lengths, block):
    return sum(max(1, -(-n // block)) for n in lengths)


def _row_lengths(case, g, rows):
    return torch.randint(case["lo"], case["hi"] + 1, (rows,), generator=g).tolist()


def _decode_inputs(case, seed):
    """Ragged rows over a pool a quarter larger than they need, N(0, 1) q, K and V."""
    g, dg = _gen(seed), _gen(seed + 1, DEV)
    dt, block = DTYPES[case["dtype"]], case["block"]
    lengths = _row_lengths(case, g, case["B"])
    n_pages = _pages(lengths, block) * 5 // 4 + 1
    tables = _tables(lengths, block, n_pages, g)
    table = torch.zeros(case["B"], max(len(t) for t in tables), dtype=torch.int32)
    for r, t in enumerate(tables):
        table[r, : len(t)] = torch.tensor(t, dtype=torch.int32)
    shape = (n_pages, block, case["H_kv"], case["D"])
    ks = [_normal(dg, *shape, dtype=dt) for _ in range(case["layers"])]
    vs = [_normal(dg, *shape, dtype=dt) for _ in range(case["layers"])]
    qs = [_normal(dg, case["B"], case["H"], case["D"], dtype=dt) for _ in range(case["layers"])]
    return qs, ks, vs, table.to(DEV), torch.tensor(lengths, dtype=torch.int32, device=DEV), lengths


def _lengths(case):
    return [int(n) for n in case["lengths"].split(",")]


def _offsets(lengths):
    cu = [0]
    for n in lengths:
        cu.append(cu[-1] + n)
    return cu


def _slots(lengths, tables, block):
    parts = [torch.tensor(t).repeat_interleave(block)[:n] * block + torch.arange(n) % block for n, t in zip(lengths, tables)]
    return torch.cat(parts)


def _prefill_inputs(case, seed):
    g = _gen(seed, DEV)
    T, dt = sum(_lengths(case)), DTYPES[case["dtype"]]
    return [tuple(_normal(g, T, h, case["D"], dtype=dt) for h in (case["H"], case["H_kv"], case["H_kv"]))
            for _ in range(case["layers"])]


def _write_inputs(case, seed):
    g, dg = _gen(seed), _gen(seed + 1, DEV)
    lengths, dt = _lengths(case), DTYPES[case["dtype"]]
    slots = _slots(lengths, _tables(lengths, BLOCK, case["pages"], g), BLOCK).to(DEV)
    kv = [tuple(_normal(dg, sum(lengths), case["H_kv"], case["D"], dtype=dt) for _ in range(2)) for _ in range(case["layers"])]
    return slots, kv


def _tokenops_inputs(case, seed):
    """The tensors that the projections and the attention of a block hand to its other ops: normalised
    rows give projections of about unit scale; norm weights near one; a residual stream of unit scale."""
    g, dg = _gen(seed), _gen(seed + 1, DEV)
    lengths, dt = _lengths(case), DTYPES[case["dtype"]]
    T, C, inter, D = sum(lengths), case["hidden"], case["inter"], case["D"]
    s = {"embed": _normal(dg, 4096, C, dtype=dt), "tokens": torch.randint(0, 4096, (T,), generator=g).to(DEV),
         "qkv": _normal(dg, T, (case["H"] + 2 * case["H_kv"]) * D, dtype=dt), "o": _normal(dg, T, C, dtype=dt, scale=0.5),
         "gate_up": _normal(dg, T, 2 * inter, dtype=dt), "down": _normal(dg, T, C, dtype=dt, scale=0.5)}
    for name, n in (("ln1", C), ("ln2", C), ("ln3", C), ("qn", D), ("kn", D)):
        s[name] = (1.0 + 0.1 * _normal(dg, n, dtype=torch.float32)).to(dt)
    n_pages = _pages(lengths, BLOCK) + 8
    s["slots"] = _slots(lengths, _tables(lengths, BLOCK, n_pages, g), BLOCK).to(DEV)
    s["pos"] = torch.cat([torch.arange(n) for n in lengths]).to(DEV)
    s["cos"], s["sin"] = rope_table(D, 1e6, max(lengths), DEV, dt)
    return s, n_pages


def _model(case, seed):
    """The package's own model shape, N(0, 0.02) weights drawn on the card, norms near one."""
    cfg = Qwen3Config(n_layer=case["layers"])
    g = _gen(seed + 7, DEV)

    def w(*shape):
        return _normal(g, *shape, dtype=torch.bfloat16, scale=cfg.std)

    def norm(n):
        return (1.0 + 0.1 * _normal(g, n, dtype=torch.float32)).to(torch.bfloat16)

    H, Hk, D, C = cfg.n_head, cfg.n_kv_head, cfg.head_dim, cfg.hidden
    ws = {"embed": w(cfg.vocab, C), "norm": norm(C)}
    for i in range(cfg.n_layer):
        p = "l%d." % i
        ws.update({p + "wq": w(H * D, C), p + "wk": w(Hk * D, C), p + "wv": w(Hk * D, C), p + "wo": w(C, H * D),
                   p + "wg": w(cfg.inter, C), p + "wu": w(cfg.inter, C), p + "wd": w(C, cfg.inter),
                   p + "ln1": norm(C), p + "ln2": norm(C), p + "qn": norm(D), p + "kn": norm(D)})
    return cfg, ws


def _seats_inputs(case, seed):
    g, dg = _gen(seed), _gen(seed + 1, DEV)
    cfg, ws = _model(case, seed)
    lengths = _row_lengths(case, g, case["S"])
    n_pages = case["S"] * (case["hi"] // BLOCK + 1)
    tables = _tables([n + 1 for n in lengths], BLOCK, n_pages, g)
    shape = (n_pages, BLOCK, cfg.n_kv_head, cfg.head_dim)
    kv = [(_normal(dg, *shape, dtype=torch.bfloat16), _normal(dg, *shape, dtype=torch.bfloat16)) for _ in range(cfg.n_layer)]
    return cfg, ws, lengths, tables, n_pages, kv, torch.randint(0, cfg.vocab, (case["S"],), generator=g)


def _model_inputs(case, seed):
    g = _gen(seed)
    cfg, ws = _model(case, seed)
    lengths = _lengths(case)
    prompts = [torch.randint(0, cfg.vocab, (n,), generator=g).tolist() for n in lengths]
    n_pages = _pages(lengths, BLOCK) + 8
    return cfg, ws, prompts, _tables(lengths, BLOCK, n_pages, g), n_pages


# ------------------------------------------------------------------------------- passes
def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        qs, ks, vs, table, seqlen, _ = _decode_inputs(case, seed)
        s = {"case": case, "q": qs, "plan": paged_decode_plan(qs[0], ks, vs, table, seqlen)}
        if case["graph"]:
            _run_decode(s)  # once eagerly, as a program does before it captures
            torch.cuda.synchronize()
            s["replay"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["replay"]):
                s["out"] = _run_decode(s)
        return s
    if kind == "prefill":
        cu = _offsets(_lengths(case))
        return {"case": case, "qkv": _prefill_inputs(case, seed), "cu": cu, "longest": max(_lengths(case)),
                "backend": backend_for(torch.device(DEV))}
    if kind == "write":
        slots, kv = _write_inputs(case, seed)
        pool = PagedPool(case["layers"], case["pages"], BLOCK, case["H_kv"], case["D"], dtype=DTYPES[case["dtype"]],
                         device=DEV, n_head=case["H"])
        return {"case": case, "pool": pool, "slots": slots, "kv": kv}
    if kind == "tokenops":
        s, n_pages = _tokenops_inputs(case, seed)
        s["pool"] = PagedPool(1, n_pages, BLOCK, case["H_kv"], case["D"], dtype=DTYPES[case["dtype"]], device=DEV,
                              n_head=case["H"])
        s["case"] = case
        return s
    if kind == "seats":
        cfg, ws, lengths, tables, n_pages, kv, tokens = _seats_inputs(case, seed)
        model = Qwen3(cfg, ws, DEV, max_pos=4096)
        pool = model.new_pool(n_pages, BLOCK)
        dec = SeatDecoder(model, pool, case["S"], max(len(t) for t in tables), 8)
        dec.capture()
        for i, (k, v) in enumerate(kv):
            pool.keys[i].copy_(k)
            pool.values[i].copy_(v)
        for seat, (t, n) in enumerate(zip(tables, lengths)):
            dec.admit(seat, t, n, int(tokens[seat]))
        return {"case": case, "dec": dec, "pool": pool, "pos": dec.pos.clone(), "tokens": dec.tokens.clone()}
    cfg, ws, prompts, tables, n_pages = _model_inputs(case, seed)
    model = Qwen3(cfg, ws, DEV, max_pos=4096)
    return {"case": case, "model": model, "pool": model.new_pool(n_pages, BLOCK), "prompts": prompts, "tables": tables}


def _run_decode(s):
    plan = s["plan"]
    return [plan.run(layer, q) for layer, q in enumerate(s["q"])]


def run(s):
    kind = s["case"]["kind"]
    if kind == "decode":
        if "replay" in s:
            s["replay"].replay()
            return s["out"]
        return _run_decode(s)
    if kind == "prefill":
        return [s["backend"].prefill_varlen(q, k, v, cu_seqlens=s["cu"], max_seqlen=s["longest"]) for q, k, v in s["qkv"]]
    if kind == "write":
        pool = s["pool"]
        for layer, (k, v) in enumerate(s["kv"]):
            pool.write_slots(layer, s["slots"], k, v)
        return {"keys": pool.keys, "values": pool.values}
    if kind == "tokenops":
        pool = s["pool"]
        x = torch.nn.functional.embedding(s["tokens"], s["embed"])
        T = x.shape[0]
        k = torch.empty((T, pool.n_kv_head, pool.head_dim), dtype=pool.dtype, device=x.device)
        v = torch.empty_like(k)
        _, h1 = add_rms_norm(x, None, s["ln1"], EPS)
        q = pool.write_qk_norm_rope(0, s["slots"], s["qkv"], s["qn"], s["kn"], s["cos"], s["sin"], s["pos"], EPS,
                                    k_out=k, v_out=v)
        _, h2 = add_rms_norm(x, s["o"], s["ln2"], EPS)
        m = silu_mul(s["gate_up"])
        x, h3 = add_rms_norm(x, s["down"], s["ln3"], EPS)
        return {"h1": h1, "q": q, "k": k, "v": v, "h2": h2, "m": m, "x": x, "h3": h3, "keys": pool.keys[0],
                "values": pool.values[0]}
    if kind == "seats":
        dec = s["dec"]
        # the seats' state before the step, so that every pass is the same step
        dec.pos.copy_(s["pos"])
        dec.tokens.copy_(s["tokens"])
        dec.steps.zero_()
        dec.step()
        # the residual stream that the picks are made from, and the caches of the first and last layer
        return {"x": dec.x, "pos": dec.pos, "keys": [s["pool"].keys[0], s["pool"].keys[-1]],
                "values": [s["pool"].values[0], s["pool"].values[-1]]}
    logits = s["model"].prefill(s["prompts"], s["pool"], s["tables"])
    return {"logits": logits, "keys": [s["pool"].keys[0], s["pool"].keys[-1]],
            "values": [s["pool"].values[0], s["pool"].values[-1]]}


# ------------------------------------------------------------------------------- what a pass needs
def _pairs(lengths):
    return sum(n * (n + 1) // 2 for n in lengths)


def _layer_weights(cfg):
    return ((cfg.n_head + 2 * cfg.n_kv_head) * cfg.head_dim * cfg.hidden + cfg.hidden * cfg.n_head * cfg.head_dim
            + 3 * cfg.inter * cfg.hidden)


def work(case):
    kind = case["kind"]
    if kind in ("decode", "seats"):
        rows = case["B"] if kind == "decode" else case["S"]
        tokens = rows * (case["lo"] + case["hi"]) / 2  # lengths are uniform in [lo, hi]
    if kind == "decode":
        es = DTYPES[case["dtype"]].itemsize
        H, Hk, D = case["H"], case["H_kv"], case["D"]
        layer = tokens * 2 * Hk * D * es + 2 * rows * H * D * es
        return {"bytes": case["layers"] * layer, "flops": case["layers"] * 4 * tokens * H * D}
    if kind == "prefill":
        lengths = _lengths(case)
        T, es = sum(lengths), DTYPES[case["dtype"]].itemsize
        return {"bytes": case["layers"] * T * (2 * case["H"] + 2 * case["H_kv"]) * case["D"] * es,
                "flops": case["layers"] * 4 * case["H"] * case["D"] * _pairs(lengths)}
    if kind == "write":
        T, es = sum(_lengths(case)), DTYPES[case["dtype"]].itemsize
        return {"bytes": case["layers"] * T * (4 * case["H_kv"] * case["D"] * es + 8), "flops": 0}
    if kind == "tokenops":
        T, es = sum(_lengths(case)), DTYPES[case["dtype"]].itemsize
        H, Hk, D, C, inter = case["H"], case["H_kv"], case["D"], case["hidden"], case["inter"]
        # embedding rows in; three norms out; two residual inputs; x out; q/k/v in, q out, k and v out twice; gate and up in, one out
        values = C * (1 + 3 + 2 + 1) + (H + 2 * Hk) * D + H * D + 4 * Hk * D + 3 * inter
        return {"bytes": T * values * es, "flops": T * (12 * C + 10 * (H + Hk) * D + 6 * inter)}
    cfg = Qwen3Config(n_layer=case["layers"])
    H, Hk, D, C, V = cfg.n_head, cfg.n_kv_head, cfg.head_dim, cfg.hidden, cfg.vocab
    if kind == "seats":
        weights = cfg.n_layer * _layer_weights(cfg) + V * C
        return {"bytes": 2 * weights + cfg.n_layer * tokens * 4 * Hk * D,
                "flops": 2 * rows * weights + cfg.n_layer * 4 * tokens * H * D}
    lengths = _lengths(case)
    T, n = sum(lengths), len(lengths)
    return {"bytes": 2 * (cfg.n_layer * _layer_weights(cfg) + V * C) + cfg.n_layer * T * 4 * Hk * D + 2 * T * C + 2 * n * V,
            "flops": cfg.n_layer * (2 * T * _layer_weights(cfg) + 4 * H * D * _pairs(lengths)) + 2 * n * V * C}


def tolerance(case):
    """About four times the distance from 64 bits that each kind measures (two correct paths round
    some of their 16-bit values the other way): decode 1.7e-3 in bf16 and 2.1e-4 in fp16, prefill
    2.0e-3 and 2.5e-4, the token ops 3.9e-3 and 5e-4 (rounded op by op), a model's logits 1.4e-2."""
    kind, bf16 = case["kind"], case.get("dtype") == "bf16"
    if kind == "write":
        return "exact"  # a copy
    if kind in ("seats", "model"):
        # 16-bit roundings of one layer travel through all that follow
        return {"rel": 0.03, "max": 0.5}
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 2e-4}
    if kind == "tokenops":
        return {"rel": 1.6e-2, "max": 0.06} if bf16 else {"rel": 2e-3, "max": 8e-3}
    if kind == "prefill":  # probabilities are rounded to the inputs' 16 bits before their product with V
        return {"rel": 8e-3, "max": 0.08} if bf16 else {"rel": 1e-3, "max": 0.01}
    return {"rel": 7e-3, "max": 0.04} if bf16 else {"rel": 9e-4, "max": 6e-3}


# ------------------------------------------------------------------------------- in 64 bits
def _attend64(q, k, v, causal):
    """q (Lq, H, D), k and v (Lk, H_kv, D) in 64 bits; causal: query i sees keys 0..i."""
    Lq, H, D = q.shape
    Hk = k.shape[1]
    out = torch.empty_like(q)
    step = max(1, (1 << 27) // max(1, k.shape[0] * (H // Hk)))  # score rows at a time
    for h in range(Hk):
        kh, vh = k[:, h], v[:, h]
        qh = q.view(Lq, Hk, H // Hk, D)[:, h]
        for at in range(0, Lq, step):
            to = min(Lq, at + step)
            keys = to if causal else k.shape[0]
            sc = (qh[at:to].reshape(-1, D) @ kh[:keys].t().contiguous()).view(to - at, H // Hk, keys) / math.sqrt(D)
            if causal:
                ahead = torch.arange(keys, device=q.device) > torch.arange(at, to, device=q.device).unsqueeze(1)
                sc = sc.masked_fill(ahead.unsqueeze(1), -math.inf)
            p = torch.softmax(sc, -1)
            out.view(Lq, Hk, H // Hk, D)[at:to, h] = (p.view(-1, keys) @ vh[:keys]).view(to - at, H // Hk, D)
    return out


def _norm64(x, w):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w


def _rope64(x, cos, sin):
    half = x.shape[-1] // 2
    a, b = x[..., :half], x[..., half:]
    cos, sin = cos.unsqueeze(-2), sin.unsqueeze(-2)
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def _gather64(pool, table, n, block):
    """The first n tokens of one row's pages, in 64 bits."""
    pages = torch.as_tensor(table, device=pool.device)[: -(-n // block)].long()
    return pool[pages].reshape(-1, *pool.shape[2:])[:n].double()


def _exact_decode(case, seed):
    qs, ks, vs, table, _, lengths = _decode_inputs(case, seed)
    outs = []
    for q, k, v in zip(qs, ks, vs):
        o = torch.zeros(q.shape, dtype=torch.float64, device=DEV)
        for r, n in enumerate(lengths):
            o[r] = _attend64(q[r: r + 1].double(), _gather64(k, table[r], n, case["block"]),
                             _gather64(v, table[r], n, case["block"]), False)[0]
        outs.append(o)
    return outs


def _exact_prefill(case, seed):
    cu = _offsets(_lengths(case))
    outs = []
    for q, k, v in _prefill_inputs(case, seed):
        outs.append(torch.cat([_attend64(q[a:b].double(), k[a:b].double(), v[a:b].double(), True)
                               for a, b in zip(cu, cu[1:])]))
    return outs


def _exact_tokenops(case, seed):
    s, n_pages = _tokenops_inputs(case, seed)
    d = {k: v.double() if v.is_floating_point() else v for k, v in s.items()}
    T, H, Hk, D = d["tokens"].numel(), case["H"], case["H_kv"], case["D"]
    x = d["embed"][d["tokens"]]
    h1 = _norm64(x, d["ln1"])
    q, k, v = d["qkv"].view(T, H + 2 * Hk, D).split([H, Hk, Hk], 1)
    cos, sin = d["cos"][d["pos"]], d["sin"][d["pos"]]
    q, k = _rope64(_norm64(q, d["qn"]), cos, sin), _rope64(_norm64(k, d["kn"]), cos, sin)
    pools = []
    for t in (k, v):
        pool = torch.zeros(n_pages * BLOCK, Hk, D, dtype=torch.float64, device=DEV)
        pool[d["slots"]] = t
        pools.append(pool.view(n_pages, BLOCK, Hk, D))
    x = x + d["o"]
    h2 = _norm64(x, d["ln2"])
    gate, up = d["gate_up"].chunk(2, -1)
    m = torch.nn.functional.silu(gate) * up
    x = x + d["down"]
    return {"h1": h1, "q": q, "k": k, "v": v, "h2": h2, "m": m, "x": x, "h3": _norm64(x, d["ln3"]), "keys": pools[0],
            "values": pools[1]}


def _angles(cfg, length):
    cos, sin = rope_table(cfg.head_dim, cfg.rope_theta, length, DEV, torch.bfloat16)
    return cos.double(), sin.double()


def _layers64(cfg, ws, x, pos, attend):
    """Every block of the model on rows x at positions pos; attend(i, q, k, v) gives their attention."""
    cos, sin = (t[pos] for t in _angles(cfg, 4096))
    H, Hk, D = cfg.n_head, cfg.n_kv_head, cfg.head_dim
    for i in range(cfg.n_layer):
        w = {n: ws["l%d.%s" % (i, n)].double() for n in ("wq", "wk", "wv", "wo", "wg", "wu", "wd", "ln1", "ln2", "qn", "kn")}
        h = _norm64(x, w["ln1"])
        q, k, v = ((h @ w[n].t()).view(-1, m, D) for n, m in (("wq", H), ("wk", Hk), ("wv", Hk)))
        q, k = _rope64(_norm64(q, w["qn"]), cos, sin), _rope64(_norm64(k, w["kn"]), cos, sin)
        x = x + attend(i, q, k, v).reshape(x.shape[0], H * D) @ w["wo"].t()
        h = _norm64(x, w["ln2"])
        x = x + (torch.nn.functional.silu(h @ w["wg"].t()) * (h @ w["wu"].t())) @ w["wd"].t()
    return x


def _exact_seats(case, seed):
    cfg, ws, lengths, tables, n_pages, kv, tokens = _seats_inputs(case, seed)
    pos = torch.tensor(lengths, device=DEV)
    caches = {}

    def attend(i, q, k, v):
        pools = [t.double() for t in kv[i]]
        for r, n in enumerate(lengths):
            slot = (tables[r][n // BLOCK], n % BLOCK)
            pools[0][slot], pools[1][slot] = k[r], v[r]
        if i in (0, cfg.n_layer - 1):
            caches[i] = pools
        return torch.cat([_attend64(q[r: r + 1], _gather64(pools[0], tables[r], n + 1, BLOCK),
                                    _gather64(pools[1], tables[r], n + 1, BLOCK), False) for r, n in enumerate(lengths)])

    x = _layers64(cfg, ws, ws["embed"][tokens.to(DEV)].double(), pos, attend)
    ends = (caches[0], caches[cfg.n_layer - 1])
    return {"x": x, "pos": None, "keys": [c[0] for c in ends], "values": [c[1] for c in ends]}


def _exact_model(case, seed):
    cfg, ws, prompts, tables, n_pages = _model_inputs(case, seed)
    lengths = [len(p) for p in prompts]
    cu = _offsets(lengths)
    pos = torch.cat([torch.arange(n) for n in lengths]).to(DEV)
    slots = _slots(lengths, tables, BLOCK).to(DEV)
    caches = {}

    def attend(i, q, k, v):
        if i in (0, cfg.n_layer - 1):
            caches[i] = []
            for t in (k, v):
                pool = torch.zeros(n_pages * BLOCK, *t.shape[1:], dtype=torch.float64, device=DEV)
                pool[slots] = t
                caches[i].append(pool.view(n_pages, BLOCK, *t.shape[1:]))
        return torch.cat([_attend64(q[a:b], k[a:b], v[a:b], True) for a, b in zip(cu, cu[1:])])

    tokens = torch.tensor([t for p in prompts for t in p], device=DEV)
    x = _layers64(cfg, ws, ws["embed"][tokens].double(), pos, attend)
    h = _norm64(x[torch.tensor(cu[1:], device=DEV) - 1], ws["norm"].double())
    ends = (caches[0], caches[cfg.n_layer - 1])
    return {"logits": h @ ws["embed"].double().t(), "keys": [c[0] for c in ends], "values": [c[1] for c in ends]}


def exact(case, seed):
    kind = case["kind"]
    if kind == "write":
        return None  # bytes
    with torch.no_grad():
        return {"decode": _exact_decode, "prefill": _exact_prefill, "tokenops": _exact_tokenops, "seats": _exact_seats,
                "model": _exact_model}[kind](case, seed)
