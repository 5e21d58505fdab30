"""The work this library is called for, as measurable cases.

A case is one call (or the calls that always go together) of the per-token layer path through
`padra_amd.ops`: the decode step's gather + norm + Q/K + KV store, the same chain over a prefill
chunk, the local ring's neighbours of that chunk, SwiGLU and the expert combine of the MoE half,
the FP8 row encoding of the norm, and decode attention over the three cache formats.  The
geometries are those of the repository's own workloads: hidden 2048 with 16 query heads (the
benchmark) and hidden 2304 with 32 query heads (the reference model), 4 KV heads of 128, expert
widths 1024 and 896, chunks of at most 2048 tokens, local rings of 1024 rows.  Activations are BF16
or the reference's own fp32 buffers of BF16-exact values.

listed() names twelve; draw() gives more of the same ranges.
"""
from __future__ import annotations

import math

import torch

from padra_amd import abi, ops

D = 128          # head dimension
HKV = 4          # KV heads
F = HKV * D      # features of a cache row
EPS = 1e-6
TABLE_ROWS = 40960
FORMATS = {"bf16": abi.KV_BF16, "q8": abi.KV_Q8, "q8_0": abi.KV_Q8_0}
ROW_BYTES = {"bf16": 2 * F, "q8": F + 4 * HKV, "q8_0": 544}  # of K, and of V again
GEOMETRY = {2048: 16, 2304: 32}  # hidden: query heads


def listed():
    return [
        # One user's decode step, layer 0: token gather, residual norm, Q/K norm + RoPE and the
        # BF16 cache row in one launch.  The smallest call there is: latency and host time.
        {"name": "decode 1 bf16", "kind": "decode", "seqs": 1, "hidden": 2304, "kv": "bf16",
         "act": "bf16", "embed": True},
        # A serving batch's decode step with the 8-bit cache that long contexts use.
        {"name": "decode 64 q8_0", "kind": "decode", "seqs": 64, "hidden": 2048, "kv": "q8_0",
         "act": "bf16", "embed": True},
        # The full prefill chunk of a global layer, BF16 storage (the benchmark's config 1).
        {"name": "prefill 2048 bf16", "kind": "prefill", "tokens": 2048, "hidden": 2048,
         "kv": "bf16", "act": "bf16", "local": False},
        # The reference model's prefill on its own fp32 buffers, the last chunk of a prompt (an
        # odd length) into a local ring that is narrower than the chunk.
        {"name": "prefill 1531 q8_0 f32", "kind": "prefill", "tokens": 1531, "hidden": 2304,
         "kv": "q8_0", "act": "f32", "local": True},
        # A local layer's cache work around a chunk's attention: decode of the old ring rows,
        # encoding of the chunk, commit of its last rows into the ring.
        {"name": "ring chunk 2048 q8_0", "kind": "ring", "tokens": 2048, "kv": "q8_0",
         "act": "bf16"},
        # Expert activations of a full chunk (top 8 of the experts, benchmark config 3).
        {"name": "swiglu 16384x1024", "kind": "swiglu", "rows": 16384, "width": 1024,
         "act": "bf16"},
        # Expert combine + residual + next layer's norm + FP8 rows on fp32 buffers.
        {"name": "combine norm 2048 f32", "kind": "combine", "rows": 2048, "hidden": 2304,
         "act": "f32", "fp8": True},
        # Input norm and FP8 rows of a chunk, fp32 buffers.
        {"name": "norm fp8 2048 f32", "kind": "norm_fp8", "rows": 2048, "hidden": 2304,
         "act": "f32"},
        # One user's decode attention over a long context, global layer, the reference's splits.
        {"name": "attention 1x32k bf16", "kind": "attention", "seqs": 1, "keys": 32768,
         "q_heads": 32, "kv": "bf16", "act": "bf16", "local": False, "splits": 0, "fp8": False},
        # A small batch over q8 caches, output coded to FP8 for the O projection.
        {"name": "attention 8x8k q8 fp8", "kind": "attention", "seqs": 8, "keys": 8000,
         "q_heads": 32, "kv": "q8", "act": "bf16", "local": False, "splits": 0, "fp8": True},
        # A serving batch at ragged positions over q8_0 caches: the largest.
        {"name": "attention 64x32k q8_0", "kind": "attention", "seqs": 64, "keys": 32768,
         "q_heads": 16, "kv": "q8_0", "act": "bf16", "local": False, "splits": 0, "fp8": False},
        # A local layer of a small batch: 1024-row rings, the split count tuned for this card.
        {"name": "attention 12 local bf16", "kind": "attention", "seqs": 12, "keys": 3000,
         "q_heads": 32, "kv": "bf16", "act": "f32", "local": True, "splits": -1, "fp8": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Kinds by how often a layer runs them (decode and its attention most); sizes spread over
    their logarithm."""
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "ring", "swiglu", "combine",
                       "norm_fp8", "attention", "attention", "attention", "attention"])
    act = rng.choice(["bf16", "f32"])
    hidden = rng.choice(sorted(GEOMETRY))
    kv = rng.choice(sorted(FORMATS))
    if kind == "decode":
        return {"kind": kind, "seqs": _log(rng, 1, 64), "hidden": hidden, "kv": kv, "act": act,
                "embed": act == "bf16"}
    if kind == "prefill":
        return {"kind": kind, "tokens": _log(rng, 16, 2048), "hidden": hidden, "kv": kv,
                "act": act, "local": rng.random() < .5}
    if kind == "ring":
        return {"kind": kind, "tokens": _log(rng, 16, 2048), "kv": kv, "act": act}
    if kind == "swiglu":
        return {"kind": kind, "rows": _log(rng, 8, 16384), "width": rng.choice([896, 1024]),
                "act": act}
    if kind == "combine":
        return {"kind": kind, "rows": _log(rng, 1, 2048), "hidden": hidden, "act": act,
                "fp8": rng.random() < .7}
    if kind == "norm_fp8":
        return {"kind": kind, "rows": _log(rng, 1, 2048), "hidden": hidden, "act": act}
    seqs = _log(rng, 1, 64)
    local = rng.random() < .35
    # no more keys in all than the largest listed case
    keys = _log(rng, 64, 131072 if local else min(131072, (64 * 32768) // seqs))
    return {"kind": kind, "seqs": seqs, "keys": keys, "q_heads": rng.choice([16, 32]), "kv": kv,
            "act": act, "local": local, "splits": rng.choice([0, -1]),
            "fp8": kv != "q8_0" and rng.random() < .4}


# ---- inputs ------------------------------------------------------------------------------

class _State:
    pass


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _act_dtype(case):
    return torch.float32 if case["act"] == "f32" else torch.bfloat16


def _normal(g, shape, dtype=torch.bfloat16, sigma=1.0, outliers=None):
    """BF16 normals; `outliers`: one channel in a hundred is twenty times larger."""
    t = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(sigma)
    if outliers is not None:
        t.index_copy_(-1, outliers, t.index_select(-1, outliers) * 20)
    return t.to(torch.bfloat16).to(dtype)


def _channels(g, n):
    return torch.randperm(n, generator=g, device="cuda")[:n // 100]


def _weights(g, n):
    return (torch.rand(n, generator=g, device="cuda") + .5).to(torch.bfloat16)


def _table():
    if not hasattr(_table, "t"):
        _table.t = ops.RopeTable(TABLE_ROWS, D).cuda()
    return _table.t


def _empty_cache(kv, rows):
    if kv == "bf16":
        k = torch.zeros((rows, F), dtype=torch.bfloat16, device="cuda")
        return k, torch.zeros_like(k), None
    if kv == "q8":
        k = torch.zeros((rows, F), dtype=torch.int8, device="cuda")
        return k, torch.zeros_like(k), torch.zeros((rows, HKV, 2), device="cuda")
    k = torch.zeros((rows, 544), dtype=torch.uint8, device="cuda")
    return k, torch.zeros_like(k), None


def _filled_plane(g, kv, rows):
    """K or V rows as the store kernels leave them: unit normals, or the codes of such."""
    if kv == "bf16":
        return torch.randn((rows, F), generator=g, device="cuda", dtype=torch.bfloat16)
    out = torch.empty((rows, F if kv == "q8" else 544), dtype=torch.uint8, device="cuda")
    for at in range(0, rows, 1 << 18):
        n = min(1 << 18, rows - at)
        codes = torch.randn((n, F), generator=g, device="cuda", dtype=torch.bfloat16).mul_(
            45.).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
        if kv == "q8":
            out[at:at + n] = codes
        else:
            d = (torch.rand((n, 16), generator=g, device="cuda") * .015 + .015).half()
            out[at:at + n, :32] = d.view(torch.uint8)
            out[at:at + n, 32:] = codes
    return out.view(torch.int8) if kv == "q8" else out


def _filled_cache(g, kv, rows):
    k, v = _filled_plane(g, kv, rows), _filled_plane(g, kv, rows)
    scales = None
    if kv == "q8":
        scales = torch.rand((rows, HKV, 2), generator=g, device="cuda") * .015 + .015
    return k, v, scales


def _spread(seqs, keys):
    """Ragged window lengths of a batch, 1..keys, the longest among them; the same for every
    seed, so that a case's work does not depend on it."""
    return [max(1, int(keys * (1 - (i * .6180339887) % 1))) for i in range(seqs)]


def _decode_states(positions, tokens, capacity):
    rows = [[t, p, capacity, 16, p, min(p, 1024), 0, 0] for p, t in zip(positions, tokens)]
    return torch.tensor(rows, dtype=torch.int32, device="cuda")


def _prefill_state(base, tokens, capacity):
    return torch.tensor([base, 0, tokens, capacity, base, 1, 1, 1], dtype=torch.int32,
                        device="cuda")


def _chain_inputs(s, g, tokens, hidden, dtype):
    hq = GEOMETRY[hidden]
    channels = _channels(g, hidden)
    s.x = _normal(g, (tokens, hidden), dtype, outliers=channels)
    s.r = _normal(g, (tokens, hidden), dtype, outliers=channels)
    s.y = torch.empty_like(s.x)
    s.gamma = _weights(g, hidden)
    s.q = _normal(g, (tokens, hq * D), dtype, outliers=_channels(g, hq * D)).view(tokens, hq, D)
    s.k = _normal(g, (tokens, F), dtype, outliers=_channels(g, F)).view(tokens, HKV, D)
    s.v = _normal(g, (tokens, F), dtype, outliers=_channels(g, F)).view(tokens, HKV, D)
    # The call works in place, and a program makes new q and k for each; with the unit weights
    # of a freshly initialised model a pass over its own result meets the same distribution.
    s.qn = torch.ones(D, dtype=torch.bfloat16, device="cuda")
    s.kn = torch.ones(D, dtype=torch.bfloat16, device="cuda")
    s.table = _table()


DECODE_CAP = 8192  # rows of each sequence's cache in a decode step
VOCAB = 98304


def _prefill_sizes(case):
    """capacity, ring rows, base position and first stored chunk row."""
    tokens, capacity = case["tokens"], 8192
    cap = 1024 if case.get("local", True) else capacity
    first = max(0, tokens - cap) if cap < capacity else 0
    return capacity, cap, min(3 * tokens + 5, capacity - tokens), first


def prepare(case, seed):
    g = _gen(seed)
    s = _State()
    s.kind = case["kind"]
    s.bad = torch.zeros(1, dtype=torch.int32, device="cuda")
    if s.kind == "decode":
        n, hidden = case["seqs"], case["hidden"]
        _chain_inputs(s, g, n, hidden, _act_dtype(case))
        positions = [min(p, DECODE_CAP - 1) for p in _spread(n, DECODE_CAP - 1)]
        ids = torch.randint(0, VOCAB, (n,), generator=g, device="cuda").tolist()
        s.states = _decode_states(positions, ids, DECODE_CAP)
        s.pos = ops.positions_decode(s.states, maximum=DECODE_CAP, vocab=VOCAB)
        s.cache = _empty_cache(case["kv"], n * DECODE_CAP)
        s.kv = ops.kv_cache(FORMATS[case["kv"]], s.cache[0], s.cache[1], DECODE_CAP,
                            scales=s.cache[2], seq_stride=DECODE_CAP)
        s.embed = _normal(g, (VOCAB, hidden)) if case["embed"] else None
    elif s.kind == "prefill":
        tokens = case["tokens"]
        _chain_inputs(s, g, tokens, case["hidden"], _act_dtype(case))
        capacity, cap, base, first = _prefill_sizes(case)
        s.state = _prefill_state(base, tokens, capacity)
        s.pos = ops.positions_prefill(s.state, maximum=capacity)
        s.cache = _empty_cache(case["kv"], cap)
        s.kv = ops.kv_cache(FORMATS[case["kv"]], s.cache[0], s.cache[1], cap, scales=s.cache[2],
                            first=first)
    elif s.kind == "ring":
        tokens, kv = case["tokens"], case["kv"]
        capacity, cap, base, first = _prefill_sizes(case)
        s.k = _normal(g, (tokens, HKV, D), _act_dtype(case))
        s.v = _normal(g, (tokens, HKV, D), _act_dtype(case))
        s.state = _prefill_state(base, tokens, capacity)
        s.pos = ops.positions_prefill(s.state, maximum=capacity)
        s.zero = ops.positions_base(0)
        s.tokens = tokens
        s.chunk = _empty_cache(kv, tokens)
        s.chunk_kv = ops.kv_cache(FORMATS[kv], s.chunk[0], s.chunk[1], tokens, scales=s.chunk[2])
        s.ring = _filled_cache(g, kv, cap)
        s.ring_kv = ops.kv_cache(FORMATS[kv], s.ring[0], s.ring[1], cap, scales=s.ring[2],
                                 first=first)
        s.prefix = None
        if kv == "q8_0":
            s.prefix = tuple(torch.zeros((cap, F), dtype=torch.bfloat16, device="cuda")
                             for _ in range(2))
    elif s.kind == "swiglu":
        shape = (case["rows"], case["width"])
        s.gate = _normal(g, shape, _act_dtype(case), sigma=2.)
        s.up = _normal(g, shape, _act_dtype(case), sigma=2.)
        s.out = torch.empty_like(s.gate)
        s.table = torch.empty(65536, dtype=torch.int16, device="cuda")
        ops.SiluTableBuild(s.table)
    elif s.kind == "combine":
        rows, hidden = case["rows"], case["hidden"]
        s.x = _normal(g, (rows, hidden), _act_dtype(case), outliers=_channels(g, hidden))
        s.down = _normal(g, (rows, 8, hidden), _act_dtype(case))
        s.weights = torch.softmax(torch.randn((rows, 8), generator=g, device="cuda"), -1)
        s.y = torch.empty_like(s.x)
        s.gamma = _weights(g, hidden)
        s.packed = s.scales = None
        if case["fp8"]:
            s.packed = torch.empty((rows, hidden), dtype=torch.uint8, device="cuda")
            s.scales = torch.empty(rows, device="cuda")
    elif s.kind == "norm_fp8":
        rows, hidden = case["rows"], case["hidden"]
        s.x = _normal(g, (rows, hidden), _act_dtype(case), outliers=_channels(g, hidden))
        s.y = torch.empty_like(s.x)
        s.gamma = _weights(g, hidden)
        s.packed = torch.empty((rows, hidden), dtype=torch.uint8, device="cuda")
        s.scales = torch.empty(rows, device="cuda")
    else:
        n, hq = case["seqs"], case["q_heads"]
        capacity, cap = _attention_sizes(case)
        s.q = _normal(g, (n, hq, D), _act_dtype(case), sigma=2.)
        s.out = torch.empty_like(s.q)
        s.states = _decode_states([w - 1 for w in _spread(n, case["keys"])], [5] * n, capacity)
        s.pos = ops.positions_decode(s.states, maximum=capacity)
        s.cache = _filled_cache(g, case["kv"], n * cap)
        s.kv = ops.kv_cache(FORMATS[case["kv"]], s.cache[0], s.cache[1], cap, scales=s.cache[2],
                            seq_stride=cap)
        s.local, s.splits = case["local"], case["splits"]
        s.packed = s.scales = None
        if case["fp8"]:
            s.packed = torch.empty((n, hq * D), dtype=torch.uint8, device="cuda")
            s.scales = torch.empty(n, device="cuda")
        # a decode loop keeps its scratch: one query, sized once
        s.scratch = ops.DecodeAttention(s.q, s.kv, s.out, s.pos, s.bad, kv_heads=HKV,
                                        local=s.local, splits=s.splits)
    return s


def _attention_sizes(case):
    """The context's capacity and the rows of each sequence's cache."""
    capacity = max(1024, -(-case["keys"] // 1024) * 1024)
    return capacity, 1024 if case["local"] else capacity


# ---- one pass ----------------------------------------------------------------------------

def run(s):
    if s.kind == "decode" and s.embed is not None:
        ops.EmbedResidualNormQKRopeStore(s.embed, None, s.x, s.r, s.y, s.gamma, s.q, s.k, s.v,
                                         s.qn, s.kn, s.table, s.pos, s.kv, s.bad,
                                         tree=abi.TREE_256)
    elif s.kind == "decode":
        ops.ResidualNormQKRopeStore(s.x, s.r, s.y, s.gamma, s.q, s.k, s.v, s.qn, s.kn, s.table,
                                    s.pos, s.kv, s.bad, tree=abi.TREE_256)
    elif s.kind == "prefill":
        ops.ResidualNormQKRopeStore(s.x, s.r, s.y, s.gamma, s.q, s.k, s.v, s.qn, s.kn, s.table,
                                    s.pos, s.kv, s.bad)
    elif s.kind == "ring":
        if s.prefix is not None:
            ops.KvQ8_0DequantizePrefix(s.ring[0], s.ring[1], s.prefix[0], s.prefix[1], s.pos,
                                       s.tokens, s.bad)
        ops.KVStore(s.k, s.v, s.zero, s.chunk_kv, s.bad)
        ops.KVCommit(s.chunk_kv, s.ring_kv, s.pos, s.tokens, HKV, s.bad)
        return {"prefix": s.prefix, "chunk": s.chunk, "ring": s.ring, "bad": s.bad}
    elif s.kind == "swiglu":
        ops.SwiGLU(s.gate, s.up, s.out, s.table, s.bad)
        return {"out": s.out, "bad": s.bad}
    elif s.kind == "combine":
        ops.CombineNorm(s.x, s.down, s.weights, s.y, s.gamma, s.bad, packed=s.packed,
                        scales=s.scales)
        return {"x": s.x, "y": s.y, "packed": s.packed, "scales": s.scales, "bad": s.bad}
    elif s.kind == "norm_fp8":
        ops.NormFP8(s.x, s.y, s.gamma, s.packed, s.scales, s.bad)
        return {"y": s.y, "packed": s.packed, "scales": s.scales, "bad": s.bad}
    else:
        ops.DecodeAttention(s.q, s.kv, s.out, s.pos, s.bad, kv_heads=HKV, local=s.local,
                            splits=s.splits, scratch=s.scratch, packed=s.packed,
                            scales=s.scales)
        return {"out": s.out, "packed": s.packed, "scales": s.scales, "bad": s.bad}
    return {"x": s.x, "y": s.y, "q": s.q, "k": s.k, "cache": s.cache, "bad": s.bad}


# ---- what a pass cannot do without -------------------------------------------------------

def work(case):
    e = 4 if case.get("act") == "f32" else 2
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        n = case["seqs"] if kind == "decode" else case["tokens"]
        hidden = case["hidden"]
        hq = GEOMETRY[hidden]
        stored = n - (_prefill_sizes(case)[3] if kind == "prefill" else 0)
        row = 4 * hidden * e + (2 * hq + 2 * HKV + HKV) * D * e + 2 * D
        return {"bytes": n * row + stored * 2 * ROW_BYTES[case["kv"]] + 2 * hidden + 4 * D,
                "flops": n * (6 * hidden + 10 * (hq + HKV) * D)}
    if kind == "ring":
        tokens, kv = case["tokens"], case["kv"]
        _, cap, base, first = _prefill_sizes(case)
        moved = 2 * tokens * F * e + 2 * tokens * ROW_BYTES[kv]   # encode
        moved += 4 * (tokens - first) * ROW_BYTES[kv]             # commit
        if kv == "q8_0":
            moved += 2 * min(base, cap) * (544 + 2 * F)           # decode of the old rows
        return {"bytes": moved, "flops": 0 if kv == "bf16" else 2 * tokens * F * 12}
    if kind == "swiglu":
        n = case["rows"] * case["width"]
        return {"bytes": 3 * n * e, "flops": 4 * n}
    if kind == "combine":
        n = case["rows"] * case["hidden"]
        return {"bytes": n * (11 * e + (1 if case["fp8"] else 0)) + 36 * case["rows"],
                "flops": 22 * n}
    if kind == "norm_fp8":
        n = case["rows"] * case["hidden"]
        return {"bytes": n * (2 * e + 1) + 4 * case["rows"], "flops": 8 * n}
    lengths = _spread(case["seqs"], case["keys"])
    keys = sum(min(w, 1024) if case["local"] else w for w in lengths)
    hq = case["q_heads"]
    rows = case["seqs"] * hq * D * (2 * e + (1 if case["fp8"] else 0))  # q, out and its codes
    return {"bytes": keys * 2 * ROW_BYTES[case["kv"]] + rows, "flops": 4 * keys * hq * D}


def tolerance(case):
    """Every operation but attention is defined bit for bit (the reference's rounding points and
    summation orders).  Attention's sums have no defined order and its exponentials no defined
    last bits; its outputs are rounded to BF16 once, its probabilities too for the BF16 and q8
    caches, and the values decoded from a q8 cache.  Measured against exact(): rel 1.7e-3 (BF16,
    q8_0) and 4.3e-3 (q8)."""
    if case["kind"] == "attention":
        return {"rel": 1e-2, "max": 8e-2, "differ": 1e-2}
    return "exact"


# ---- the same in 64 bits -----------------------------------------------------------------

def _norm64(v, weight):
    return v * torch.rsqrt(v.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _rope64(v, table, positions):
    """NeoX rotation of [T][heads][D] rows at their positions."""
    row = table[positions].double()
    cos, sin = row[:, None, :D // 2], row[:, None, D // 2:]
    a, b = v[..., :D // 2], v[..., D // 2:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _exact_chain(case, s):
    if case["kind"] == "decode":
        positions = s.states[:, 1].long()
        slots = torch.arange(len(positions), device="cuda") * DECODE_CAP + positions
        stored = slice(None)
    else:
        _, cap, base, first = _prefill_sizes(case)
        positions = base + torch.arange(case["tokens"], device="cuda")
        stored = slice(first, None)
        slots = positions[stored] % cap
    x = s.x.double()
    if case["kind"] == "decode" and s.embed is not None:
        x = s.embed[s.states[:, 0].long()].double()
    x = x + s.r.double()
    q = _rope64(_norm64(s.q.double(), s.qn), s.table, positions)
    k = _rope64(_norm64(s.k.double(), s.kn), s.table, positions)
    cache = [None, None, None]
    k_rows, v_rows = k[stored], s.v.double()[stored]
    if case["kv"] == "bf16":
        cache = [torch.zeros(s.cache[0].shape, dtype=torch.float64, device="cuda")
                 for _ in range(2)] + [None]
        cache[0][slots] = k_rows.reshape(-1, F)
        cache[1][slots] = v_rows.reshape(-1, F)
    elif case["kv"] == "q8":
        cache[2] = torch.zeros(s.cache[2].shape, dtype=torch.float64, device="cuda")
        cache[2][slots] = torch.stack([k_rows.abs().amax(-1), v_rows.abs().amax(-1)], -1) / 127
    return {"x": x, "y": _norm64(x, s.gamma), "q": q, "k": k, "cache": cache, "bad": None}


def _hadamard64(v, n):
    """Orthonormal transforms of the last axis' blocks of n."""
    h = torch.ones((1, 1), dtype=torch.float64, device=v.device)
    while h.shape[0] < n:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return ((v.reshape(-1, n) @ h) / math.sqrt(n)).reshape(v.shape)


def _plane64(case, plane, scale):
    """The values of K or V rows [n] as [n][HKV][D]."""
    if case["kv"] == "bf16":
        return plane.double().view(-1, HKV, D)
    if case["kv"] == "q8":
        return plane.double().view(-1, HKV, D) * scale.double()[..., None]
    d = plane[:, :32].contiguous().view(torch.float16).double()
    codes = plane[:, 32:].contiguous().view(torch.int8).double()
    return (codes.view(-1, 16, 32) * d[..., None]).view(-1, HKV, D)


def _exact_attention(case, s):
    n, hq = case["seqs"], case["q_heads"]
    _, cap = _attention_sizes(case)
    group = hq // HKV
    out = torch.empty((n, hq, D), dtype=torch.float64, device="cuda")
    q = s.q.double()
    if case["kv"] == "q8_0":  # the path codes the rotated query in blocks of 32
        q = _hadamard64(q, D)
        blocks = q.view(n, hq, 4, 32)
        d = blocks.abs().amax(-1, keepdim=True) / 127
        q = (torch.round(blocks / d.clamp_min(1e-300)) * d).view(n, hq, D)
    for i, length in enumerate(_spread(n, case["keys"])):
        window = min(length, 1024) if case["local"] else length
        rows = i * cap + (length - window + torch.arange(window, device="cuda")) % cap
        scales = s.cache[2][rows] if case["kv"] == "q8" else None
        k = _plane64(case, s.cache[0][rows], None if scales is None else scales[..., 0])
        v = _plane64(case, s.cache[1][rows], None if scales is None else scales[..., 1])
        for h in range(HKV):
            heads = slice(h * group, (h + 1) * group)
            p = torch.softmax(q[i, heads] @ k[:, h].T / math.sqrt(D), -1)
            out[i, heads] = p @ v[:, h]
    if case["kv"] == "q8_0":  # V rows are rotated in halves
        out = _hadamard64(out, D // 2)
    scales = None
    if case["fp8"]:
        scales = out.abs().amax((1, 2)) / 448
    return {"out": out, "packed": None, "scales": scales, "bad": None}


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _exact_chain(case, s)
    if kind == "ring":
        prefix = None
        if s.prefix is not None:
            _, cap, base, _ = _prefill_sizes(case)
            rows = min(base, cap)
            prefix = [torch.zeros((cap, F), dtype=torch.float64, device="cuda") for _ in range(2)]
            for out, plane in zip(prefix, s.ring):
                out[:rows] = _plane64(case, plane[:rows], None).reshape(rows, F)
        chunk = [None, None, None]
        if case["kv"] == "bf16":
            chunk = [s.k.double().view(-1, F), s.v.double().view(-1, F), None]
        elif case["kv"] == "q8":
            chunk[2] = torch.stack([s.k.double().abs().amax(-1), s.v.double().abs().amax(-1)],
                                   -1) / 127
        return {"prefix": prefix, "chunk": chunk, "ring": None, "bad": None}
    if kind == "swiglu":
        g = s.gate.double()
        return {"out": g * torch.sigmoid(g) * s.up.double(), "bad": None}
    if kind == "combine":
        x = s.x.double()
        for e in range(8):
            x = x + s.down[:, e].double() * s.weights[:, e:e + 1].double()
        y = _norm64(x, s.gamma)
        scales = y.abs().amax(-1) / 448 if case["fp8"] else None
        return {"x": x, "y": y, "packed": None, "scales": scales, "bad": None}
    if kind == "norm_fp8":
        y = _norm64(s.x.double(), s.gamma)
        return {"y": y, "packed": None, "scales": y.abs().amax(-1) / 448, "bad": None}
    return _exact_attention(case, s)
