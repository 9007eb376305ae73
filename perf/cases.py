"""What a serving engine has the KV-cache hot path do, as measurable cases.

Every case is one engine step's work as a program sees it: the step's rows
(decode rows of one query token, prefill chunks of several) over a paged pool
whose blocks lie scattered, called through the package's public entry points:

* ``attention``: ``paged_flash_attention`` of one layer, the metadata of the
  step in hand as it is for every layer after the first;
* ``layer``: ``hip_paged_attention_forward``, what a model calls per layer:
  the step's K/V appended, then attention;
* ``append``: ``_PagedKVCache.write`` alone;
* ``copy``: ``_PagedKVCache.copy_blocks``, the copy-on-write of a step;
* ``step``: ``step_inputs`` and then every layer, the whole KV side of a step.

Row lengths come from the case itself (``lens`` seeds them), values and block
placement from the seed given to ``prepare``.
"""
import importlib
import math
import random

import torch

sea = importlib.import_module("serving-engine_amd")

BLOCK = sea.BLOCK_SIZE
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

_DEFAULTS = dict(kind="attention", dtype="bf16", hq=32, hkv=8, d=128, layout="kv-interleaved", layers=1,
                 decode_rows=0, decode_lo=0, decode_hi=0, shared=0, chunks=0, chunk_lo=0, chunk_hi=0,
                 prior_lo=0, prior_hi=0, pairs=0, partition=0, deterministic=False, lens=1)


def _case(**kw):
    return {**_DEFAULTS, **kw}


def listed():
    return [
        # The smallest step: four short fp32 conversations, multi-head
        # attention at head_dim 64.  Latency and launches.
        _case(name="layer_fp32_4rows", kind="layer", dtype="fp32", hq=12, hkv=12, d=64,
              decode_rows=4, decode_lo=17, decode_hi=130),
        # One interactive user: a single decode row of a GQA model.
        _case(name="decode_1row", decode_rows=1, decode_lo=1001, decode_hi=1001),
        # An ordinary decode batch of a serving engine: 64 conversations.
        _case(name="decode_64rows", decode_rows=64, decode_lo=128, decode_hi=2048, lens=2),
        # 256 conversations behind one system prompt: the first 64 blocks are
        # the same physical blocks.
        _case(name="decode_prefix_256rows", decode_rows=256, decode_lo=64, decode_hi=512, shared=1024, lens=4),
        # Long documents: 16 rows of 32k tokens, 2 GB of K/V per layer.
        _case(name="decode_long_16rows", decode_rows=16, decode_lo=32768, decode_hi=32768),
        # A step under a 256-token budget: 31 decode rows and what is left of
        # the budget as one prompt's next chunk.
        _case(name="mixed_budget_256", decode_rows=31, decode_lo=256, decode_hi=2048, chunks=1, chunk_lo=225,
              chunk_hi=225, prior_lo=1024, prior_hi=1024, lens=5),
        # A loaded engine with chunked prefill: 8 chunks of 512 tokens on
        # contexts of up to 4096, beside 56 decode rows; append included.
        _case(name="layer_mixed_8x512", kind="layer", decode_rows=56, decode_lo=256, decode_hi=2048, chunks=8,
              chunk_lo=512, chunk_hi=512, prior_lo=0, prior_hi=4096, lens=3),
        # A whole 8192-token prompt in one step (no token budget).
        _case(name="prefill_8192", chunks=1, chunk_lo=8192, chunk_hi=8192),
        # A ragged step of a model whose query groups hold three heads.
        _case(name="ragged_24_8_heads", hq=24, hkv=8, decode_rows=13, decode_lo=17, decode_hi=1500, chunks=5,
              chunk_lo=3, chunk_hi=300, prior_lo=0, prior_hi=700, lens=7),
        # Prompts of a small fp32 model (8 query heads on 2 kv heads).
        _case(name="prefill_fp32_3prompts", dtype="fp32", hq=8, hkv=2, d=64, chunks=3, chunk_lo=201, chunk_hi=512,
              lens=8),
        # Copy-on-write of a step that forks 256 requests: 32 layers at once.
        _case(name="copy_256pairs_32layers", kind="copy", layers=32, pairs=256),
        # The whole KV side of a decode step: metadata, launch list, then
        # append and attention of 16 layers, fp16 at head_dim 64.
        _case(name="step_16rows_16layers", kind="step", dtype="fp16", d=64, layers=16, decode_rows=16,
              decode_lo=64, decode_hi=1024, lens=9),
    ]


# Head counts and head_dim of the models an engine serves.
_SHAPES = [(32, 8, 128), (32, 8, 128), (32, 8, 128), (8, 8, 128), (16, 8, 128), (64, 8, 128), (32, 8, 64),
           (24, 8, 128), (16, 4, 256), (12, 4, 96), (12, 12, 64), (8, 2, 64)]
# Bounds of a drawn case: K/V and query bytes, and attention operations (fp32
# arithmetic runs at a sixteenth of the 16-bit rate).
_MAX_BYTES = 2 << 30
_MAX_FLOPS = 5e11


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        limit = _MAX_FLOPS / 16 if c["dtype"] == "fp32" else _MAX_FLOPS
        if w["bytes"] <= _MAX_BYTES and w["flops"] <= limit:
            return c


def _draw(rng):
    hq, hkv, d = rng.choice(_SHAPES)
    c = _case(hq=hq, hkv=hkv, d=d, dtype=rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"]),
              layout=rng.choice(["kv-interleaved"] * 4 + ["head-major", "token-major"]),
              lens=rng.randrange(1, 1 << 20))
    kind = rng.choice(["decode"] * 4 + ["prefill"] * 3 + ["mixed"] * 4 + ["append", "copy", "step"])
    if kind == "copy":
        c.update(kind="copy", layers=_log_int(rng, 1, 32), pairs=_log_int(rng, 1, 256))
        return c
    if kind == "append":
        if rng.random() < 0.5:
            c.update(kind="append", decode_rows=_log_int(rng, 1, 256), decode_lo=16, decode_hi=2048)
        else:
            c.update(kind="append", chunks=1, chunk_lo=16, chunk_hi=_log_int(rng, 16, 8192))
        return c
    if kind in ("decode", "mixed", "step"):
        hi = _log_int(rng, 32, 32768)
        lo = hi if rng.random() < 0.2 else max(1, int(hi * rng.uniform(0.05, 0.9)))
        c.update(decode_rows=_log_int(rng, 1, 256), decode_lo=lo, decode_hi=hi)
        if kind == "decode":
            if rng.random() < 0.2:
                c["shared"] = BLOCK * _log_int(rng, 4, 256)
            c["deterministic"] = rng.random() < 0.15
            c["partition"] = rng.choice([0] * 9 + [512])
    if kind in ("prefill", "mixed"):
        hi = _log_int(rng, 2, 8192 if kind == "prefill" else 1024)
        prior = 0 if rng.random() < 0.3 else _log_int(rng, 16, 16384)
        c.update(chunks=1 if rng.random() < 0.5 else _log_int(rng, 1, 16), chunk_lo=max(2, int(hi * rng.uniform(0.2, 1.0))),
                 chunk_hi=hi, prior_lo=prior // 4, prior_hi=prior)
    if kind == "step":
        c.update(kind="step", layers=_log_int(rng, 2, 24))
        if rng.random() < 0.5:
            c.update(chunks=1, chunk_lo=16, chunk_hi=256, prior_lo=0, prior_hi=1024)
    elif rng.random() < 0.3:
        c["kind"] = "layer"
    return c


# ------------------------------------------------------------------ lengths --

def _rows(c):
    """(q_len, k_len, position of the first query) of every row."""
    rng = random.Random(c["lens"])
    rows = []
    for _ in range(c["decode_rows"]):
        k = c["shared"] + rng.randint(c["decode_lo"], c["decode_hi"])
        rows.append((1, k, k - 1))
    for _ in range(c["chunks"]):
        q = rng.randint(c["chunk_lo"], c["chunk_hi"])
        p = rng.randint(c["prior_lo"], c["prior_hi"])
        rows.append((q, p + q, p))
    return rows


def _nblocks(k):
    return -(-k // BLOCK)


def _es(c):
    return 4 if c["dtype"] == "fp32" else 2


def work(case):
    c = {**_DEFAULTS, **case}
    es, kv_row = _es(c), 2 * c["hkv"] * c["d"] * _es(c)
    if c["kind"] == "copy":
        return {"bytes": 2.0 * c["pairs"] * c["layers"] * BLOCK * kv_row, "flops": 0.0}
    rows = _rows(c)
    tokens = sum(q for q, _, _ in rows)
    appended = tokens * (2 * kv_row + 8)
    if c["kind"] == "append":
        return {"bytes": float(appended), "flops": 0.0}
    # a shared prefix's keys are read once for all the rows that read them
    keys = sum(k for _, k, _ in rows) - c["shared"] * max(0, c["decode_rows"] - 1)
    nbytes = keys * kv_row + tokens * c["hq"] * (2 * c["d"] * es + 4) + 4 * sum(_nblocks(k) for _, k, _ in rows)
    pairs = sum(q * p + q * (q + 1) // 2 for q, _, p in rows)
    if c["kind"] in ("layer", "step"):
        # the step's own keys are read from the new K/V
        nbytes += appended - tokens * kv_row
    layers = c["layers"] if c["kind"] == "step" else 1
    return {"bytes": float(layers * nbytes), "flops": float(layers * 4 * c["hq"] * c["d"] * pairs)}


# ------------------------------------------------------------------- inputs --

def _tables(c, rows, seed):
    """(block table of every row, blocks in the pool): scattered blocks, a
    quarter of the pool unused; decode rows begin with the shared blocks."""
    ns = c["shared"] // BLOCK
    need = [_nblocks(k) - (ns if i < c["decode_rows"] else 0) for i, (_, k, _) in enumerate(rows)]
    total = ns + sum(need)
    n = max(4, -(-5 * total // 4))
    ids = random.Random(seed).sample(range(n), total)
    common, at, out = ids[:ns], ns, []
    for i, m in enumerate(need):
        out.append((common if i < c["decode_rows"] else []) + ids[at:at + m])
        at += m
    return out, n


def _values(c, seed, n, tokens):
    """Generator of the pool's K/V per layer, [N, Hkv, 2, block, D], then a
    function giving Q, K and V of the step's tokens, [T, heads, D]."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kw = dict(generator=gen, device="cuda", dtype=DTYPES[c["dtype"]])
    layers = (torch.randn(n, c["hkv"], 2, BLOCK, c["d"], **kw) for _ in range(c["layers"]))
    return layers, lambda heads: torch.randn(tokens, heads, c["d"], **kw)


def _inputs(c, seed):
    rows = _rows(c)
    if c["kind"] == "copy":
        n = max(4, 2 * c["pairs"] + c["pairs"] // 2)
        ids = random.Random(seed).sample(range(n), 2 * c["pairs"])
        layers, _ = _values(c, seed, n, 0)
        return rows, (ids[:c["pairs"]], ids[c["pairs"]:]), n, layers, None
    tables, n = _tables(c, rows, seed)
    layers, tokens = _values(c, seed, n, sum(q for q, _, _ in rows))
    return rows, tables, n, layers, tokens


def _scheduler_output(c, rows, tables):
    out = sea.SchedulerOutput()
    for i, ((q, k, p), t) in enumerate(zip(rows, tables)):
        rid = f"r{i}"
        if i < c["decode_rows"]:
            req = sea.Request(rid, [0] * (k - 1), output_token_ids=[0], phase=sea.RequestPhase.NEEDS_DECODE,
                              block_table=t, num_computed_tokens=k - 1)
        else:
            req = sea.Request(rid, [0] * k, phase=sea.RequestPhase.NEEDS_PREFILL, block_table=t, num_computed_tokens=p)
            out.prefill_chunk_sizes[rid] = q
        out.scheduled_requests.append(req)
    return out


class _Layer:
    def __init__(self, idx):
        self.layer_idx = idx


class _State:
    pass


def prepare(case, seed):
    c = {**_DEFAULTS, **case}
    rows, tables, n, layers, tokens = _inputs(c, seed)
    s = _State()
    s.case = c
    pool = sea.allocate_kv_cache(c["layers"], n, c["hkv"], c["d"], dtype=DTYPES[c["dtype"]], device="cuda",
                                 layout=c["layout"])
    for i, vals in enumerate(layers):
        pool[i].copy_(vals.permute(2, 0, 3, 1, 4))
    s.cache = sea._PagedKVCache(pool)
    if c["kind"] == "copy":
        s.src, s.dst = tables
        return s
    s.scale = 1.0 / math.sqrt(c["d"])
    # [T, heads, D] from the projections; the model hands them on as [1, heads, T, D]
    q, k, v = tokens(c["hq"]), tokens(c["hkv"]), tokens(c["hkv"])
    s.q, s.q4 = q, q.transpose(0, 1).unsqueeze(0)
    s.k4, s.v4 = k.transpose(0, 1).unsqueeze(0), v.transpose(0, 1).unsqueeze(0)
    s.modules = [_Layer(i) for i in range(c["layers"])]
    s.step = _scheduler_output(c, rows, tables)
    if c["kind"] != "step":
        s.meta, s.slots, _ = sea.step_inputs(s.step, "cuda", s.cache)
    s.kb, s.vb = s.cache.blocks(0)
    return s


def run(state):
    s, c = state, state.case
    kind = c["kind"]
    if kind == "attention":
        return sea.paged_flash_attention(s.q, s.kb, s.vb, s.meta, c["hq"], c["hkv"], s.scale,
                                         partition_tokens=c["partition"], deterministic=c["deterministic"])
    if kind == "copy":
        s.cache.copy_blocks(s.src, s.dst)
        return s.cache.kv_cache
    if kind == "append":
        s.cache.write(s.k4, s.v4, 0, s.slots)
        return s.kb, s.vb
    if kind == "layer":
        o, _ = sea.hip_paged_attention_forward(s.modules[0], s.q4, s.k4, s.v4, None, s.scale, cache=s.cache,
                                               write_index=s.slots, paged_metadata=s.meta)
        return o, s.kb, s.vb
    meta, slots, positions = sea.step_inputs(s.step, "cuda", s.cache)
    outs = []
    for module in s.modules:
        o, _ = sea.hip_paged_attention_forward(module, s.q4, s.k4, s.v4, None, s.scale, cache=s.cache,
                                               write_index=slots, paged_metadata=meta)
        outs.append(o)
    return outs, slots, positions, s.cache.kv_cache


def tolerance(case):
    c = {**_DEFAULTS, **case}
    if c["kind"] in ("append", "copy"):
        return "exact"
    return dict(_TOLERANCE[c["dtype"]])


# bf16 and fp16: probabilities rounded to the type before their product with
# V, and outputs rounded to it; fp32: sums in another order.
_TOLERANCE = {"bf16": {"rel": 1e-2, "max": 1e-1}, "fp16": {"rel": 1.5e-3, "max": 1.5e-2},
              "fp32": {"rel": 4e-6, "max": 4e-5}}


# -------------------------------------------------------------------- exact --

def _attend(q, k, v, first):
    """q [n, Hq, D] at positions first.. over k, v [m, Hkv, D], causal, fp64:
    (o [n, Hq, D], natural-log sum of exponentials [n, Hq])."""
    n, hq, d = q.shape
    m, hkv, _ = k.shape
    g = hq // hkv
    qh = q.double().view(n, hkv, g, d).permute(1, 2, 0, 3).reshape(hkv, g * n, d)
    kh = k.double().permute(1, 2, 0).contiguous()  # [Hkv, D, m]
    vh = v.double().permute(1, 0, 2).contiguous()  # [Hkv, m, D]
    hidden = torch.arange(m, device=q.device)[None, :] > first + torch.arange(n, device=q.device)[:, None]
    hidden = hidden.repeat(g, 1)
    o, lse = [], []
    step = max(1, (1 << 28) // max(1, g * n * m))  # kv heads whose scores fit 2 GB
    for h in range(0, hkv, step):
        s = torch.matmul(qh[h:h + step], kh[h:h + step]) / math.sqrt(d)
        s.masked_fill_(hidden, -math.inf)
        ls = torch.logsumexp(s, dim=-1)
        o.append(torch.matmul(torch.exp_(s.sub_(ls[..., None])), vh[h:h + step]))
        lse.append(ls)
        del s
    o = torch.cat(o).view(hkv, g, n, d).permute(2, 0, 1, 3).reshape(n, hq, d)
    return o, torch.cat(lse).view(hkv, g, n).permute(2, 0, 1).reshape(n, hq)


def exact(case, seed):
    c = {**_DEFAULTS, **case}
    if c["kind"] in ("append", "copy"):
        return None
    rows, tables, n, layers, tokens = _inputs(c, seed)
    pools = list(layers)
    q, nk, nv = tokens(c["hq"]), tokens(c["hkv"]), tokens(c["hkv"])
    outs = []
    for pool in pools:
        o, lse, at = [], [], 0
        for (ql, kl, p), t in zip(rows, tables):
            kv = pool[torch.tensor(t, device="cuda")]  # [blocks, Hkv, 2, block, D]
            kv = kv.permute(2, 0, 3, 1, 4).reshape(2, -1, c["hkv"], c["d"])[:, :kl]
            if c["kind"] != "attention":  # the step's tokens hold the appended K/V
                kv = kv.clone()
                kv[0, p:p + ql], kv[1, p:p + ql] = nk[at:at + ql], nv[at:at + ql]
            ro, rl = _attend(q[at:at + ql], kv[0], kv[1], p)
            o.append(ro)
            lse.append(rl)
            at += ql
        outs.append((torch.cat(o), torch.cat(lse)))
    if c["kind"] == "attention":
        return outs[0]
    if c["kind"] == "layer":
        return outs[0][0].unsqueeze(0), None, None
    return [o.unsqueeze(0) for o, _ in outs], None, None, None
