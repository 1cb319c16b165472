"""The work that users of this package have it do, as timed cases over its public entry points.

A case is a dict of plain values; `kind` says which path it takes:

  attend    one decode step of attention over compressed pages (`PagedKVPool.decode_attention` or, with exact recent
            tokens read in place from the engine's paged cache, `.decode_attention_ring`)
  serve     one layer's part of a serving engine's decode step: the step's tokens are written into the pages and the
            attention over them is answered (`BatchedLayerState.write` + `.attend`)
  write     quantise and store tokens (`PagedKVPool.append` for runs of one length, `.append_ragged` for prompts)
  chat      one sequence through the store: prompt, then tokens one by one, each captured and attended to
            (`KVCaptureEngine`, `compute_hybrid_attention`)
  estimate  keys to codes, all inner products with a block of queries, codes back to keys (`TurboQuantProd`)
  cache     the self-contained cache: a prompt, then tokens one by one (`TurboQuantKVCache`)

`listed()` names one size of each kind of use; `draw()` gives others of the same ranges.
"""

import math
import types

import torch

from turboquant_amd.capture import KVCaptureEngine
from turboquant_amd.integration.batched import BatchedLayerState
from turboquant_amd.integration.vllm import LayerConfig
from turboquant_amd.kv_cache import TurboQuantKVCache
from turboquant_amd.paged import PAGE_TOKENS, PagedKVPool
from turboquant_amd.quantizer import TurboQuantProd
from turboquant_amd.score import compute_hybrid_attention
from turboquant_amd.store import CompressedKVStore

GROUP = 32                                  # channels per value group, the default everywhere
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEVICE = "cuda:0"


def listed():
    return [
        # ---- decode: attention over compressed history -------------------------------------------------------------
        # a batch of chats of a grouped-query model, compressed history only
        dict(name="gqa_batch", kind="attend", seqs=16, shortest=8192, longest=8192, q_heads=32, kv_heads=8, head_dim=128,
             key_bits=3, value_bits=4, ring=0, dtype="bf16"),
        # a few documents of 131,072 tokens, wide heads, the smallest codes
        dict(name="long_context", kind="attend", seqs=4, shortest=131072, longest=131072, q_heads=16, kv_heads=2,
             head_dim=256, key_bits=3, value_bits=2, ring=0, dtype="bf16"),
        # many requests of very different length at once, the first layers' 4-bit keys, the newest 128 tokens exact, an
        # odd number of heads per KV head
        dict(name="ragged_hybrid", kind="attend", seqs=96, shortest=61, longest=8190, q_heads=40, kv_heads=8, head_dim=128,
             key_bits=4, value_bits=4, ring=128, dtype="fp16"),
        # latent attention: every query head on one KV head of 576
        dict(name="latent_batch", kind="attend", seqs=16, shortest=8192, longest=8192, q_heads=128, kv_heads=1,
             head_dim=576, key_bits=4, value_bits=4, ring=0, dtype="bf16"),
        # the largest: a layer of a full decode batch, page write and attention, the newest tokens exact
        dict(name="serve_full_batch", kind="serve", seqs=32, shortest=32768, longest=32768, q_heads=32, kv_heads=8,
             head_dim=128, key_bits=3, value_bits=4, ring=128, dtype="bf16"),
        # ---- quantise and store ------------------------------------------------------------------------------------
        # the page write of a decode step: one token of each sequence, where launches and latency are what counts
        dict(name="token_write", kind="write", seqs=32, shortest=1, longest=1, kv_heads=8, head_dim=128, key_bits=3,
             value_bits=4, dtype="bf16", held=1000),
        # a prompt of 32,768 tokens
        dict(name="prompt_write", kind="write", seqs=1, shortest=32768, longest=32768, kv_heads=8, head_dim=128,
             key_bits=3, value_bits=2, dtype="bf16", held=0),
        # a prefill step of several prompts of odd lengths behind what their sequences hold already, wide heads
        dict(name="prompts_ragged", kind="write", seqs=9, shortest=17, longest=4099, kv_heads=2, head_dim=256, key_bits=3,
             value_bits=2, dtype="fp16", held=77),
        # a prompt of latent keys and values
        dict(name="prompt_latent", kind="write", seqs=1, shortest=8192, longest=8192, kv_heads=1, head_dim=576, key_bits=4,
             value_bits=4, dtype="bf16", held=0),
        # ---- one sequence ------------------------------------------------------------------------------------------
        # a chat turn in one layer: prompt, then reply tokens one by one, all of them small calls
        dict(name="chat_turn", kind="chat", prompt=1500, reply=24, q_heads=32, kv_heads=8, head_dim=128, key_bits=3,
             value_bits=2, ring=128, dtype="bf16"),
        # keys -> codes -> inner products and back, in fp32: the smallest case
        dict(name="key_estimates", kind="estimate", heads=1, keys=4096, queries=32, head_dim=128, key_bits=3, dtype="fp32"),
        # the cache object with a prompt and a few tokens behind it (its buffers and weights meet in fp32 products)
        dict(name="cache_object", kind="cache", batch=1, heads=8, prompt=4096, reply=8, head_dim=128, key_bits=3,
             value_bits=2, buffer=128, dtype="fp32"),
    ]


# ---- drawn cases ----------------------------------------------------------------------------------------------------------

def _between(rng, lo, hi):
    """A whole number spread over the logarithm of lo .. hi."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _geometry(rng, kind):
    d = rng.choice([64, 128, 128, 128, 256, 576])
    if d == 576:
        kv = 1
    elif d == 256:
        kv = rng.choice([1, 2, 4, 8])
    else:
        kv = rng.choice([1, 2, 4, 8, 8])
    per = rng.choice([8, 16, 32, 64, 128]) if d == 576 else rng.choice([1, 2, 4, 4, 5, 7, 8, 8, 16])
    c = dict(kv_heads=kv, head_dim=d, key_bits=rng.choice([4, 4, 3]) if d == 576 else rng.choice([2, 3, 3, 3, 4]),
             value_bits=rng.choice([2, 4, 4]), dtype=rng.choice(["bf16", "bf16", "bf16", "fp16"]))
    if kind != "write":
        c["q_heads"] = kv * per
    return c


def draw(rng):
    """A case of the same ranges, no more work than the largest listed ones."""
    most = [work(c) for c in listed()]
    while True:
        case = _draw(rng)
        w = work(case)
        if all(w[k] <= max(m[k] for m in most) for k in ("bytes", "flops")):
            return case


def _draw(rng):
    kind = rng.choice(["attend", "attend", "attend", "serve", "write", "write", "write", "chat", "estimate", "cache"])
    if kind in ("attend", "serve"):
        c = _geometry(rng, kind)
        longest = _between(rng, 200, 131072)
        shortest = longest if rng.random() < 0.5 else max(33, longest // rng.choice([2, 8, 100]))
        cost = longest * c["kv_heads"] * c["head_dim"]
        room = (1 << 30) // cost
        if c["head_dim"] == 576:
            room = min(room, (1 << 24) // (longest * c["q_heads"]))
        c["seqs"] = _between(rng, 1, max(1, min(256, room)))
        c.update(kind=kind, shortest=shortest, longest=longest, ring=rng.choice([0, 128]))
        return c
    if kind == "write":
        c = _geometry(rng, kind)
        if rng.random() < 0.35:
            c.update(kind=kind, seqs=_between(rng, 1, 256), shortest=1, longest=1, held=_between(rng, 1, 2000))
            return c
        longest = _between(rng, 16, 32768 if c["head_dim"] < 576 else 8192)
        room = (32768 * 8 * 128 if c["head_dim"] < 576 else 8192 * 576) // (longest * c["kv_heads"] * c["head_dim"])
        c.update(kind=kind, seqs=_between(rng, 1, max(1, min(32, room))), longest=longest,
                 shortest=longest if rng.random() < 0.3 else max(1, longest // rng.choice([2, 10, 200])),
                 held=rng.choice([0, 0, 77, 512]))
        if c["head_dim"] == 576 and c["seqs"] * longest > 8192:
            c["seqs"] = 1
        return c
    if kind == "chat":
        d = rng.choice([64, 128, 128, 256])
        kv = rng.choice([2, 4, 8])
        return dict(kind=kind, prompt=_between(rng, 100, 8000), reply=_between(rng, 8, 32), kv_heads=kv,
                    q_heads=kv * rng.choice([1, 4, 5, 8]), head_dim=d, key_bits=rng.choice([3, 3, 4]),
                    value_bits=rng.choice([2, 4]), ring=128, dtype=rng.choice(["bf16", "fp16"]))
    if kind == "estimate":
        heads = rng.choice([1, 2, 8])
        return dict(kind=kind, heads=heads, keys=_between(rng, 300, 16384), queries=_between(rng, 1, 128),
                    head_dim=rng.choice([64, 128, 128, 256]), key_bits=rng.choice([2, 3, 3, 4]),
                    dtype=rng.choice(["fp32", "bf16"]))
    return dict(kind="cache", batch=rng.choice([1, 1, 2]), heads=rng.choice([4, 8]), prompt=_between(rng, 150, 8000),
                reply=_between(rng, 2, 8), head_dim=rng.choice([64, 128, 128]), key_bits=rng.choice([3, 3, 4]),
                value_bits=rng.choice([2, 4]), buffer=128, dtype="fp32")


# ---- inputs ---------------------------------------------------------------------------------------------------------------

def _rows(gen, shape, dtype, outliers=None):
    """N(0, 1) rows (..., heads, d); `outliers` (heads, d) scales the few channels in which real keys are large."""
    x = torch.randn(*shape, generator=gen, device=DEVICE, dtype=torch.float32)
    if outliers is not None:
        x *= outliers
    return x.to(dtype)


def _outliers(gen, heads, d):
    """Scales of (heads, d) channels: four per head ten times as large as the others."""
    s = torch.ones(heads, d, device=DEVICE)
    picked = torch.rand(heads, d, generator=gen, device=DEVICE).argsort(dim=1)[:, :4]
    return s.scatter_(1, picked, 10.0)


def _lengths(case):
    """One length per sequence, spread over the logarithm of shortest .. longest; the first is the longest."""
    n, lo, hi = case["seqs"], case["shortest"], case["longest"]
    return [int(round(hi * (lo / hi) ** (i / max(1, n - 1)))) for i in range(n)]


def _pool(case, quantizer, pages):
    return PagedKVPool(quantizer, case["kv_heads"], pages, value_bits=case["value_bits"], value_group_size=GROUP,
                       dtype=DTYPES[case["dtype"]], device=torch.device(DEVICE))


def _table(gen, lengths):
    """Block tables of sequences whose pages lie anywhere in the pool: (B, longest) int32 and the pool's page count."""
    width = max(-(-n // PAGE_TOKENS) for n in lengths)
    pages = len(lengths) * width
    order = torch.rand(pages, generator=gen, device=DEVICE).argsort().to(torch.int32)
    return order.reshape(len(lengths), width).contiguous(), pages


def _fill(pool, gen, case, table, lengths, scales):
    """Every sequence's first lengths[b] tokens, written the way an engine writes a prompt."""
    dtype = DTYPES[case["dtype"]]
    for b, n in enumerate(lengths):
        if n > 0:
            shape = (1, n, case["kv_heads"], case["head_dim"])
            pool.append(_rows(gen, shape, dtype, scales), _rows(gen, shape, dtype), table[b:b + 1])


def _sections(pool):
    """The pages as the numbers that they hold: packed keys, (norm, residual norm) pairs, packed values, scales and zeros."""
    L, data = pool.layout, pool.data
    d, groups = pool.head_dim, pool.head_dim // pool.value_group_size
    keys = data[..., L.off_keys:L.off_keys + L.d // 8 * (L.mse_bits + 1) * PAGE_TOKENS]
    norms = data[..., L.off_meta:L.off_meta + 8 * PAGE_TOKENS].view(torch.float32)
    codes = data[..., L.off_vdata:L.off_vdata + d * L.value_bits // 8 * PAGE_TOKENS]
    size = 2 * groups * PAGE_TOKENS
    scale = data[..., L.off_vscale:L.off_vscale + size].view(pool.dtype)
    zero = data[..., L.off_vzero:L.off_vzero + size].view(pool.dtype)
    return {"keys": keys, "norms": norms, "codes": codes, "scale": scale, "zero": zero}


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dev, dtype, d = torch.device(DEVICE), DTYPES[case["dtype"]], case["head_dim"]
    kind = case["kind"]
    s = types.SimpleNamespace(case=case)

    if kind in ("attend", "serve", "write"):
        s.quantizer = TurboQuantProd(d, bits=case["key_bits"], device=dev)
        lengths = _lengths(case)
        scales = _outliers(gen, case["kv_heads"], d)

    if kind in ("attend", "serve"):
        s.table, pages = _table(gen, lengths)
        s.pool = _pool(case, s.quantizer, pages)
        _fill(s.pool, gen, case, s.table, lengths, scales)
        s.seq_lens = torch.tensor(lengths, dtype=torch.int32, device=dev)
        s.longest = max(lengths)
        s.query = _rows(gen, (case["seqs"], case["q_heads"], d), dtype)
        s.exact = None
        if case["ring"]:
            s.exact = _rows(gen, (2, pages, PAGE_TOKENS, case["kv_heads"], d), dtype)
        if kind == "serve":
            cfg = LayerConfig(head_dim=d, num_kv_heads=case["kv_heads"], num_query_heads=case["q_heads"],
                              key_bits=case["key_bits"], value_bits=case["value_bits"], value_group_size=GROUP,
                              ring_capacity=case["ring"] or 128, device=dev)
            s.layer = BatchedLayerState(config=cfg, quantizer=s.quantizer, pool=s.pool)
            n = case["seqs"]
            s.meta = types.SimpleNamespace(num_actual_tokens=n, max_query_len=1, max_seq_len=s.longest,
                                           seq_lens=s.seq_lens, block_table=s.table,
                                           query_start_loc=torch.arange(n + 1, dtype=torch.int32, device=dev))
            s.key = _rows(gen, (n, case["kv_heads"], d), dtype, scales)
            s.value = _rows(gen, (n, case["kv_heads"], d), dtype)

    elif kind == "write":
        held = case["held"]
        ragged = len(set(lengths)) > 1
        # (what a sequence holds before this step's run varies by a few tokens, as it does in a batch)
        before = [held + 7 * b % 23 if held else 0 for b in range(case["seqs"])]
        s.table, pages = _table(gen, [n + h for n, h in zip(lengths, before)])
        s.pool = _pool(case, s.quantizer, pages)
        _fill(s.pool, gen, case, s.table, before, scales)
        s.start = torch.tensor(before, dtype=torch.int32, device=dev) if held or ragged else None
        s.ragged = ragged
        if ragged:
            rows = (sum(lengths), case["kv_heads"], d)
            s.run_len = torch.tensor(lengths, dtype=torch.int32, device=dev)
            s.row0 = (torch.cumsum(s.run_len, 0) - s.run_len).to(torch.int32)
            s.max_run = max(lengths)
        else:
            rows = (case["seqs"], lengths[0], case["kv_heads"], d)
        s.key, s.value = _rows(gen, rows, dtype, scales), _rows(gen, rows, dtype)
        s.sections = _sections(s.pool)

    elif kind == "chat":
        n = case["prompt"] + case["reply"]
        s.store = CompressedKVStore(head_dim=d, num_kv_heads=case["kv_heads"], key_bits=case["key_bits"],
                                    value_bits=case["value_bits"], value_group_size=GROUP, device=dev)
        s.engine = KVCaptureEngine(s.store, ring_capacity=case["ring"], device=dev, dtype=dtype)
        s.key = _rows(gen, (n, case["kv_heads"], d), dtype, _outliers(gen, case["kv_heads"], d))
        s.value = _rows(gen, (n, case["kv_heads"], d), dtype)
        s.query = _rows(gen, (n, case["q_heads"], d), dtype)

    elif kind == "estimate":
        s.quantizer = TurboQuantProd(d, bits=case["key_bits"], device=dev)
        x = _rows(gen, (case["heads"], case["keys"], d), torch.float32)
        length = 0.5 + 1.5 * torch.rand(case["heads"], case["keys"], 1, generator=gen, device=dev)
        s.key = (x / x.norm(dim=-1, keepdim=True) * length).to(dtype)
        s.query = _rows(gen, (case["heads"], case["queries"], d), dtype)

    else:
        s.cache = TurboQuantKVCache(d, key_bits=case["key_bits"], value_bits=case["value_bits"], value_group_size=GROUP,
                                    buffer_size=case["buffer"], device=dev, dtype=dtype)
        shape = (case["batch"], case["heads"], case["prompt"] + case["reply"], d)
        s.key = _rows(gen, shape, dtype) * _outliers(gen, case["heads"], d)[None, :, None]
        s.value = _rows(gen, shape, dtype)
        s.query = _rows(gen, shape[:2] + (case["reply"], d), dtype)
    return s


# ---- one pass -------------------------------------------------------------------------------------------------------------

def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "attend":
        if s.exact is not None:
            return s.pool.decode_attention_ring(s.query, s.table, s.seq_lens, s.exact[0], s.exact[1], case["ring"],
                                                max_len=s.longest)
        return s.pool.decode_attention(s.query, s.table, s.seq_lens, max_len=s.longest)
    if kind == "serve":
        s.layer.write(s.key, s.value, s.meta)
        return s.layer.attend(s.query, s.meta, kv_cache=s.exact, hybrid=s.exact is not None)
    if kind == "write":
        if s.ragged:
            s.pool.append_ragged(s.key, s.value, s.row0, s.run_len, s.start, s.table, max_run=s.max_run)
        else:
            s.pool.append(s.key, s.value, s.table, start_pos=s.start)
        return s.sections
    if kind == "chat":
        n = case["prompt"]
        s.engine.reset()
        s.engine.ingest_prefill(s.key[:n], s.value[:n], n)
        outs = []
        for t in range(n, n + case["reply"]):
            s.engine.ingest_decode(s.key[t:t + 1], s.value[t:t + 1], 1)
            recent_k, recent_v = s.engine.ring.peek()
            outs.append(compute_hybrid_attention(s.query[t:t + 1], s.store, recent_k, recent_v, case["q_heads"]))
        return outs
    if kind == "estimate":
        code = s.quantizer.quantize(s.key)
        scores = s.quantizer.attention_score(s.query, code)
        return {"indices": code.mse_indices, "signs": code.qjl_signs, "norms": code.norms,
                "residual_norms": code.residual_norms, "scores": scores, "keys": s.quantizer.dequantize(code)}
    n = case["prompt"]
    s.cache.prefill(s.key[..., :n, :], s.value[..., :n, :])
    outs = []
    for i in range(case["reply"]):
        t = n + i
        s.cache.append(s.key[..., t:t + 1, :], s.value[..., t:t + 1, :])
        scores = s.cache.attention_scores(s.query[..., i:i + 1, :])
        outs.append((scores, s.cache.attend(torch.softmax(scores, dim=-1))))
    return outs


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------

def _token_bytes(d, key_bits, value_bits, size):
    """Bytes of a token of one KV head in the store: key codes and signs, two norms, value codes, scales and zeros."""
    return d * key_bits // 8 + size + 4 + d * value_bits // 8 + 2 * size * (d // GROUP)


def work(case):
    kind, d, kb = case["kind"], case["head_dim"], case["key_bits"]
    size = 4 if case["dtype"] == "fp32" else 2
    if kind in ("attend", "serve"):
        lengths, hkv, hq = _lengths(case), case["kv_heads"], case["q_heads"]
        exact = sum(min(n, case["ring"]) for n in lengths)
        held = sum(lengths) - exact
        stored = _token_bytes(d, kb, case["value_bits"], size)
        nbytes = hkv * (held * stored + exact * 2 * d * size) + 2 * case["seqs"] * hq * d * size
        # score on the indices, score on the signs, value: 2 d each; the query's two products with d x d matrices
        flops = hq * (held * 6 * d + exact * 4 * d) + case["seqs"] * hq * 4 * d * d
        if kind == "serve":
            nbytes += case["seqs"] * hkv * (2 * d * size + stored)
            flops += case["seqs"] * hkv * 6 * d * d
        return {"bytes": nbytes, "flops": flops}
    if kind == "write":
        vectors = sum(_lengths(case)) * case["kv_heads"]
        nbytes = vectors * (2 * d * size + _token_bytes(d, kb, case["value_bits"], size)) + 2 * 4 * d * d
        return {"bytes": nbytes, "flops": vectors * 6 * d * d}
    if kind == "chat":
        hkv, hq, n, ring = case["kv_heads"], case["q_heads"], case["prompt"], case["ring"]
        stored = _token_bytes(d, kb, case["value_bits"], size)
        old = n if n >= ring else 0                         # (a full ring moves to the store with the first reply token)
        old += sum(1 for t in range(n, n + case["reply"]) if n < ring <= t) and ring
        nbytes = hkv * (old * (2 * d * size + stored))
        flops = old * hkv * 6 * d * d
        for t in range(case["reply"]):
            recent = n + t + 1 - old
            nbytes += hkv * (old * stored + max(0, recent) * 2 * d * size) + 2 * hq * d * size
            flops += hq * (old * 6 * d + max(0, recent) * 4 * d + 4 * d * d)
        return {"bytes": nbytes, "flops": flops}
    if kind == "estimate":
        vectors, nq = case["heads"] * case["keys"], case["heads"] * case["queries"]
        mse = kb - 1
        width = 1 if mse == 1 else (2 if mse == 2 else 4)
        code = d * width // 8 + d // 8 + size + 4
        nbytes = vectors * (d * size + code + 4 * d + 4 * case["queries"]) + nq * d * size
        return {"bytes": nbytes, "flops": vectors * (6 + 4) * d * d + vectors * case["queries"] * 4 * d + nq * 4 * d * d}
    heads, n, reply, buf = case["batch"] * case["heads"], case["prompt"], case["reply"], case["buffer"]
    mse = kb - 1
    width = 1 if mse == 1 else (2 if mse == 2 else 4)
    code = d * width // 8 + d // 8 + size + 4 + d * case["value_bits"] // 8 + 2 * size * (d // GROUP)
    new = max(0, n + reply - buf)
    nbytes = heads * new * (2 * d * size + code)
    flops = heads * new * 6 * d * d
    for t in range(reply):
        total = n + t + 1
        recent = min(total, buf)
        nbytes += heads * ((total - recent) * code + recent * 2 * d * size + 3 * d * size + total * 8)
        flops += heads * ((total - recent) * 6 * d + recent * 4 * d + 4 * d * d)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """How far two correct implementations at the same precision come apart.

    Decode: bf16 weights against packed values; seen against a float64 evaluation of the same pages: 2e-3 .. 4e-3, and at
    head_dim 576 5e-3; between two ways to split the tokens 3e-3 .. 6e-3.
    Codes: an index flips where a 32-bit sum falls on the other side of a threshold, in about one vector of 20,000; the
    vector's residual, a tenth of its signs and its inner products change with it (by about a tenth, the residual's norm
    by nothing: the threshold lies half way). Norms seen against float64: 7e-8 .. 2e-7."""
    kind = case["kind"]
    if kind in ("attend", "serve"):
        return {"rel": 0.02, "max": 0.25} if case["head_dim"] == 576 else {"rel": 0.012, "max": 0.16}
    if kind == "chat":
        return {"rel": 0.012, "max": 0.16}
    if kind == "write":
        return {"rel": 1e-6, "max": 1e-4, "differ": 1e-4}
    vectors = case["heads"] * (case["keys"] if kind == "estimate" else case["batch"] * case["prompt"])
    flipped = max(2.0, 2e-4 * vectors) / vectors
    return {"rel": min(0.02, 0.15 * math.sqrt(flipped)), "max": 0.9, "differ": min(0.01, 0.6 * flipped)}
