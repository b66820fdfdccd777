"""Timed cases of the public entry points: decode attention over compressed
and plain BF16 KV, the decode loop (append, plan update, attention), the
prefill and single-tensor encoders, and container decode.

A case is a dict of plain values; ``op`` says which call it makes:

  attend   kvexp_hip_attention_run of a kept plan (Context.plan / Plan.run)
  loop     128 steps of AppendSet.append + torch.ops.kvexp.decode_attention_kv
  prefill  AppendSet.append of whole prompts into empty caches
  encode   kvexp_hip_encode of one tensor (returns its size, so it waits)
  decode   Context.decode of one container

Keys: K = N(0, 1) times a per-channel scale 2^U(-6, 4) with two channels x 32,
6 % of the 128-token blocks in a band of three binades (they encode as 2-bit);
values: N(0, 0.5^2) with 0.3 % of the elements 20 binades down (escapes).
Queries are scaled so that a score's standard deviation is about 3, as
1 / sqrt(head_dim) leaves it in a model.
"""
import ctypes
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "compressed-kv-attention_amd"))

import kvexp_amd  # noqa: E402
from kvexp_amd import torch_ops  # noqa: E402

STEPS = 128  # decode steps of one `loop` pass: one new block per container


def listed():
    return [
        # one KV head and one query at 8K tokens: the smallest call, where launches and latency count
        dict(name="attend_one_head", op="attend", sequences=1, heads=1, group=1, dim=64, seq=8192, block=128, order=0,
             raw=False, lse=True),
        # a decode step of a 24-layer model, 2 KV heads x 7 queries, 32K context (the benchmark's shape)
        dict(name="attend_32k", op="attend", sequences=1, heads=48, group=7, dim=64, seq=32768, block=128, order=0,
             raw=False, lse=False),
        # the same model over a batch of sequences of 1K to 32K tokens, in the AVX-512 BF16 score order
        dict(name="attend_ragged", op="attend", sequences=8, heads=48, group=7, dim=64, seq=32768, block=128, order=1,
             raw=False, lse=False),
        # eight layers x 8 KV heads x 4 queries at head_dim 128 and 64K tokens: the largest
        dict(name="attend_d128_64k", op="attend", sequences=1, heads=64, group=4, dim=128, seq=65536, block=128,
             order=0, raw=False, lse=False),
        # the widest head, the longest blocks and a ragged last block
        dict(name="attend_d256", op="attend", sequences=4, heads=8, group=8, dim=256, seq=25003, block=255, order=0,
             raw=False, lse=False),
        # a head_dim that is no power of two
        dict(name="attend_d96", op="attend", sequences=1, heads=64, group=4, dim=96, seq=16411, block=128, order=0,
             raw=False, lse=False),
        # plain BF16 KV at 8K tokens (the recent, uncompressed part of a cache), odd length
        dict(name="attend_raw_8k", op="attend", sequences=1, heads=48, group=7, dim=64, seq=8191, block=128, order=0,
             raw=True, lse=False),
        # 128 steps of a decode loop at 8K tokens: every step appends a token to 96 containers and attends
        dict(name="loop_8k", op="loop", heads=48, group=7, dim=64, seq=8192 + 37, block=128),
        # a 32K-token prompt of the 24-layer model compressed: 96 containers in one call
        dict(name="prefill_32k", op="prefill", caches=96, dim=64, seq=32768, block=128),
        # prompts at head_dim 256, where a block holds 32,768 elements
        dict(name="prefill_d256", op="prefill", caches=32, dim=256, seq=8150, block=128),
        # one tensor of a short prompt
        dict(name="encode_one", op="encode", dim=64, seq=4099, block=128),
        # a long container back to BF16
        dict(name="decode_d128", op="decode", dim=128, seq=131072, block=128),
    ]


def _log(rng, lo, hi):
    """An integer between lo and hi, spread over their logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    dim = rng.choice([32, 64, 64, 80, 96, 128, 128, 192, 256])
    block = rng.choice([128, 128, 128, 64, 255])
    op = rng.choice(["attend"] * 6 + ["loop", "prefill", "prefill", "encode", "decode"])
    if op == "attend":
        sequences = rng.choice([1, 1, 2, 4])
        heads = _log(rng, 1, 64)
        tokens = 100_000_000 // (dim * heads * sequences)  # at most attend_32k's elements
        return dict(op="attend", sequences=sequences, heads=heads, group=rng.randint(1, 8), dim=dim,
                    seq=max(300, min(_log(rng, 300, 65536), tokens)), block=block,
                    order=int(dim % 32 == 0 and rng.random() < 0.3), raw=rng.random() < 0.25,
                    lse=rng.random() < 0.2)
    if op == "loop":
        heads = _log(rng, 2, 48)
        return dict(op="loop", heads=heads, group=rng.randint(1, 8), dim=rng.choice([64, 128]), seq=_log(rng, 600, 8192),
                    block=128)
    if op == "prefill":
        caches = _log(rng, 2, 96)
        return dict(op="prefill", caches=caches, dim=dim,
                    seq=max(300, min(_log(rng, 300, 32768), 100_000_000 // (dim * caches))), block=block)
    return dict(op=op, dim=dim, seq=_log(rng, 300, 131072), block=block)


# ------------------------------------------------------------------ inputs --
def lengths(case):
    """Tokens of each sequence of an attend case: all alike, or for a batch spread over [1/32, 1] of the longest
    (the same for every seed)."""
    n, seq = case["sequences"], case["seq"]
    if n == 1:
        return [seq]
    r = random.Random(n * 1000003 + seq)
    return [seq] + [max(1, _log(r, max(1, seq // 32), seq)) for _ in range(n - 1)]


def _generator(seed, *pos):
    g = torch.Generator(device="cuda")
    s = seed
    for p in pos:
        s = (s * 1000003 + p + 1) % (1 << 62)
    g.manual_seed(s)
    return g


def _keys(g, n, seq, dim):
    """[n, seq, dim] BF16 keys and the channels' scales."""
    scale = torch.exp2(torch.rand(n, 1, dim, generator=g, device="cuda") * 10 - 6)
    out = torch.rand(n, 1, dim, generator=g, device="cuda").argsort(2) < 2
    scale = torch.where(out, scale * 32, scale)
    k = torch.empty(n, seq, dim, dtype=torch.bfloat16, device="cuda")
    for i in range(n):
        x = torch.randn(seq, dim, generator=g, device="cuda")
        narrow = (torch.rand((seq + 127) // 128, generator=g, device="cuda") < 0.06).repeat_interleave(128)[:seq, None]
        band = torch.rand(seq, dim, generator=g, device="cuda") * 1.7475 + 0.25  # 0.25 to below 2: three binades
        k[i] = (torch.where(narrow, torch.copysign(band, x), x) * scale[i]).to(torch.bfloat16)
    return k, scale


def _values(g, n, seq, dim):
    v = torch.empty(n, seq, dim, dtype=torch.bfloat16, device="cuda")
    for i in range(n):
        x = torch.randn(seq, dim, generator=g, device="cuda") * 0.5
        v[i] = torch.where(torch.rand(seq, dim, generator=g, device="cuda") < 0.003, x * 2.0**-20, x).to(torch.bfloat16)
    return v


def _queries(g, scale, n_q):
    """[n, n_q, dim] BF16 queries for keys of these channel scales."""
    n, _, dim = scale.shape
    norm = scale.square().sum(2, keepdim=True).sqrt()
    return (torch.randn(n, n_q, dim, generator=g, device="cuda") * 3 / norm).to(torch.bfloat16)


def _attend_inputs(case, seed):
    """Per sequence (k, v, q); the queries of every sequence's heads one after another."""
    parts = []
    for i, length in enumerate(lengths(case)):
        g = _generator(seed, 1, i)
        k, scale = _keys(g, case["heads"], length, case["dim"])
        v = _values(g, case["heads"], length, case["dim"])
        parts.append((k, v, _queries(g, scale, case["group"])))
    return parts


def _loop_inputs(case, seed):
    """Keys and values of the context and the steps after it, and each step's queries."""
    g = _generator(seed, 2)
    k, scale = _keys(g, case["heads"], case["seq"] + STEPS, case["dim"])
    v = _values(g, case["heads"], case["seq"] + STEPS, case["dim"])
    q = torch.stack([_queries(g, scale, case["group"]) for _ in range(STEPS)])
    return k, v, q


def _tokens(case, seed, n):
    """[n, seq, dim] BF16 bits, the first half keys and the rest values."""
    g = _generator(seed, 3)
    nk = (n + 1) // 2
    k = _keys(g, nk, case["seq"], case["dim"])[0]
    return torch.cat([k, _values(g, n - nk, case["seq"], case["dim"])]).view(torch.int16)


_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = kvexp_amd.Context(0)
    return _ctx


def _caches(ctx, n, dim, tokens, block):
    """n empty appendable containers in a pool: their bytes and indexes are rows of three tensors."""
    cap = max(kvexp_amd.encode_bound(tokens, dim, block), 1)
    cap = (cap + 255) // 256 * 256
    nb = (tokens + block - 1) // block + 1
    pool = dict(blob=torch.zeros(n, cap, dtype=torch.uint8, device="cuda"),
                offsets=torch.zeros(n, nb, dtype=torch.int64, device="cuda"),
                first=torch.zeros(n, nb, dtype=torch.int32, device="cuda"))
    caches = []
    for i in range(n):
        c = kvexp_amd.Cache(ctx, dim, 1, block)
        c.max_tokens, c.capacity, c.index_capacity = tokens, cap, nb
        c.blob, c.offsets, c.first = pool["blob"][i], pool["offsets"][i], pool["first"][i]
        c.append(None, 0)
        caches.append(c)
    return caches, pool


def _rewind(aset, tokens):
    """The set's containers at their first `tokens` tokens again (what follows is appended anew)."""
    aset.jobs["n_tokens"] = tokens
    for c in aset.caches:
        c.seq = tokens


# ------------------------------------------------------------------- cases --
def prepare(case, seed):
    ctx = _context()
    op = case["op"]
    s = dict(case=case, ctx=ctx)
    if op == "attend":
        heads, q = [], []
        seqs = [n for n in lengths(case) for _ in range(case["heads"])]
        splits = ctx.suggest_splits_batch(seqs, case["block"], case["dim"], case["group"], case["order"])
        for k, v, qs in _attend_inputs(case, seed):
            q.append(qs)
            for h in range(case["heads"]):
                kh, vh = k[h].view(torch.int16), v[h].view(torch.int16)
                n = kh.shape[0]
                if case["raw"]:
                    heads.append(dict(k=kh, v=vh, seq=n, splits=splits))
                else:
                    heads.append(dict(kx=ctx.encode(kh, n, case["dim"], case["block"]),
                                      vx=ctx.encode(vh, n, case["dim"], case["block"]), seq=n, splits=splits))
        s["q"] = torch.cat(q).contiguous()
        s["plan"] = ctx.plan(heads, case["group"], case["dim"], case["block"], case["order"])
        s["out"] = torch.zeros(s["q"].shape, dtype=torch.float32, device="cuda")
        s["lse"] = torch.zeros(s["q"].shape[:2], dtype=torch.float32, device="cuda") if case["lse"] else None
    elif op == "loop":
        k, v, s["q"] = _loop_inputs(case, seed)
        n, seq, dim = case["heads"], case["seq"], case["dim"]
        tokens = torch.cat([k, v]).view(torch.int16)
        caches, s["pool"] = _caches(ctx, 2 * n, dim, seq + STEPS, case["block"])
        s["set"] = ctx.append_set(caches)
        s["set"].append(tokens[:, :seq].contiguous(), seq)
        s["new"] = tokens[:, seq:].transpose(0, 1).contiguous()
        s["kv"] = torch_ops.register_kv(caches[:n], caches[n:], case["group"], dim,
                                        ctx.suggest_splits(n, seq, case["block"], dim, case["group"]), case["block"])
    elif op == "prefill":
        s["tokens"] = _tokens(case, seed, case["caches"])
        caches, s["pool"] = _caches(ctx, case["caches"], case["dim"], case["seq"], case["block"])
        s["set"] = ctx.append_set(caches)
    elif op == "encode":
        s["tokens"] = _tokens(case, seed, 1)
        nb = (case["seq"] + case["block"] - 1) // case["block"] + 1
        s["blob"] = torch.zeros(kvexp_amd.encode_bound(case["seq"], case["dim"], case["block"]), dtype=torch.uint8,
                                device="cuda")
        s["offsets"] = torch.zeros(nb, dtype=torch.int64, device="cuda")
        s["first"] = torch.zeros(nb, dtype=torch.int32, device="cuda")
    else:
        s["enc"] = ctx.encode(_tokens(case, seed, 1), case["seq"], case["dim"], case["block"])
        s["out"] = torch.zeros(case["seq"] * case["dim"], dtype=torch.int16, device="cuda")
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    op = case["op"]
    if op == "attend":
        s["plan"].run(s["q"], s["out"], s["lse"])
        return [s["out"]] if s["lse"] is None else [s["out"], s["lse"]]
    if op == "loop":
        _rewind(s["set"], case["seq"])
        n, outs = case["heads"], []
        for i in range(STEPS):
            s["set"].append(s["new"][i], 1)
            outs.append(torch.ops.kvexp.decode_attention_kv(s["q"][i], s["kv"], [case["seq"] + i + 1] * n))
        return [torch.stack(outs), s["pool"]["blob"], s["pool"]["offsets"], s["pool"]["first"]]
    if op == "prefill":
        _rewind(s["set"], 0)
        s["set"].append(s["tokens"], case["seq"])
        return [s["pool"]["blob"], s["pool"]["offsets"], s["pool"]["first"]]
    if op == "encode":
        size = ctypes.c_size_t(0)
        kvexp_amd.check(kvexp_amd.lib().kvexp_hip_encode(
            ctx.h, s["tokens"].data_ptr(), case["seq"], case["dim"], case["block"], s["blob"].data_ptr(),
            s["blob"].numel(), s["offsets"].data_ptr(), s["first"].data_ptr(), ctypes.byref(size),
            torch.cuda.current_stream().cuda_stream))
        return [s["blob"], s["offsets"], s["first"], size.value]
    return [ctx.decode(s["enc"], out=s["out"])]


def _coded(tokens, dim, block):
    """Bytes of a container of this many tokens, all blocks 4-bit, without escapes."""
    return (tokens + block - 1) // block * (8 + dim) + tokens * dim * 3 // 2


def work(case):
    op, dim = case["op"], case["dim"]
    if op == "attend":
        ns, n_q = lengths(case), case["group"]
        kv = sum(4 * n * dim if case["raw"] else 2 * _coded(n, dim, case["block"]) for n in ns) * case["heads"]
        rows = len(ns) * case["heads"] * n_q
        return dict(bytes=kv + rows * dim * 6 + (rows * 4 if case["lse"] else 0),
                    flops=4 * dim * n_q * case["heads"] * sum(ns))
    if op == "loop":
        n, n_q = case["heads"], case["group"]
        kv = 2 * n * _coded(case["seq"] + STEPS // 2, dim, case["block"])
        tail = 2 * n * (dim * 2 + _coded(case["block"] // 2, dim, case["block"]))  # a token in, its block out
        return dict(bytes=STEPS * (kv + tail + n * n_q * dim * 6),
                    flops=STEPS * 4 * dim * n_q * n * (case["seq"] + STEPS // 2))
    n = case["caches"] if op == "prefill" else 1
    return dict(bytes=n * (2 * case["seq"] * dim + _coded(case["seq"], dim, case["block"])), flops=0)


def tolerance(case):
    # bytes, indexes and tokens are whole values, the same from every correct
    # codec; attention sums thousands of 32-bit products: measured against 64
    # bits, the outputs are at most 2.4e-6 off (2-norm)
    if case["op"] in ("attend", "loop"):
        return {"rel": 1e-5}
    return "exact"


def _attention64(k, v, q):
    """[n_q, dim] attention and [n_q] log-sum-exp of one head in 64 bits."""
    s = q.double() @ k.double().T
    m = s.max(1, keepdim=True).values
    e = torch.exp(s - m)
    total = e.sum(1, keepdim=True)
    return (e @ v.double()) / total, (m + torch.log(total))[:, 0]


def exact(case, seed):
    op = case["op"]
    if op == "attend":
        out, lse = [], []
        for k, v, q in _attend_inputs(case, seed):
            for h in range(case["heads"]):
                o, l64 = _attention64(k[h], v[h], q[h])
                out.append(o)
                lse.append(l64)
        return [torch.stack(out)] + ([torch.stack(lse)] if case["lse"] else [])
    if op == "loop":
        k, v, q = _loop_inputs(case, seed)
        n = case["heads"]
        out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
        for h in range(n):
            kd, vd = k[h].double(), v[h].double()
            s = q[:, h].double() @ kd.T  # [steps, n_q, tokens]
            at = torch.arange(kd.shape[0], device="cuda")
            seen = at[None, :] <= case["seq"] + torch.arange(STEPS, device="cuda")[:, None]
            out[:, h] = torch.softmax(s.masked_fill(~seen[:, None], -math.inf), 2) @ vd
        return [out, None, None, None]
    if op == "decode":
        return [_tokens(case, seed, 1).reshape(-1)]
    return None
