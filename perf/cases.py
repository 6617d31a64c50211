"""What a user of the paged KV-cache path has it do, as measurable cases.

A case is one layer (or the first few layers) of a serving engine's work: a decode step, a prefill
chunk, a whole prompt, a batched append.  Sizes are the configurations of ``infurnace_amd.workloads``
(Qwen3-0.6B: 16 query / 8 kv heads x 128; Qwen3-8B: 32 / 8 x 128), their tensor-parallel shards, and
sizes around them.  ``listed`` gives the fixed cases, ``draw`` more of the same ranges.

Every case starts from what an engine holds before the call: the pool with earlier tokens' K/V, the
block tables (pages in random order), the lengths, and the step's projections on the GPU.
"""
import math

import torch

from infurnace_amd.kernels import (decode_plan, paged_attention, qk_norm_rope_append, qk_norm_rope_append_and_prefill,
                                   qk_norm_rope_store_and_decode, rope_table, store_kv, store_kv_and_decode,
                                   store_kv_and_prefill, store_kv_layers)

BS = 16            # tokens per page
EPS = 1e-6         # the models' RMSNorm epsilon
ROPE_BASE = 1e6    # the models' rotary base


def listed():
    return [
        # One user's decode step on the small model: the latency of a call (config 1's sizes).
        dict(name="decode_single", kind="decode", form="append", hq=16, hkv=8, d=128, batch=1, lo=512, hi=512,
             layers=4),
        # A lightly loaded server: a few short chats, from the fp32 projections in one call per layer.
        dict(name="decode_short", kind="decode", form="prep", hq=16, hkv=8, d=128, batch=7, lo=33, hi=901, layers=4),
        # The ordinary batch: 32 ragged contexts up to 4096 tokens (config 2's sizes).
        dict(name="decode_ragged", kind="decode", form="append", hq=16, hkv=8, d=128, batch=32, lo=128, hi=4096,
             layers=2),
        # A full server of the larger model: 128 long contexts, attention alone.
        dict(name="decode_large", kind="decode", form="plain", hq=32, hkv=8, d=128, batch=128, lo=1023, hi=8190,
             layers=1),
        # One of two tensor-parallel ranks of the larger model (its heads halved), ordinary contexts.
        dict(name="decode_shard", kind="decode", form="append", hq=16, hkv=4, d=128, batch=48, lo=100, hi=4000,
             layers=2),
        # 64 rows over one cached 4096-token prefix with 512 tokens of their own (config 5's sizes).
        dict(name="decode_shared", kind="shared", hq=32, hkv=8, d=128, batch=64, prefix=4096, own_min=512, own=512,
             layers=2),
        # A 2048-token prompt in four 512-token chunks (config 3's sizes).
        dict(name="prefill_chunks", kind="prefill", form="append", hq=16, hkv=8, d=128, start=0, tokens=512, chunks=4),
        # The rest of a prompt after a prefix-cache hit: odd length, at a page boundary that is no tile boundary.
        dict(name="prefill_ragged", kind="prefill", form="append", hq=32, hkv=8, d=128, start=720, tokens=333,
             chunks=1),
        # A chunk from the fp32 projections through the single fused call.
        dict(name="prefill_prep", kind="prefill", form="fused", hq=16, hkv=8, d=128, start=1024, tokens=512, chunks=1),
        # A large chunk deep in a long prompt of the larger model, from the fp32 projections as the runner does it.
        dict(name="prefill_long", kind="prefill", form="prep", hq=32, hkv=8, d=128, start=6144, tokens=2048, chunks=1),
        # A whole long prompt in one call.
        dict(name="prefill_prompt", kind="prefill", form="append", hq=16, hkv=8, d=128, start=0, tokens=8192,
             chunks=1),
        # Every layer's K/V of a 2048-token prompt stored at once (config 3's append).
        dict(name="append_layers", kind="append", hkv=8, d=128, layers=28, tokens=2048),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "shared", "prefill", "prefill", "prefill", "append"])
    if kind == "decode":
        form = rng.choice(["plain", "append", "prep"])
        hq, hkv, d = rng.choice([(16, 8, 128), (16, 8, 128), (32, 8, 128), (32, 8, 128), (8, 4, 128), (16, 4, 128),
                                 (8, 2, 128), (16, 8, 64)])
        batch = _log(rng, 1, 160)
        hi = _log(rng, 64, 8190)
        # (the listed cases' largest: about 590,000 keys)
        hi = max(64, min(hi, 590000 // batch))
        lo = rng.randint(1, hi)
        keys = batch * (lo + hi) // 2
        return dict(kind=kind, form=form, hq=hq, hkv=hkv, d=d, batch=batch, lo=lo, hi=hi,
                    layers=4 if keys < 10000 else 2 if keys < 100000 else 1)
    if kind == "shared":
        own = _log(rng, 17, 1024)
        return dict(kind=kind, hq=rng.choice([16, 32]), hkv=8, d=128, batch=_log(rng, 2, 96),
                    prefix=BS * _log(rng, 64, 512), own_min=rng.randint(1, own), own=own, layers=2)
    if kind == "prefill":
        hq, hkv, d = rng.choice([(16, 8, 128), (16, 8, 128), (32, 8, 128), (16, 4, 128), (16, 8, 64)])
        form = rng.choice(["append", "append", "prep", "fused"])
        tokens = _log(rng, 17, 6000)
        if form == "fused":  # (aligned starts are what that call takes; ordinary chunk sizes)
            tokens = min(tokens, 2048)
            start = 32 * rng.randint(0, 64)
        else:
            start = rng.choice([0, BS * rng.randint(0, 256), rng.randint(0, 4096)])
        while 4 * hq * d * tokens * (start + tokens / 2) > 2.6e11:  # (no more than the listed prompts)
            tokens = tokens * 3 // 4
        return dict(kind=kind, form=form, hq=hq, hkv=hkv, d=d, start=start, tokens=tokens, chunks=1)
    hkv, d = rng.choice([(8, 128), (8, 128), (4, 128), (8, 64)])
    return dict(kind=kind, hkv=hkv, d=d, layers=rng.choice([1, 28, 36]), tokens=_log(rng, 1, 1600))


# ---- sizes that depend on the case alone ----------------------------------------------------------


def _lens(c):
    """The rows' lengths: spread over [lo, hi] (golden-ratio steps), one row at hi."""
    if c["kind"] == "shared":  # every row its own tail
        lo, hi = c["prefix"] + c["own_min"], c["prefix"] + c["own"]
    else:
        lo, hi = c["lo"], c["hi"]
    return [hi - int((i * 0.6180339887498949 % 1.0) * (hi - lo)) for i in range(c["batch"])]


def _pages(n):
    return -(-n // BS)


def _starts(c):
    return [c["start"] + i * c["tokens"] for i in range(c["chunks"])]


def work(c):
    """Each key and value row once, the queries and outputs, the appended rows; 4 hq d flops a (query, key) pair."""
    hkv, d = c["hkv"], c["d"]
    row = 2 * 2 * hkv * d  # a token's K and V
    if c["kind"] == "append":
        n = c["layers"] * c["tokens"]
        return {"bytes": 2 * n * row + 4 * c["tokens"], "flops": 0}
    hq = c["hq"]
    prep = c.get("form") in ("prep", "fused")
    q_in = hq * d * (4 if prep else 2)
    new = row * (2 if prep else 1) if c.get("form") != "plain" else 0  # the step's own K/V as they arrive
    put = row if c.get("form") != "plain" else 0
    if c["kind"] in ("decode", "shared"):
        lens = _lens(c)
        n = sum(lens)
        keys = n - (c["batch"] - 1) * c["prefix"] if c["kind"] == "shared" else n
        keys -= c["batch"] if new else 0  # (an appended key arrives with the step)
        rows = c["batch"] * (q_in + 2 * hq * d + new + put + (d * 4 if prep else 0))
        table = 4 * sum(_pages(x) for x in lens) + 4 * c["batch"]
        return {"bytes": c["layers"] * (keys * row + rows + table), "flops": c["layers"] * 4 * hq * d * n}
    total, flops = 0, 0
    t = c["tokens"]
    for s in _starts(c):
        total += s * row + t * (q_in + 2 * hq * d + new + put + (d * 4 if prep else 0)) + 4 * _pages(s + t)
        flops += 4 * hq * d * (t * s + t * (t + 1) // 2)
    return {"bytes": total, "flops": flops}


def tolerance(c):
    if c["kind"] == "append":
        return "exact"
    # (fp16 inputs, outputs and probabilities: up to 4.6e-4 and 3.5e-3 from 64 bits measured)
    return {"rel": 2e-3, "max": 1.5e-2}


# ---- inputs ---------------------------------------------------------------------------------------


def _rand(gen, *shape, scale=1.0, dtype=torch.float16):
    t = torch.randn(shape, generator=gen, device="cuda", dtype=dtype)
    return t.mul_(scale) if scale != 1.0 else t


def _pool(c, gen, layers, pages):
    return _rand(gen, layers, 2, pages, BS, c["hkv"], c["d"])


def _norms(c, gen, state, max_positions):
    """Norm weights around one and the rotary table, kept by a model for its life."""
    state["qw"] = 1.0 + 0.1 * _rand(gen, c["d"], dtype=torch.float32)
    state["kw"] = 1.0 + 0.1 * _rand(gen, c["d"], dtype=torch.float32)
    state["rope"] = rope_table(max_positions, c["d"], ROPE_BASE, device="cuda")


def prepare(c, seed):
    """Queries are scaled by 2, so that the softmax has a spread like a trained model's rather than a flat one."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)
    s = {"case": c}
    hkv, d = c["hkv"], c["d"]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    if c["kind"] == "append":
        pages = _pages(c["tokens"]) + 32
        s["pool"] = _pool(c, gen, c["layers"], pages)
        order = torch.randperm(pages, generator=gen, device="cuda")
        pos = torch.arange(c["tokens"], device="cuda")
        s["slots"] = (order[pos // BS] * BS + pos % BS).to(torch.int32)
        s["k"] = _rand(gen, c["layers"], c["tokens"], hkv, d)
        s["v"] = _rand(gen, c["layers"], c["tokens"], hkv, d)
        return s
    hq = c["hq"]
    if c["kind"] in ("decode", "shared"):
        b, lens, layers = c["batch"], _lens(c), c["layers"]
        need = [_pages(x) for x in lens]
        common = c["prefix"] // BS if c["kind"] == "shared" else 0
        pages = common + sum(n - common for n in need) + 16
        s["pool"] = _pool(c, gen, layers, pages)
        order = torch.randperm(pages, generator=gen, device="cuda").to(torch.int32).cpu()
        table = torch.full((b, max(need)), int(order[-1]), dtype=torch.int32)
        at = common
        for i, n in enumerate(need):
            table[i, :common] = order[:common]
            table[i, common:n] = order[at:at + n - common]
            at += n - common
        last = torch.tensor(lens) - 1
        slots = table[torch.arange(b), last // BS] * BS + last % BS
        s["table"], s["lens"], s["slots"], s["max_len"] = table.cuda(), i32(lens), slots.to(torch.int32).cuda(), max(lens)
        if c["kind"] == "shared":
            s["prefix"] = order[:common].clone().cuda()
        if c.get("form") == "prep":
            s["q"] = _rand(gen, layers, b, hq, d, dtype=torch.float32)
            s["k"] = _rand(gen, layers, b, hkv, d, dtype=torch.float32)
            s["v"] = _rand(gen, layers, b, hkv, d, dtype=torch.float32)
            s["pos"] = i32([x - 1 for x in lens])
            _norms(c, gen, s, max(lens))
        else:
            s["q"] = _rand(gen, layers, b, hq, d, scale=2.0)
            s["k"] = _rand(gen, layers, b, hkv, d)
            s["v"] = _rand(gen, layers, b, hkv, d)
        return s
    total = c["start"] + c["tokens"] * c["chunks"]
    pages = _pages(total) + 16
    s["pool"] = _pool(c, gen, 1, pages)
    order = torch.randperm(pages, generator=gen, device="cuda")
    s["table"] = order[:_pages(total)].to(torch.int32)
    pos = torch.arange(c["start"], total, device="cuda")
    s["slots"] = (order[pos // BS] * BS + pos % BS).to(torch.int32)
    s["pos"] = pos.to(torch.int32)
    n = c["tokens"] * c["chunks"]
    if c["form"] == "append":
        s["q"], s["k"], s["v"] = _rand(gen, n, hq, d, scale=2.0), _rand(gen, n, hkv, d), _rand(gen, n, hkv, d)
    else:
        f32 = torch.float32
        s["q"], s["k"], s["v"] = (_rand(gen, n, hq, d, dtype=f32), _rand(gen, n, hkv, d, dtype=f32),
                                  _rand(gen, n, hkv, d, dtype=f32))
        _norms(c, gen, s, total)
    return s


# ---- one pass -------------------------------------------------------------------------------------


def run(s):
    c = s["case"]
    pool = s["pool"]
    if c["kind"] == "append":
        store_kv_layers(pool, s["slots"], None, s["k"], s["v"])
        return {"pool": pool}
    if c["kind"] == "decode":
        outs, table, lens, form = [], s["table"], s["lens"], c["form"]
        slots = None if form == "plain" else s["slots"]
        # (a step of several layers keeps one plan for them, as the runner does)
        plan = (decode_plan(s["q"][0].shape, pool, table, lens, None, slots, max_seq_len=s["max_len"], lazy=True)
                if c["layers"] > 1 else None)
        for i in range(c["layers"]):
            if form == "plain":
                o = paged_attention(s["q"][i], pool, table, lens, layer=i, max_seq_len=s["max_len"], plan=plan)
            elif form == "append":
                o = store_kv_and_decode(s["q"][i], pool, table, lens, None, slots, s["k"][i], s["v"][i], layer=i,
                                        max_seq_len=s["max_len"], plan=plan)
            else:
                o = qk_norm_rope_store_and_decode(s["q"][i], s["k"][i], s["v"][i], s["qw"], s["kw"], s["rope"],
                                                  s["pos"], slots, None, pool, table, lens, layer=i, eps=EPS,
                                                  max_seq_len=s["max_len"], plan=plan)
            outs.append(o)
        return {"out": outs} if form == "plain" else {"out": outs, "pool": pool}
    if c["kind"] == "shared":
        outs = []
        for i in range(c["layers"]):
            store_kv(pool, s["slots"], None, s["k"][i], s["v"][i], layer=i)
            outs.append(paged_attention(s["q"][i], pool, s["table"], s["lens"], layer=i, max_seq_len=s["max_len"],
                                        shared_prefix_pages=s["prefix"]))
        return {"out": outs, "pool": pool}
    outs = []
    for i, start in enumerate(_starts(c)):
        part = slice(i * c["tokens"], (i + 1) * c["tokens"])
        q, k, v = s["q"][part], s["k"][part], s["v"][part]
        if c["form"] == "append":
            o = store_kv_and_prefill(q, pool, s["table"], k, v, query_start=start)
        elif c["form"] == "fused":
            o = qk_norm_rope_append_and_prefill(q, k, v, s["qw"], s["kw"], s["rope"], pool, s["table"],
                                                query_start=start, eps=EPS)
        else:
            q16 = qk_norm_rope_append(q, k, v, s["qw"], s["kw"], s["rope"], s["pos"][part], s["slots"][part], None,
                                      pool, eps=EPS)
            o = paged_attention(q16, pool, s["table"], None, query_start=start)
        outs.append(o)
    return {"out": outs, "pool": pool}


# ---- the same in 64 bits --------------------------------------------------------------------------


def _norm_rope64(x, w, rope, pos):
    x = x.double()
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()
    half = x.shape[-1] // 2
    cos, sin = rope[pos.long()].double()[:, None, :].split(half, -1)
    a, b = x.split(half, -1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _attend64(q, k, v, limit):
    """q [n, hq, d], k and v [m, hkv, d]; query i sees keys [0, limit[i])."""
    n, hq, d = q.shape
    hkv = k.shape[1]
    g = hq // hkv
    out = torch.empty((n, hq, d), dtype=torch.float64, device=q.device)
    key = torch.arange(k.shape[0], device=q.device)
    for h in range(hkv):
        kt, vh = k[:, h].t().contiguous(), v[:, h].contiguous()
        for at in range(0, n, 1024):
            part = q[at:at + 1024, h * g:(h + 1) * g]
            rows = part.shape[0]
            s = part.reshape(rows * g, d) @ kt / math.sqrt(d)
            hide = key[None, :] >= limit[at:at + 1024, None]
            s = s.view(rows, g, -1).masked_fill_(hide[:, None, :], -math.inf)
            p = torch.softmax(s, -1).view(rows * g, -1)
            out[at:at + 1024, h * g:(h + 1) * g] = (p @ vh).view(rows, g, d)
    return out


def exact(c, seed):
    s = prepare(c, seed)
    hkv, d = c["hkv"], c["d"]
    if c["kind"] == "append":
        return None  # (a copy: compared byte for byte)
    prep = c.get("form") in ("prep", "fused")
    layers = c.get("layers", 1)
    outs = []
    pool = s["pool"].double() if c.get("form") != "plain" else s["pool"]
    slots = s["slots"].long()
    for i in range(layers):
        q, k, v = (s[x][i] if c["kind"] != "prefill" else s[x] for x in "qkv")
        q64, k64, v64 = q.double(), k.double(), v.double()
        if prep:
            q64, k64 = _norm_rope64(q, s["qw"], s["rope"], s["pos"]), _norm_rope64(k, s["kw"], s["rope"], s["pos"])
        flat = pool[i].view(2, -1, hkv, d)
        if c.get("form") != "plain":
            flat[0, slots], flat[1, slots] = k64, v64
        if c["kind"] == "prefill":
            total = c["start"] + c["tokens"] * c["chunks"]
            pos = torch.arange(total, device="cuda")
            at = s["table"].long()[pos // BS] * BS + pos % BS
            limit = torch.arange(c["start"] + 1, total + 1, device="cuda")
            whole = _attend64(q64, flat[0, at], flat[1, at], limit)
            outs = [whole[j * c["tokens"]:(j + 1) * c["tokens"]] for j in range(c["chunks"])]
        else:
            rows = []
            for b, n in enumerate(_lens(c)):
                pos = torch.arange(n, device="cuda")
                at = s["table"][b].long()[pos // BS] * BS + pos % BS
                rows.append(_attend64(q64[b:b + 1], flat[0, at].double(), flat[1, at].double(),
                                      torch.tensor([n], device="cuda")))
            outs.append(torch.cat(rows))
    return {"out": outs} if c.get("form") == "plain" else {"out": outs, "pool": pool}
