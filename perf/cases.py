"""The workloads this backend is timed on: one FULL-attention layer at a time, as vLLM
calls it on one tensor-parallel rank.

Every case goes through a public entry point: ``OscarAttentionBackendImpl.forward`` (the
write and the read of a step), ``do_kv_cache_update`` (the standalone write) or
``ops.rotate``.  A ``forward`` case is a batch: request i has ``histories[i]`` cached
tokens and ``chunks[i]`` new ones; a request without history is a fresh prompt.

A case's fields: ``kind``; ``hq`` / ``hk`` / ``d`` (query heads, KV heads, head width);
``dtype`` of the activations; ``wide`` (legacy slots of 2 d bytes); ``clip`` (the serve
defaults' sort clip, K 0.96 and V 0.92, else none); and the sizes.
"""
import math
import os
import random

import numpy as np
import torch

BLOCK = 128           # tokens per cache page
RECENT = 256          # FP32 window per request (the default)
ARENA_TOKENS = 8192   # seats of the window arena (the default)
KINDS = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# one rank of the served model: 6 query heads on 1 KV head of width 256, bf16
_MODEL = dict(hq=6, hk=1, d=256, dtype="bf16", wide=False, clip=False)


def _text(values):
    return ",".join(str(int(v)) for v in values)


def _numbers(text):
    return [int(v) for v in text.split(",")]


def _ragged(n, low, high, seed):
    r = random.Random(seed)
    return [r.randint(low, high) for _ in range(n)]


def _forward(name, histories, chunks, **other):
    return dict(_MODEL, name=name, kind="forward", histories=_text(histories), chunks=_text(chunks), **other)


def listed():
    narrow = dict(hq=16, hk=2, d=128, dtype="fp16")
    return [
        # one user early in a chat: the smallest step, where launches and latency count
        _forward("decode_1x500", [500], [1]),
        # one user, long context, a token and three drafts to verify
        _forward("verify_1x24k", [24576], [4]),
        # the serving steady state: eight long contexts verifying drafts
        _forward("verify_8x24k", [24576] * 8, [4] * 8),
        # a full server: 64 contexts of any length, one token each, with the serve defaults' clip
        _forward("decode_64_ragged", _ragged(64, 1024, 32768, 5), [1] * 64, clip=True),
        # a model of narrow heads in fp16, two KV heads per rank, legacy slots, odd lengths
        _forward("verify_12_narrow", _ragged(12, 700, 9000, 6), [3] * 12, **dict(_MODEL, **narrow, wide=True)),
        # chunked prefill beside decodes: a chunk of a long prompt, 16 decodes, a short new prompt
        _forward("mixed_chunk_400", [12000] + [8192] * 16 + [0], [400] + [1] * 16 + [700]),
        # a fresh prompt of ordinary length
        _forward("prompt_2048", [0], [2048]),
        # three fresh prompts of odd lengths in one batch, narrow fp16 heads
        _forward("prompts_narrow", [0, 0, 0], [777, 131, 1500], **dict(_MODEL, **narrow)),
        # the largest call: a long continuation of a long cached prompt
        _forward("continue_15360_9256", [15360], [9256]),
        # the standalone write of a long prompt, with the serve defaults' clip
        dict(_MODEL, name="update_15360_clip", kind="update", tokens=15360, clip=True),
        # the standalone write of a medium prompt on a rank that holds four KV heads
        dict(_MODEL, name="update_901_hk4", kind="update", tokens=901, hq=24, hk=4),
        # the inverse rotation of a long chunk's attention output
        dict(name="rotate_back_55536", kind="rotate", rows=55536, d=256, dtype="fp32", out="bf16", transpose=True),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _pairs(case):
    """Visible query-key pairs of a forward batch."""
    return sum(c * h + c * (c + 1) // 2 for h, c in zip(_numbers(case["histories"]), _numbers(case["chunks"])))


def draw(rng):
    """One more case: the same kinds of call over their whole ranges, odd sizes among them."""
    shape = dict(_MODEL)
    shape.update(rng.choice([{}, {}, {}, dict(hq=12, hk=2), dict(hq=8, d=128), dict(hq=16, hk=2, d=128, dtype="fp16"),
                             dict(dtype="fp16")]))
    shape["wide"], shape["clip"] = rng.random() < 0.2, rng.random() < 0.4
    kind = rng.choice(["decode"] * 5 + ["chunk"] * 2 + ["prompt"] * 2 + ["update"] * 2 + ["rotate"])
    if kind == "rotate":
        dtype = rng.choice(["fp32", "bf16", "fp16"])
        return dict(kind="rotate", rows=_log(rng, 5, 55000), d=shape["d"], dtype=dtype,
                    out="bf16" if dtype == "fp32" else dtype, transpose=rng.random() < 0.6)
    if kind == "update":
        return dict(shape, kind="update", tokens=_log(rng, 2, 15000 // shape["hk"]))
    if kind == "decode":
        n = _log(rng, 1, 64)
        top = min(32768, 900000 // (n * shape["hk"]))
        low = _log(rng, 64, top // 2)
        histories, chunks = [rng.randint(low, top) for _ in range(n)], [rng.randint(1, 5)] * n
    elif kind == "prompt":
        n = rng.randint(1, 4)
        histories, chunks = [0] * n, [_log(rng, 33, 4000) for _ in range(n)]
    else:
        n = rng.randint(0, 12)
        histories = [_log(rng, 300, 15000)] + [_log(rng, 200, 8000) for _ in range(n)]
        chunks = [_log(rng, 40, 8000)] + [1] * n
    case = dict(shape, kind="forward", histories=_text(histories), chunks=_text(chunks))
    while 4 * case["d"] * case["hq"] * _pairs(case) > 1.0e12:
        chunks[0] = chunks[0] * 2 // 3
        case["chunks"] = _text(chunks)
    return case


# ---------------------------------------------------------------- inputs (plain torch)
def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _rotation(d, gen):
    """A random-sign normalised Hadamard matrix, fp32."""
    h = torch.ones(1, 1, dtype=torch.float64)
    while h.shape[0] < d:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    sign = (torch.rand(d, generator=gen, device=gen.device) < 0.5).double() * 2 - 1
    return (sign[:, None] * h.to(gen.device) / math.sqrt(d)).float().contiguous()


def _new_kv(n, hk, d, dtype, gen):
    """K or V of new tokens: N(0, 1) with four outlier channels, as key projections have them."""
    x = torch.randn(n, hk, d, generator=gen, device=gen.device)
    x[..., torch.randperm(d, generator=gen, device=gen.device)[:4]] *= 8
    return x.to(dtype)


def _fill(cache_k, cache_v, d, gen):
    """Every slot of the caches as a server leaves it: the INT2 codes, scales and zeros of
    rotated vectors (K slot: four fp16 constants, codes from byte 32; V slot: codes)."""
    k, v = cache_k.view(torch.uint8).view(-1, cache_k.shape[-1]), cache_v.view(torch.uint8).view(-1, cache_v.shape[-1])
    shifts = torch.tensor([1, 4, 16, 64], device=k.device)
    for a in range(0, k.shape[0], 1 << 16):
        b = min(a + (1 << 16), k.shape[0])
        meta = []
        for slots, at in ((k, 32), (v, 0)):
            y = torch.randn(b - a, d, generator=gen, device=k.device) * 1.4
            low, high = y.amin(1, keepdim=True), y.amax(1, keepdim=True)
            scale, zero = ((high - low) / 3).half(), low.half()
            codes = ((y - zero.float()) / scale.float() + 0.5).floor().clamp(0, 3).to(torch.int64)
            slots[a:b, at:at + d // 4] = (codes.view(b - a, d // 4, 4) * shifts).sum(-1).to(torch.uint8)
            meta += [scale, zero]
        k[a:b, :8] = torch.cat(meta, 1).contiguous().view(torch.uint8)


def _read(cache_k, cache_v, d, slots):
    """The fp32 K and V values of cache slots (token slots, all KV heads): [n, hk, d]."""
    hk = cache_k.shape[2]
    k = cache_k.view(torch.uint8).view(-1, hk, cache_k.shape[-1])[slots]
    v = cache_v.view(torch.uint8).view(-1, hk, cache_v.shape[-1])[slots]
    meta = k[..., :8].contiguous().view(torch.float16).float()
    shifts = torch.tensor([0, 2, 4, 6], device=k.device)
    out = []
    for x, s, z in ((k[..., 32:32 + d // 4], meta[..., 0:1], meta[..., 1:2]), (v[..., :d // 4], meta[..., 2:3], meta[..., 3:4])):
        codes = ((x.to(torch.int32)[..., None] >> shifts) & 3).reshape(*x.shape[:-1], d).float()
        out.append(codes * s + z)
    return out


def _last_of(seats):
    """Indexes of the last occurrence of each seat, ascending."""
    _, first = np.unique(seats[::-1], return_index=True)
    return np.sort(len(seats) - 1 - first)


def _inputs(case, seed):
    """Everything a call reads, from the seed alone, as a dict of tensors and host lists."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(seed)
    if case["kind"] == "rotate":
        x = torch.randn(case["rows"], case["d"], generator=gen, device=dev).to(KINDS[case["dtype"]])
        return dict(x=x, r=_rotation(case["d"], gen))
    hq, hk, d, dtype = case["hq"], case["hk"], case["d"], KINDS[case["dtype"]]
    update = case["kind"] == "update"
    histories = [0] if update else _numbers(case["histories"])
    chunks = [case["tokens"]] if update else _numbers(case["chunks"])
    lengths = [h + c for h, c in zip(histories, chunks)]
    pages = [-(-n // BLOCK) for n in lengths]
    blocks = sum(pages) + 8
    order = np.random.default_rng(seed).permutation(blocks).astype(np.int32)
    table = np.zeros((len(pages), max(pages)), np.int32)
    at = 0
    for r, p in enumerate(pages):
        table[r, :p] = order[at:at + p]
        at += p

    def slots_of(r, a, b):
        pos = np.arange(a, b)
        return table[r, pos // BLOCK].astype(np.int64) * BLOCK + pos % BLOCK

    width = 2 * d if case["wide"] else d
    k_cache = torch.zeros(blocks, BLOCK, hk, width, dtype=torch.int8, device=dev)
    v_cache = torch.zeros_like(k_cache)
    rk, rv = _rotation(d, gen), _rotation(d, gen)
    _fill(k_cache, v_cache, d, gen)
    # the window arena: the last RECENT tokens of each history, where the seat is still theirs
    rows = max(-(-ARENA_TOKENS // BLOCK), -(-RECENT // BLOCK) + 3)
    stage_k = torch.zeros(rows, BLOCK, hk, d, dtype=torch.float32, device=dev)
    stage_v = torch.zeros_like(stage_k)
    owner = torch.full((rows, BLOCK), -1, dtype=torch.int64, device=dev)
    held = np.concatenate([slots_of(r, max(h - RECENT, 0), h) for r, h in enumerate(histories)])
    if held.size:
        seats = held // BLOCK % rows * BLOCK + held % BLOCK
        last = _last_of(seats)
        seat, slot = torch.from_numpy(seats[last]).to(dev), torch.from_numpy(held[last]).to(dev)
        for arena, y in zip((stage_k, stage_v), _read(k_cache, v_cache, d, slot)):
            spread = y.amax(-1, keepdim=True) - y.amin(-1, keepdim=True)
            noise = torch.rand(y.shape, generator=gen, device=dev) - 0.5
            arena.view(rows * BLOCK, hk, d)[seat] = y + noise * spread / 3
        owner.view(-1)[seat] = slot // BLOCK
    new = np.concatenate([slots_of(r, h, h + c) for r, (h, c) in enumerate(zip(histories, chunks))])
    n = len(new)
    return dict(
        q=torch.randn(n, hq, d, generator=gen, device=dev).to(dtype), k=_new_kv(n, hk, d, dtype, gen),
        v=_new_kv(n, hk, d, dtype, gen), rk=rk, rv=rv, k_cache=k_cache, v_cache=v_cache, stage_k=stage_k,
        stage_v=stage_v, owner=owner, table=torch.from_numpy(table).to(dev), slots=torch.from_numpy(new).to(dev),
        host_slots=new, host_table=table, starts=[0] + np.cumsum(chunks).tolist(), lengths=lengths, histories=histories)


# ---------------------------------------------------------------- what a server holds
class _Layer:
    layer_name = "model.layers.0.self_attn.attn"


class _Metadata:
    pass


def prepare(case, seed):
    x = _inputs(case, seed)
    if case["kind"] == "rotate":
        x["y"] = torch.empty(x["x"].shape, dtype=KINDS[case["out"]], device=x["x"].device)
        return dict(x, kind="rotate", transpose=case["transpose"])
    from oscar_amd import integration
    from oscar_amd.backend import OscarAttentionBackendImpl

    clip = {"OSCAR_ASCEND_K_CLIP_RATIO": "0.96", "OSCAR_ASCEND_V_CLIP_RATIO": "0.92"} if case["clip"] else {}
    names = ("OSCAR_ASCEND_K_CLIP_RATIO", "OSCAR_ASCEND_V_CLIP_RATIO", "OSCAR_ASCEND_VERBOSE")
    before = {name: os.environ.pop(name, None) for name in names}
    os.environ.update(clip, OSCAR_ASCEND_VERBOSE="0")
    impl = OscarAttentionBackendImpl.__new__(OscarAttentionBackendImpl)
    impl.head_size, impl.num_heads, impl.num_kv_heads = case["d"], case["hq"], case["hk"]
    impl.scale = case["d"] ** -0.5
    impl.key_cache = impl.value_cache = None
    impl._oscar_setup()
    for name in names:
        os.environ.pop(name, None)
        if before[name] is not None:
            os.environ[name] = before[name]
    # the layer as cache initialization leaves it: rotations, window arena, scratch
    layer, cache = _Layer(), (x["k_cache"], x["v_cache"])
    impl._set_caches(cache)
    layer._oscar_rots = (x["rk"], x["rv"])
    impl._ensure_staging(layer, cache)
    layer._oscar_stage_k, layer._oscar_stage_v, layer._oscar_slot_owner = x["stage_k"], x["stage_v"], x["owner"]
    layer._oscar_stage_rows = x["owner"].shape[0]
    n = x["q"].shape[0]
    integration.reserve_device_scratch([impl], [cache], max_tokens=n, max_len=max(x["lengths"]),
                                       max_seqs=len(x["lengths"]))
    md = _Metadata()
    md.num_actual_tokens = n
    md.slot_mapping = x["slots"]
    md.query_start_loc_cpu = torch.tensor(x["starts"], dtype=torch.int32)
    md.seq_lens_list = list(x["lengths"])
    md.block_tables = x["table"]
    q, k, v = (x[name].view(n, -1) for name in "qkv")
    return dict(kind=case["kind"], impl=impl, layer=layer, cache=cache, md=md, q=q, k=k if case["kind"] == "forward" else x["k"],
                v=v if case["kind"] == "forward" else x["v"], out=torch.empty_like(q), slots=x["slots"])


def run(state):
    if state["kind"] == "rotate":
        from oscar_amd import ops

        return ops.rotate(state["x"], state["r"], transpose=state["transpose"], out=state["y"], out_dtype=state["y"].dtype)
    impl, layer, cache = state["impl"], state["layer"], state["cache"]
    if state["kind"] == "update":
        impl.do_kv_cache_update(layer, state["k"], state["v"], cache, state["slots"])
        return dict(k_cache=cache[0], v_cache=cache[1], owner=layer._oscar_slot_owner)
    out = impl.forward(layer, state["q"], state["k"], state["v"], cache, state["md"], output=state["out"])
    return dict(out=out, k_cache=cache[0], v_cache=cache[1], owner=layer._oscar_slot_owner,
                stage_k=layer._oscar_stage_k, stage_v=layer._oscar_stage_v)


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    d = case["d"]
    size = {"bf16": 2, "fp16": 2, "fp32": 4}
    if case["kind"] == "rotate":
        rows = case["rows"]
        return dict(bytes=rows * d * (size[case["dtype"]] + size[case["out"]]) + 4 * d * d, flops=2 * rows * d * d)
    hq, hk = case["hq"], case["hk"]
    slot = 8 + d // 2
    if case["kind"] == "update":
        n = case["tokens"]
        return dict(bytes=n * (hk * (4 * d + slot) + 16) + 8 * d * d, flops=4 * n * hk * d * d)
    histories, chunks = _numbers(case["histories"]), _numbers(case["chunks"])
    n = sum(chunks)
    cached = sum(c for h, c in zip(histories, chunks) if h)
    total = 8 * d * d + n * (hk * (4 * d + slot) + 16 + 4 * hq * d)
    for h, c in zip(histories, chunks):
        staged = min(h, RECENT)
        total += hk * ((h - staged) * slot + staged * 8 * d) + min(c, RECENT) * hk * 8 * d
    # scores and values; the rotations of the new K and V, and of cached requests' queries and outputs
    return dict(bytes=total, flops=4 * d * hq * _pairs(case) + 4 * d * d * (n * hk + cached * hq))


# ---------------------------------------------------------------- exactness
def tolerance(case):
    """Cache bytes and owner tags are exact.  An output is rounded to 16 bits once, and the
    rotated queries, keys and values once before it: another order of the sums shows as
    that many roundings."""
    if case["kind"] == "update":
        return "exact"
    if case["kind"] == "rotate":
        return {"rel": 4e-3, "max": 2e-2} if case["out"] == "bf16" else {"rel": 5e-4, "max": 3e-3}
    if case["dtype"] == "fp16":
        return {"rel": 3e-3, "max": 5e-2}
    return {"rel": 1.2e-2, "max": 2e-1}


def _attend(q, keys, values, history, scale):
    """fp64 attention of one KV head: q [c, heads, d]; query i sees keys [0, history + i + 1)."""
    c = q.shape[0]
    out = torch.empty_like(q)
    pos = torch.arange(keys.shape[0], device=q.device)
    for h in range(q.shape[1]):
        for a in range(0, c, 2048):
            b = min(a + 2048, c)
            s = (q[a:b, h].contiguous() @ keys.t().contiguous()) * scale
            s.masked_fill_(pos[None, :] > history + torch.arange(a, b, device=q.device)[:, None], -math.inf)
            out[a:b, h] = torch.softmax(s, -1) @ values
    return out


def exact(case, seed):
    if case["kind"] == "update":
        return None  # bytes and tags only
    x = _inputs(case, seed)
    if case["kind"] == "rotate":
        r = x["r"].double()
        return x["x"].double() @ (r.t().contiguous() if case["transpose"] else r)
    d, hk, hq, dtype = case["d"], case["hk"], case["hq"], KINDS[case["dtype"]]
    group, rows = hq // hk, x["owner"].shape[0]
    rk, rv = x["rk"].double(), x["rv"].double()
    q, k, v = (x[name].double() for name in "qkv")
    k_rot, v_rot = k @ rk, v @ rv
    # the write: the last token on a seat owns it if it is in its request's window
    slots = x["host_slots"]
    seats = slots // BLOCK % rows * BLOCK + slots % BLOCK
    starts, lengths = x["starts"], x["lengths"]
    position = np.concatenate([np.arange(n - (b - a), n) for n, a, b in zip(lengths, starts, starts[1:])])
    edge = np.concatenate([np.full(b - a, n - RECENT) for n, a, b in zip(lengths, starts, starts[1:])])
    last = _last_of(seats)
    kept = last[position[last] >= edge[last]]
    stage_k, stage_v, owner = x["stage_k"].double(), x["stage_v"].double(), x["owner"].view(-1).clone()
    owner[torch.from_numpy(seats).to(owner.device)] = -1
    seat, token = torch.from_numpy(seats[kept]).to(owner.device), torch.from_numpy(kept).to(owner.device)
    seen = x["stage_k"].view(-1, hk, d), x["stage_v"].view(-1, hk, d)
    out = torch.empty_like(q)
    for r, (a, b) in enumerate(zip(starts, starts[1:])):
        h = x["histories"][r]
        if h == 0:  # a fresh prompt attends in the original domain
            for g in range(hk):
                out[a:b, g * group:(g + 1) * group] = _attend(q[a:b, g * group:(g + 1) * group], k[a:b, g].contiguous(),
                                                              v[a:b, g].contiguous(), 0, d ** -0.5)
            continue
        pos = np.arange(h)
        block = x["host_table"][r, pos // BLOCK].astype(np.int64)
        slot = torch.from_numpy(block * BLOCK + pos % BLOCK).to(owner.device)
        place = torch.from_numpy(block % rows * BLOCK + pos % BLOCK).to(owner.device)
        mine = (owner[place] == slot // BLOCK)[:, None, None]
        # a history value is a 16-bit number by contract: dtype(fp16(x))
        keys, values = (torch.where(mine, arena[place], y).half().to(dtype).double()
                        for arena, y in zip(seen, _read(x["k_cache"], x["v_cache"], d, slot)))
        q_rot = q[a:b] @ rk
        for g in range(hk):
            heads = slice(g * group, (g + 1) * group)
            o = _attend(q_rot[:, heads], torch.cat([keys[:, g], k_rot[a:b, g]]), torch.cat([values[:, g], v_rot[a:b, g]]),
                        h, d ** -0.5)
            out[a:b, heads] = o @ rv.t().contiguous()
    stage_k.view(-1, hk, d)[seat] = k_rot[token]
    stage_v.view(-1, hk, d)[seat] = v_rot[token]
    return dict(out=out.view(out.shape[0], -1), k_cache=None, v_cache=None, owner=None, stage_k=stage_k, stage_v=stage_v)
