"""The work that programs have this framework do, as measurable cases.

Every case is one pass of a serving program through the public operators
(`torch.ops.gaudirt.paged_attn`, `rotary_paged_attn`, `_advance_decode_lengths`,
`PagedMetadata`): the new K/V rows of a batch are stored into a paged bf16 pool
and every row attends its request's visible keys. Two forms:

- "op": one attention layer. The batch's PagedMetadata is made beforehand, as a
  program makes it once and uses it in every layer.
- "step": a whole scheduler step: lengths advanced (when every sequence
  decodes), device metadata built from the scheduler's tensors, then the fused
  rotary + store + attention of each layer. The request map is token-granular.

Sequence lengths are part of the case (drawn from its "lengths" number);
values, pool placement and slot order are made from the seed. `seqs` sequences
prefill a chunk of rows_lo .. rows_hi new tokens on a cached prefix of
prefix_lo .. prefix_hi tokens, `decode` sequences decode one token with
ctx_lo .. ctx_hi visible keys. With `shared` the prefix is one set of blocks.
"""

import math
import random

import numpy as np
import torch

import gaudirt_amd

MAX_ROWS = 8192        # rows of one PagedMetadata
ROPE_THETA = 10000.0
GEOMETRIES = [         # (query heads, kv heads, head_dim) of the configurations and tests
    (32, 8, 128), (32, 8, 128), (64, 8, 128), (8, 2, 128), (14, 2, 64), (16, 8, 256), (8, 8, 128), (24, 8, 128),
    (56, 8, 128), (16, 8, 128), (32, 8, 64),
]


def _case(name=None, **fields):
    case = {
        "form": "op", "seqs": 0, "rows_lo": 0, "rows_hi": 0, "prefix_lo": 0, "prefix_hi": 0, "shared": False,
        "decode": 0, "ctx_lo": 0, "ctx_hi": 0, "spread": "uniform", "q_heads": 32, "kv_heads": 8, "head_dim": 128,
        "page": 128, "softcap": 0.0, "window": -1, "layers": 1, "lengths": 1,
    }
    assert set(fields) <= set(case), set(fields) - set(case)
    case.update(fields)
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # The smallest batch: four short conversations on a small model. Launches and host work are what counts.
        _case("decode_smallest", decode=4, ctx_lo=1, ctx_hi=512, q_heads=8, kv_heads=2),
        # One user with a long conversation: a single decode row, pages of 16 tokens.
        _case("decode_single_long", decode=1, ctx_lo=15001, ctx_hi=15001, page=16),
        # A server's ordinary decode batch at the benchmark's default size.
        _case("decode_batch", decode=64, ctx_lo=512, ctx_hi=4096),
        # Long, very unequal contexts, eight query heads on each kv head.
        _case("decode_long_skewed", decode=32, ctx_lo=1024, ctx_hi=32768, spread="log", q_heads=64),
        # Wide heads with logit softcap and a sliding window, pages of 16 tokens.
        _case("decode_d256_window", decode=48, ctx_lo=128, ctx_hi=8000, q_heads=16, head_dim=256, page=16,
              softcap=50.0, window=4096),
        # A whole decode step of a full server on the scheduler's token-granular map: metadata and four layers.
        _case("step_decode", form="step", decode=256, ctx_lo=128, ctx_hi=2049, page=1, layers=4),
        # Eight requests that share a system prompt, each prefilling a 512-token chunk.
        _case("prefill_shared", seqs=8, rows_lo=512, rows_hi=512, prefix_lo=2048, prefix_hi=2048, shared=True),
        # One ragged chunk of a small model on a token-granular map: few query rows, a long prefix.
        _case("prefill_chunk_d64", seqs=1, rows_lo=263, rows_hi=263, prefix_lo=3840, prefix_hi=3840, q_heads=14,
              kv_heads=2, head_dim=64, page=1),
        # One request's next chunk deep inside a long prompt.
        _case("prefill_chunk_deep", seqs=1, rows_lo=512, rows_hi=512, prefix_lo=15000, prefix_hi=15000, page=16),
        # The largest chunk: the last 4096 tokens of a 32768-token prompt.
        _case("prefill_largest", seqs=1, rows_lo=4096, rows_hi=4096, prefix_lo=28672, prefix_hi=28672, q_heads=56),
        # Continuous batching: a scheduler step with decode rows beside two prompts' chunks, four layers.
        _case("step_mixed", form="step", seqs=2, rows_lo=137, rows_hi=400, prefix_lo=0, prefix_hi=3000, decode=48,
              ctx_lo=300, ctx_hi=4000, page=16, layers=4),
        # Ragged new prompts with wide heads, softcap and window.
        _case("prefill_d256_window", seqs=4, rows_lo=300, rows_hi=2000, q_heads=16, head_dim=256, page=16,
              softcap=50.0, window=4096),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    largest = max(work(c)["flops"] for c in listed())
    most_bytes = max(work(c)["bytes"] for c in listed())
    while True:
        q_heads, kv_heads, head_dim = rng.choice(GEOMETRIES)
        kind = rng.choice(["decode", "decode", "prefill", "prefill", "mixed", "step"])
        f = {"q_heads": q_heads, "kv_heads": kv_heads, "head_dim": head_dim, "page": rng.choice([1, 16, 16, 128]),
             "lengths": rng.randrange(1 << 20)}
        if rng.random() < 0.25:
            f["softcap"] = rng.choice([30.0, 50.0])
        if rng.random() < 0.25:
            f["window"] = rng.choice([128, 1024, 4096, 1000])
        if kind in ("decode", "mixed", "step"):
            f["decode"] = _log(rng, 1, 256)
            f["ctx_hi"] = _log(rng, 16, 32768)
            f["ctx_lo"] = max(1, int(f["ctx_hi"] * rng.choice([0.05, 0.25, 0.9])))
            f["spread"] = rng.choice(["uniform", "log"])
        if kind in ("prefill", "mixed") or (kind == "step" and rng.random() < 0.5):
            f["seqs"] = _log(rng, 1, 8)
            f["rows_hi"] = _log(rng, 16, 4096)
            f["rows_lo"] = max(1, int(f["rows_hi"] * rng.choice([0.2, 0.6, 1.0])))
            f["prefix_hi"] = rng.choice([0, _log(rng, 16, 28672), _log(rng, 16, 28672)])
            f["prefix_lo"] = int(f["prefix_hi"] * rng.choice([0.2, 0.7, 1.0]))
        if kind == "step":
            f.update(form="step", layers=rng.choice([1, 2, 4]), softcap=0.0, window=-1)
        case = _case(**f)
        if case["seqs"] * case["rows_hi"] + case["decode"] > MAX_ROWS:
            continue
        w = work(case)
        if w["flops"] <= largest and w["bytes"] <= most_bytes:
            return case


def _sequences(case):
    """(prefix, new tokens) of every sequence: the decoding ones first."""
    rng = random.Random(case["lengths"])

    def pick(lo, hi):
        if lo >= hi:
            return hi
        return min(hi, max(lo, _log(rng, lo, hi))) if case["spread"] == "log" else rng.randint(lo, hi)

    decode = [(pick(case["ctx_lo"], case["ctx_hi"]) - 1, 1) for _ in range(case["decode"])]
    chunks = []
    for _ in range(case["seqs"]):
        rows = rng.randint(case["rows_lo"], case["rows_hi"])
        chunks.append((rng.randint(case["prefix_lo"], case["prefix_hi"]), rows))
    return decode + chunks


def work(case):
    seqs = _sequences(case)
    window = case["window"] if case["window"] > 0 else 1 << 30
    rows = sum(n for _, n in seqs)
    keys = pairs = 0
    for i, (prefix, n) in enumerate(seqs):
        first = max(0, prefix + 1 - window)  # the first key that any row of the sequence sees
        shared = case["shared"] and i > case["decode"]
        keys += (prefix + n - first) - (prefix - first if shared else 0)
        full = max(0, min(n, prefix + n - window + 1))  # rows that see a whole window
        ramp = n - full
        pairs += ramp * (prefix + 1) + ramp * (ramp - 1) // 2 + full * window if full < n or prefix + 1 < window \
            else n * window
    q_width, kv_width = case["q_heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    # Keys and values once, queries and outputs once, the new rows read and written once, one table entry a page.
    per_layer = keys * kv_width * 4 + rows * q_width * 4 + rows * kv_width * 8 + 4 * (keys // case["page"] + 2 * rows)
    return {"bytes": case["layers"] * per_layer, "flops": case["layers"] * 4 * q_width * pairs}


def _rope_cache(positions, head_dim, device):
    half = head_dim // 2
    inverse = ROPE_THETA ** (-torch.arange(half, dtype=torch.float64, device=device) / half)
    angles = torch.arange(positions, dtype=torch.float64, device=device)[:, None] * inverse
    return torch.cat([angles.cos(), angles.sin()], dim=1).to(torch.bfloat16)


def _place(case, seed):
    """(token map [sequences, context] int32, slots): every sequence's tokens in blocks scattered over the pool."""
    seqs, page = _sequences(case), case["page"]
    rng = np.random.default_rng(seed)
    shared_pages = min((p for p, _ in seqs), default=0) // page if case["shared"] else 0
    own = [-(-(p + n) // page) - shared_pages for p, n in seqs]
    blocks = rng.permutation(shared_pages + sum(own) + 1).astype(np.int64)
    context = max(p + n for p, n in seqs)
    mapping = np.full((len(seqs), context), -1, dtype=np.int32)
    at = shared_pages
    for s, (prefix, n) in enumerate(seqs):
        table = np.concatenate([blocks[:shared_pages], blocks[at:at + own[s]]])
        at += own[s]
        tokens = np.arange(prefix + n)
        mapping[s, :prefix + n] = table[tokens // page] * page + tokens % page
    return mapping, len(blocks) * page


def prepare(case, seed):
    gaudirt_amd.load_extension()
    seqs = _sequences(case)
    layers, d = case["layers"], case["head_dim"]
    q_heads, kv_heads = case["q_heads"], case["kv_heads"]
    mapping, slots = _place(case, seed)
    requests = np.repeat(np.arange(len(seqs)), [n for _, n in seqs])
    positions = np.concatenate([np.arange(p, p + n) for p, n in seqs])
    locations = mapping[requests, positions].astype(np.int64)
    rows = len(positions)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def normal(*shape):
        return torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(generator=gen)

    pool = gaudirt_amd.allocate_paged_kv(layers, slots, kv_heads, d)
    pool.normal_(generator=gen)
    state = {
        "case": case, "pool": pool, "views": [gaudirt_amd.kv_pool_views(pool, i) for i in range(layers)],
        "query": [normal(rows, q_heads * d) for _ in range(layers)],
        "key": [normal(rows, kv_heads * d) for _ in range(layers)],
        "value": [normal(rows, kv_heads * d) for _ in range(layers)],
        "scale": float(np.float32(1 / math.sqrt(d))), "slots": slots,
        "where": (mapping, requests, positions, locations),
    }
    if case["form"] == "op":
        state["metadata"] = torch.classes.gaudirt.PagedMetadata(
            torch.from_numpy(locations), torch.from_numpy(requests), torch.from_numpy(positions),
            torch.from_numpy(mapping), slots)
    else:
        state["locations"] = torch.from_numpy(locations).cuda()
        state["requests"] = torch.arange(len(seqs), dtype=torch.int64, device="cuda")
        state["positions"] = torch.from_numpy(positions)
        state["mapping"] = torch.from_numpy(mapping).cuda()
        state["prefixes"] = [p for p, _ in seqs]
        state["lengths"] = [n for _, n in seqs]
        state["seq_lens"] = torch.tensor([p for p, _ in seqs], dtype=torch.int64, device="cuda")
        state["orig_lens"] = state["seq_lens"].to(torch.int32)
        state["cache"] = _rope_cache(mapping.shape[1], d, "cuda")
    return state


def run(state):
    case = state["case"]
    d, scale, softcap, window = case["head_dim"], state["scale"], case["softcap"], case["window"]
    if case["form"] == "op":
        key_pool, value_pool = state["views"][0]
        out = torch.ops.gaudirt.paged_attn(state["query"][0], state["key"][0], state["value"][0], key_pool, value_pool,
                                           state["metadata"], d, scale, softcap, window)
        return {"out": [out], "pool": state["pool"]}
    result = {}
    if not case["seqs"]:
        result["lens"] = list(torch.ops.gaudirt._advance_decode_lengths(state["seq_lens"], state["orig_lens"]))
    metadata = torch.classes.gaudirt.PagedMetadata._from_scheduler_fused(
        state["locations"], state["requests"], state["positions"], state["mapping"], state["prefixes"],
        state["lengths"], state["slots"], None, 0, case["q_heads"], case["kv_heads"], d)
    result["out"] = [
        torch.ops.gaudirt.rotary_paged_attn(state["query"][i], state["key"][i], state["value"][i], *state["views"][i],
                                            state["cache"], metadata, d, d, True, scale, softcap, window)
        for i in range(case["layers"])]
    result["pool"] = state["pool"]
    return result


def _rotate(x, cache, positions, d):
    """NeoX rotation of [rows, heads * d] in 64 bits."""
    x = x.double().view(x.shape[0], -1, 2, d // 2)
    cos, sin = cache.double()[positions].view(x.shape[0], 1, 2, d // 2).unbind(2)
    a, b = x.unbind(2)
    return torch.stack([a * cos - b * sin, b * cos + a * sin], dim=2).reshape(x.shape[0], -1)


def exact(case, seed):
    state = prepare(case, seed)
    seqs, d, kv_heads = _sequences(case), case["head_dim"], case["kv_heads"]
    group = case["q_heads"] // kv_heads
    mapping, _, positions, locations = state["where"]
    mapping = torch.from_numpy(mapping).cuda()
    positions, locations = torch.from_numpy(positions).cuda(), torch.from_numpy(locations).cuda()
    outs = []
    for layer in range(case["layers"]):
        query, key = state["query"][layer].double(), state["key"][layer]
        if case["form"] == "step":
            query = _rotate(state["query"][layer], state["cache"], positions, d)
            key = _rotate(key, state["cache"], positions, d).to(torch.bfloat16)  # the pool holds bf16
        keys, values = state["pool"][layer, 0], state["pool"][layer, 1]
        keys[:, locations] = key.view(-1, kv_heads, d).transpose(0, 1)
        values[:, locations] = state["value"][layer].view(-1, kv_heads, d).transpose(0, 1)
        out = torch.empty(query.shape, dtype=torch.float64, device="cuda")
        first = 0
        for s, (prefix, n) in enumerate(seqs):
            slots = mapping[s, :prefix + n].long()
            at = torch.arange(prefix + n, device="cuda")
            for h in range(kv_heads):
                k = keys[h, slots].double().t().contiguous()
                v = values[h, slots].double()
                for r in range(0, n, 1024):
                    m = min(1024, n - r)
                    rows = slice(first + r, first + r + m)
                    q = query[rows].view(m, -1, d)[:, h * group:(h + 1) * group].reshape(m * group, d)
                    score = q @ k * state["scale"]
                    if case["softcap"] > 0:
                        score = case["softcap"] * torch.tanh(score / case["softcap"])
                    p = positions[rows].repeat_interleave(group)[:, None]
                    hidden = at > p
                    if case["window"] > 0:
                        hidden |= at <= p - case["window"]
                    weight = torch.softmax(score.masked_fill_(hidden, -math.inf), dim=1)
                    out[rows].view(m, -1, d)[:, h * group:(h + 1) * group] = (weight @ v).view(m, group, d)
            first += n
        outs.append(out)
    result = {"out": outs, "pool": None}
    if case["form"] == "step" and not case["seqs"]:
        result["lens"] = [None, None]
    return result


def tolerance(case):
    # Outputs are bf16 (rounding them alone gives 1.7e-3) and probabilities are
    # rounded to bf16 before they meet V: 2.0e-3 .. 2.4e-3 from exact(), one
    # value up to 0.029. Steps round the rotated queries to bf16 as well:
    # 2.8e-3, up to 0.030. About four times those.
    return {"rel": 1.2e-2 if case["form"] == "step" else 9.5e-3, "max": 0.12}
