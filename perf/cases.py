"""Measured work of the paged-KV operators: what one layer of a serving step asks of them.

A case is a dict of plain values; ``prepare`` turns it into device tensors, ``run`` takes them once through
``infinicore_amd.ops`` with the arguments a serving loop passes (outputs allocated by the operator, default stream).

Families (``case["op"]``):

* ``decode``          - one query token per sequence over the paged pool (``paged_attention``)
* ``decode_step``     - the same with its producer in front: the new token's query and key rotated and K / V scattered
                        (``rope_paged_caching`` with the query), then ``paged_attention``
* ``prefill``         - runs of new tokens over their history (``paged_attention_prefill``)
* ``prefill_step``    - the same with its producer in front
* ``write``           - cache writes alone: ``rope_qk`` (rotate query and key, scatter K / V), ``rope`` (key only),
                        ``paged`` (plain scatter), ``append`` (contiguous caches)

The lengths of a batch are fixed by the case (a stratified draw between its bounds), so that the work of a pass is; the
seed decides which sequence has which length, where its pages lie, and every value.
"""
from __future__ import annotations

import math
import random

import torch

from infinicore_amd import ops

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
_INDEX = {"i64": torch.int64, "i32": torch.int32}
_ROPE_TABLE_LEN = 32768
_SPARE_PAGES = 0.10  # of the pool, as a server keeps them free


def _case(name, op, **more):
    c = dict(name=name, op=op, dtype="bf16", index="i64", page=16, alibi=False)
    c.update(more)
    return c


def listed():
    return [
        # a single user's chat: one sequence, the whole attention part of a layer; launches and latency are all there is
        _case("decode_step_one", "decode_step", seqs=1, heads=32, kv_heads=8, head=128, value=128, min_len=1023, max_len=1023),
        # the ordinary serving batch: 8B-class GQA decode, ragged lengths (the repository's headline shape)
        _case("decode_gqa_b32", "decode", seqs=32, heads=32, kv_heads=8, head=128, value=128, min_len=512, max_len=4096),
        # few long documents: the chip is filled by cutting sequences, the softmax is peaked
        _case("decode_long_b8", "decode", seqs=8, heads=32, kv_heads=8, head=128, value=128, min_len=16384, max_len=32768,
              peaked=0.01),
        # the largest decode call: a 70B-class share of a big batch, fp16
        _case("decode_share_b128", "decode", dtype="fp16", seqs=128, heads=64, kv_heads=8, head=128, value=128, min_len=1024,
              max_len=8192),
        # an older multi-head model: no grouping, heads of 64, ALiBi, 32-bit tables, pages of 32, short odd lengths
        _case("decode_mha64_alibi_b19", "decode", dtype="fp16", index="i32", page=32, alibi=True, seqs=19, heads=16,
              kv_heads=16, head=64, value=64, min_len=37, max_len=1531),
        # latent-attention cache, a tensor-parallel share of the heads / all heads on one GPU
        _case("decode_latent16_b32", "decode", seqs=32, heads=16, kv_heads=1, head=576, value=512, min_len=512, max_len=4096),
        _case("decode_latent128_b32", "decode", seqs=32, heads=128, kv_heads=1, head=576, value=512, min_len=512,
              max_len=4096),
        # short prompts of a chat service with the producer in front: a prefill call too small to fill the chip
        _case("prefill_step_short_b4", "prefill_step", seqs=4, heads=32, kv_heads=8, head=128, value=128, min_new=19,
              max_new=250, min_hist=0, max_hist=0),
        # whole prompts, and chunks over a long history (chunked prefill)
        _case("prefill_prompts_b4", "prefill", seqs=4, heads=32, kv_heads=8, head=128, value=128, min_new=1024, max_new=3072,
              min_hist=0, max_hist=0),
        _case("prefill_chunked_b16", "prefill", seqs=16, heads=32, kv_heads=8, head=128, value=128, min_new=128, max_new=512,
              min_hist=1024, max_hist=8192),
        _case("prefill_latent16_b16", "prefill", seqs=16, heads=16, kv_heads=1, head=576, value=512, min_new=128, max_new=512,
              min_hist=1024, max_hist=8192),
        # the cache writes of a prefill chunk, some of its tokens padding
        _case("write_rope_qk_4096", "write", kind="rope_qk", tokens=4096, heads=32, kv_heads=8, head=128, value=128,
              padding=0.05),
    ]


# ---- drawn cases: the same families over their whole ranges ----

_LAYOUTS = [(32, 8), (32, 8), (64, 8), (8, 8), (40, 8), (16, 16), (48, 8), (28, 4), (8, 1)]  # query / KV heads


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _span(rng, lo, hi):
    """A lower and an upper bound inside [lo, hi], at most a factor of eight apart."""
    top = _log_int(rng, lo, hi)
    return max(lo, int(top * rng.uniform(0.125, 1.0))), top


def _options(rng):
    return dict(dtype=rng.choice(["bf16", "bf16", "fp16"]), index=rng.choice(["i64", "i64", "i32"]),
                page=rng.choice([16, 16, 16, 32, 64, 128]))


def _draw_decode(rng):
    c = _options(rng)
    c["op"] = rng.choice(["decode", "decode", "decode_step"])
    c["heads"], c["kv_heads"] = rng.choice(_LAYOUTS)
    c["head"] = c["value"] = rng.choice([64, 128, 128, 128, 192, 256])
    c["alibi"] = rng.random() < 0.15
    c["seqs"] = _log_int(rng, 1, 256)
    c["min_len"], c["max_len"] = _span(rng, 16, 32768)
    return c


def _draw_latent_decode(rng):
    c = _options(rng)
    c.update(op="decode", heads=rng.choice([8, 16, 16, 32, 64, 128, 128]), kv_heads=1, head=576, value=512, alibi=False)
    c["seqs"] = _log_int(rng, 1, 128)
    c["min_len"], c["max_len"] = _span(rng, 16, 16384)
    return c


def _draw_prefill(rng):
    c = _options(rng)
    if rng.random() < 0.25:
        c.update(op="prefill", heads=16, kv_heads=1, head=576, value=512, alibi=False)
    else:
        c["op"] = rng.choice(["prefill", "prefill", "prefill_step"])
        c["heads"], c["kv_heads"] = rng.choice(_LAYOUTS)
        c["head"] = c["value"] = rng.choice([64, 128, 128, 128, 192, 256])
        c["alibi"] = rng.random() < 0.15
    c["seqs"] = _log_int(rng, 1, 32)
    c["min_new"], c["max_new"] = _span(rng, 1, 4096)
    c["min_hist"], c["max_hist"] = (0, 0) if rng.random() < 0.4 else _span(rng, 16, 8192)
    return c


def _draw_write(rng):
    c = _options(rng)
    c.update(op="write", kind=rng.choice(["rope_qk", "rope_qk", "rope", "paged", "append"]), alibi=False,
             padding=rng.choice([0.0, 0.05]))
    c["heads"], c["kv_heads"] = rng.choice(_LAYOUTS)
    c["head"] = c["value"] = rng.choice([64, 128, 128, 128, 192, 256])
    c["tokens"] = _log_int(rng, 1, 6000)
    if c["kind"] == "append":
        c["seqs"] = _log_int(rng, 1, 32)
        c["tokens"] = max(1, c["tokens"] // c["seqs"])
    return c


def draw(rng: random.Random):
    while True:
        pick = rng.random()
        if pick < 0.4:
            c = _draw_decode(rng)
        elif pick < 0.55:
            c = _draw_latent_decode(rng)
        elif pick < 0.85:
            c = _draw_prefill(rng)
        else:
            c = _draw_write(rng)
        w = work(c)
        latent = c["head"] == 576
        # no more than the largest listed cases: bytes of the decode share, flops of the prefill calls
        if w["bytes"] <= 2.4e9 and w["flops"] <= (8e11 if latent else 4e11) and (latent or w["bytes"] + w["flops"] / 100 <= 4e9):
            return c


# ---- lengths and work: functions of the case alone ----

def _stratified(count, lo, hi, salt):
    """``count`` lengths spread over [lo, hi]: one from each of as many equal parts, in no particular order."""
    rng = random.Random("%d %d %d %d" % (count, lo, hi, salt))
    got = [lo + int((i + rng.random()) / count * (hi - lo + 1)) for i in range(count)]
    rng.shuffle(got)
    return got


def _lengths(case):
    """(new tokens, tokens seen at the end of the pass) of every sequence."""
    if case["op"].startswith("decode"):
        return [1] * case["seqs"], _stratified(case["seqs"], case["min_len"], case["max_len"], 1)
    new = _stratified(case["seqs"], case["min_new"], case["max_new"], 2)
    hist = _stratified(case["seqs"], case["min_hist"], case["max_hist"], 3)
    return new, [n + h for n, h in zip(new, hist)]


def _padding_tokens(case):
    return int(case["tokens"] * case["padding"])


def _write_bytes(case, tokens, valid, with_query, index_bytes=8):
    """Reads of the new vectors, positions, slots and tables, writes of the cache rows and the rotated query."""
    kv = case["kv_heads"] * (case["head"] + case["value"]) * 2
    b = valid * kv * 2 + tokens * index_bytes
    if with_query is not None:
        b += tokens * (8 + 2 * case["head"])  # one position, one row of each table
        b += 2 * tokens * with_query * case["head"] * 2
    return b


def work(case):
    head, value, heads, kv = case["head"], case["value"], case["heads"], case["kv_heads"]
    if case["op"] == "write":
        kind = case["kind"]
        if kind == "append":
            tokens = case["tokens"] * case["seqs"]
            return {"bytes": _write_bytes(case, tokens, tokens, None, 0) + 8 * case["seqs"], "flops": 0}
        tokens, valid = case["tokens"], case["tokens"] - _padding_tokens(case)
        query = {"rope_qk": heads, "rope": 0, "paged": None}[kind]
        return {"bytes": _write_bytes(case, tokens, valid, query),
                "flops": 0 if query is None else 3 * tokens * (query + kv) * head}
    new, total = _lengths(case)
    item = 8 if case["index"] == "i64" else 4
    pages = sum(-(-t // case["page"]) for t in total)
    tokens = sum(new)
    pairs = sum(n * (t - n) + n * (n + 1) // 2 for n, t in zip(new, total))
    b = sum(total) * kv * (head + value) * 2 + tokens * heads * (head + value) * 2 + (pages + 2 * len(new)) * item
    flops = pairs * heads * 2 * (head + value)
    if case["op"].endswith("_step"):
        b += _write_bytes(case, tokens, tokens, heads)
        flops += 3 * tokens * (heads + kv) * head
    return {"bytes": b, "flops": flops}


def tolerance(case):
    if case["op"] == "write":
        return "exact"  # moved bytes, and a rotation whose every rounding is prescribed
    # Attention outputs are rounded once to the storage type, after fp32 sums over probabilities that a matrix unit may
    # take rounded to it as well. Against float64 (listed and drawn cases): bf16 at most 2.3e-3 and 1.2e-2, fp16 at most
    # 2.9e-4 and 1.2e-3; about four times that.
    return {"rel": 1e-2, "max": 0.05} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 5e-3}


# ---- inputs ----

def _rope_tables(head, dtype, device):
    freqs = 1.0 / (10000.0 ** (torch.arange(0, head, 2, device=device).float() / head))
    angles = torch.outer(torch.arange(_ROPE_TABLE_LEN, device=device).float(), freqs)
    return torch.sin(angles).to(dtype), torch.cos(angles).to(dtype)


def _prepare_write(case, gen, dev):
    dtype, kv, head, value = _DTYPES[case["dtype"]], case["kv_heads"], case["head"], case["value"]

    def normal(*shape):
        return torch.randn(shape, dtype=dtype, device=dev, generator=gen)

    state = {"case": case}
    if case["kind"] == "append":
        seqs, n = case["seqs"], case["tokens"]
        room = 2 * n + 64
        state.update(k_cache=normal(seqs, kv, room, head), v_cache=normal(seqs, kv, room, value),
                     k=normal(seqs, kv, n, head), v=normal(seqs, kv, n, value),
                     past=torch.randint(0, room - n + 1, (seqs,), device=dev, generator=gen))
        return state
    n, page = case["tokens"], case["page"]
    blocks = -(-4 * n // page) + 8
    slots = torch.randperm(blocks * page, device=dev, generator=gen)[:n]
    slots[torch.randperm(n, device=dev, generator=gen)[:_padding_tokens(case)]] = -1
    state.update(k_cache=normal(blocks, kv, page, head), v_cache=normal(blocks, kv, page, value), k=normal(n, kv, head),
                 v=normal(n, kv, value), slots=slots)
    if case["kind"] != "paged":
        state["pos"] = torch.randint(0, _ROPE_TABLE_LEN, (n,), device=dev, generator=gen)
        state["sin"], state["cos"] = _rope_tables(head, dtype, dev)
    if case["kind"] == "rope_qk":
        state["q"] = normal(n, case["heads"], head)
        state["q_out"] = torch.empty_like(state["q"])
    return state


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(seed))
    if case["op"] == "write":
        return _prepare_write(case, gen, dev)
    dtype, index = _DTYPES[case["dtype"]], _INDEX[case["index"]]
    heads, kv, head, value, page = case["heads"], case["kv_heads"], case["head"], case["value"], case["page"]

    def normal(*shape):
        return torch.randn(shape, dtype=dtype, device=dev, generator=gen)

    new, total = _lengths(case)
    order = random.Random(int(seed)).sample(range(len(new)), len(new))
    new, total = [new[i] for i in order], [total[i] for i in order]
    needed = [-(-t // page) for t in total]
    blocks = int(math.ceil(sum(needed) * (1.0 + _SPARE_PAGES)))
    pages = torch.randperm(blocks, generator=torch.Generator().manual_seed(int(seed)))
    table = torch.zeros((len(new), max(needed)), dtype=index)
    at = 0
    for s, count in enumerate(needed):
        table[s, :count] = pages[at:at + count].to(index)
        at += count

    k_cache = normal(blocks, kv, page, head)
    if case.get("peaked"):
        hot = torch.rand((blocks, 1, page, 1), device=dev, generator=gen) < case["peaked"]
        k_cache = torch.where(hot, k_cache * 8, k_cache)
    state = {"case": case, "scale": 1.0 / math.sqrt(head), "k_cache": k_cache, "v_cache": normal(blocks, kv, page, value),
             "q": normal(sum(new), heads, head), "table": table.to(dev), "lens": torch.tensor(total, dtype=index, device=dev),
             "alibi": None}
    if case["alibi"]:
        state["alibi"] = torch.tensor([2.0 ** (-8.0 * (h + 1) / heads) for h in range(heads)], device=dev)
    if case["op"].startswith("prefill"):
        cum = [0]
        for n in new:
            cum.append(cum[-1] + n)
        state["cum"] = torch.tensor(cum, dtype=index, device=dev)
    if case["op"].endswith("_step"):
        pos = torch.cat([torch.arange(t - n, t) for n, t in zip(new, total)])
        seq = torch.repeat_interleave(torch.arange(len(new)), torch.tensor(new))
        slots = table[seq, pos // page].to(torch.int64) * page + pos % page
        state.update(pos=pos.to(dev), slots=slots.to(dev), k=normal(len(pos), kv, head), v=normal(len(pos), kv, value),
                     q_rot=torch.empty_like(state["q"]))
        state["sin"], state["cos"] = _rope_tables(head, dtype, dev)
    return state


def run(state):
    s, case = state, state["case"]
    op = case["op"]
    if op == "write":
        if case["kind"] == "append":
            return ops.kv_caching(s["k_cache"], s["v_cache"], s["k"], s["v"], s["past"])
        if case["kind"] == "paged":
            return ops.paged_caching(s["k_cache"], s["v_cache"], s["k"], s["v"], s["slots"])
        if case["kind"] == "rope":
            return ops.rope_paged_caching(s["k_cache"], s["v_cache"], s["k"], s["v"], s["slots"], s["pos"], s["sin"], s["cos"])
        return ops.rope_paged_caching(s["k_cache"], s["v_cache"], s["k"], s["v"], s["slots"], s["pos"], s["sin"], s["cos"],
                                      q=s["q"], q_out=s["q_out"])
    q, written = s["q"], ()
    if op.endswith("_step"):
        written = ops.rope_paged_caching(s["k_cache"], s["v_cache"], s["k"], s["v"], s["slots"], s["pos"], s["sin"], s["cos"],
                                         q=q, q_out=s["q_rot"])
        q = s["q_rot"]
    if op.startswith("decode"):
        out = ops.paged_attention(q, s["k_cache"], s["v_cache"], s["table"], s["lens"], s["alibi"], s["scale"])
    else:
        out = ops.paged_attention_prefill(q, s["k_cache"], s["v_cache"], s["table"], s["lens"], s["cum"], s["alibi"], s["scale"])
    return (out, *written)


# ---- the same in 64 bits ----

def _rotated(x, pos, sin, cos):
    """GPT-NeoX rotation of x [tokens, heads, head] in 64 bits."""
    half = x.shape[-1] // 2
    sin, cos = sin[pos].double()[:, None, :], cos[pos].double()[:, None, :]
    lo, hi = x[..., :half].double(), x[..., half:].double()
    return torch.cat((lo * cos - hi * sin, lo * sin + hi * cos), dim=-1)


def exact(case, seed):
    if case["op"] == "write":
        return None  # moved bytes, and a rotation whose roundings are prescribed: compared bit by bit
    s = prepare(case, seed)
    q, k_cache, v_cache = s["q"], s["k_cache"], s["v_cache"]
    more = ()
    if case["op"].endswith("_step"):
        # the rotated vectors go through the storage type: that is what the caches and the rotated query hold
        q_rot = _rotated(q, s["pos"], s["sin"], s["cos"])
        k_rot = _rotated(s["k"], s["pos"], s["sin"], s["cos"]).to(k_cache.dtype)
        page, row = s["slots"] // case["page"], s["slots"] % case["page"]
        k_cache[page, :, row], v_cache[page, :, row] = k_rot, s["v"]
        q = q_rot.to(q.dtype)
        more = (None, None, q_rot)
    new, _ = _lengths(case)
    lens = s["lens"].tolist()
    cum = s["cum"].tolist() if "cum" in s else list(range(len(new) + 1))
    kv, group = case["kv_heads"], case["heads"] // case["kv_heads"]
    out = torch.empty((*q.shape[:-1], case["value"]), dtype=torch.float64, device=q.device)
    for i, total in enumerate(lens):
        pages = s["table"][i, :-(-total // case["page"])].long()
        n = cum[i + 1] - cum[i]
        last = torch.arange(total - n, total, device=q.device)  # the last token that each new token sees
        away = torch.arange(total, device=q.device)[None, :] - last[:, None]
        for g in range(kv):
            k = k_cache[pages, g].reshape(-1, case["head"])[:total].double()
            v = v_cache[pages, g].reshape(-1, case["value"])[:total].double()
            for h in range(g * group, (g + 1) * group):
                scores = (q[cum[i]:cum[i + 1], h].double() @ k.T) * s["scale"]
                if s["alibi"] is not None:
                    scores = scores + s["alibi"][h].double() * away
                scores.masked_fill_(away > 0, -math.inf)
                out[cum[i]:cum[i + 1], h] = torch.softmax(scores, dim=-1) @ v
    return (out, *more)
