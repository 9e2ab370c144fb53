"""The work that this library is timed on: attention forwards through the
public ``Runner`` entry points, over the sizes that its users run.

Every case is one call of one entry point:

* ``forward``  dense or top-left causal attention of a batch of equal-length
  sequences (``Runner.call``, ``call_gqa`` with fewer K/V heads than query
  heads, ``call_strided`` for BHSD views): training forwards and whole-prompt
  prefill, with the log-sum-exp output where a backward pass would need it;
* ``splitkv``  the same with the key range split over the GPU
  (``Runner.call_splitkv``): long keys under few queries, and decode;
* ``varlen``   packed sequences of unequal lengths (``Runner.call_varlen``);
* ``paged``    new queries against paged K/V caches
  (``Runner.call_splitkv_paged``): the decode and chunked-prefill steps of a
  serving engine.

The paths are attention forwards in BF16 at head dimension 128; there is no
other data type and no backward.  ``draw`` gives more cases of these ranges.
"""
from __future__ import annotations

import math
import random

import torch

import __graft_entry__

D = 128
SCALE = 1.0 / math.sqrt(D)
DEVICE = "cuda"
BOTTOM_RIGHT = 2          # Runner's mask code: query i of sq sees keys j <= sk - sq + i


def listed():
    return [
        # The smallest calls: a short prompt of a small model; launch and fill
        # time count, and no size is a multiple of a tile.
        dict(name="forward_tiny", op="forward", batch=3, heads=8, kv_heads=8, sq=193, sk=257, mask=0, lse=True,
             layout="bshd"),
        # The benchmark's sequence sweep, short end: a training forward at 512.
        dict(name="forward_causal_512", op="forward", batch=32, heads=8, kv_heads=8, sq=512, sk=512, mask=1,
             lse=False, layout="bshd"),
        # The ragged validation shape: cross attention of 1000 queries over
        # 3077 keys, keeping the LSE for a backward pass.
        dict(name="forward_ragged_lse", op="forward", batch=4, heads=16, kv_heads=16, sq=1000, sk=3077, mask=0,
             lse=True, layout="bshd"),
        # The benchmark's headline, dense and causal.
        dict(name="forward_dense_4096", op="forward", batch=32, heads=8, kv_heads=8, sq=4096, sk=4096, mask=0,
             lse=False, layout="bshd"),
        dict(name="forward_causal_4096", op="forward", batch=32, heads=8, kv_heads=8, sq=4096, sk=4096, mask=1,
             lse=False, layout="bshd"),
        # A long-context training forward with grouped K/V heads, from the
        # BHSD tensors that torch's own attention takes, LSE kept.
        dict(name="forward_gqa_8192", op="forward", batch=1, heads=32, kv_heads=8, sq=8192, sk=8192, mask=1,
             lse=True, layout="bhsd"),
        # A packed batch of prompts of mixed lengths (prefill or packed training).
        dict(name="varlen_prefill", op="varlen", seqs=24, heads=32, kv_heads=8, min_len=64, max_len=4096, mask=1,
             lse=False, lens_seed=1),
        # A prompt chunk against a long context on a small grid: the key range
        # has to be split to fill the GPU.
        dict(name="splitkv_prefill", op="splitkv", batch=1, heads=8, kv_heads=8, sq=1024, sk=32768, mask=0,
             lse=False),
        # One decode step of four users with long, equal contexts.
        dict(name="decode_long", op="splitkv", batch=4, heads=32, kv_heads=8, sq=1, sk=32768, mask=0, lse=False),
        # Decode steps of a serving engine over paged caches: a full batch with
        # contexts from a chat turn to a long document, and a small batch of
        # short chats, where the launches count.
        dict(name="decode_paged", op="paged", seqs=32, heads=32, kv_heads=8, sq=1, min_sk=1024, max_sk=32768,
             page_size=64, mask=0, lse=False, lens_seed=2),
        dict(name="decode_paged_short", op="paged", seqs=8, heads=32, kv_heads=8, sq=1, min_sk=100, max_sk=2000,
             page_size=64, mask=0, lse=False, lens_seed=3),
        # Chunked prefill of the same engine: new prompt chunks behind what
        # their sequences have cached already.
        dict(name="prefill_paged", op="paged", seqs=4, heads=32, kv_heads=8, sq=1024, min_sk=1024, max_sk=8192,
             page_size=64, mask=BOTTOM_RIGHT, lse=False, lens_seed=4),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    """One more case of the listed ranges (rng: random.Random)."""
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= 2.0e12 and w["bytes"] <= 2.0e9:
            return case


def _draw(rng):
    op = rng.choice(["forward", "forward", "forward", "varlen", "splitkv", "paged", "paged"])
    heads = rng.choice([8, 16, 32])
    kv_heads = heads // rng.choice([1, 1, 4, 8])
    lse = rng.random() < 0.5
    if op == "forward":
        sq = _log_int(rng, 128, 8192)
        sk = sq if rng.random() < 0.7 else _log_int(rng, 128, 8192)
        return dict(op=op, batch=_log_int(rng, 1, 32), heads=heads, kv_heads=kv_heads, sq=sq, sk=sk,
                    mask=rng.randrange(2), lse=lse, layout=rng.choice(["bshd", "bshd", "bhsd"]))
    if op == "varlen":
        high = _log_int(rng, 256, 4096)
        return dict(op=op, seqs=_log_int(rng, 4, 64), heads=heads, kv_heads=kv_heads,
                    min_len=max(1, high // rng.choice([2, 8, 64])), max_len=high, mask=rng.choice([0, 1, 1]), lse=lse,
                    lens_seed=rng.randrange(1 << 30))
    if op == "splitkv":
        if rng.random() < 0.4:
            return dict(op=op, batch=1, heads=8, kv_heads=8, sq=_log_int(rng, 64, 2048),
                        sk=_log_int(rng, 4096, 65536), mask=0, lse=lse)
        return dict(op=op, batch=_log_int(rng, 1, 16), heads=32, kv_heads=8, sq=rng.choice([1, 1, 1, 4]),
                    sk=_log_int(rng, 512, 65536), mask=0, lse=False)
    high = _log_int(rng, 512, 32768)
    low = max(1, high // rng.choice([2, 8, 32]))
    page = rng.choice([64, 64, 128])
    if rng.random() < 0.6:
        sq = rng.choice([1, 1, 1, 4])
        return dict(op=op, seqs=_log_int(rng, 1, 32), heads=32, kv_heads=8, sq=sq, min_sk=max(low, sq), max_sk=high,
                    page_size=page, mask=0 if sq == 1 else BOTTOM_RIGHT, lse=False, lens_seed=rng.randrange(1 << 30))
    sq = _log_int(rng, 64, min(2048, high))
    return dict(op=op, seqs=_log_int(rng, 1, 8), heads=heads, kv_heads=kv_heads, sq=sq, min_sk=max(low, sq),
                max_sk=high, page_size=page, mask=BOTTOM_RIGHT, lse=False, lens_seed=rng.randrange(1 << 30))


# ---- shapes ----------------------------------------------------------------
def _spread(seed, n, low, high):
    """n lengths spread over [low, high] (over their logarithm), the longest among them."""
    rng = random.Random(seed)
    lens = [_log_int(rng, low, high) for _ in range(n)]
    lens[rng.randrange(n)] = high
    return lens


def _sequences(case):
    """(queries, keys) of each sequence of the case."""
    if case["op"] == "varlen":
        return [(n, n) for n in _spread(case["lens_seed"], case["seqs"], case["min_len"], case["max_len"])]
    if case["op"] == "paged":
        keys = _spread(case["lens_seed"], case["seqs"], case["min_sk"], case["max_sk"])
        if case["sq"] <= 32:
            return [(case["sq"], n) for n in keys]
        # Chunked prefill: chunks of up to sq new tokens, ragged at the end of a prompt.
        rng = random.Random(case["lens_seed"] + 1)
        return [(case["sq"] if i == 0 else rng.randint(max(1, case["sq"] // 4), case["sq"]), n)
                for i, n in enumerate(keys)]
    return [(case["sq"], case["sk"])] * case["batch"]


def _visible(sq, sk, mask):
    """(query, key) pairs that attend to each other."""
    if mask == 0:
        return sq * sk
    shift = sk - sq if mask == BOTTOM_RIGHT else 0
    return sum(min(sk, max(0, i + 1 + shift)) for i in range(sq))


def work(case):
    seqs = _sequences(case)
    pairs = sum(_visible(sq, sk, case["mask"]) for sq, sk in seqs)
    # A top-left causal call sees no key past its last query.
    keys = sum(min(sq, sk) if case["mask"] == 1 else sk for sq, sk in seqs)
    queries = sum(sq for sq, _ in seqs)
    size = 2 * queries * case["heads"] * D * 2 + 2 * keys * case["kv_heads"] * D * 2
    if case["lse"]:
        size += queries * case["heads"] * 4
    return {"bytes": size, "flops": 4 * case["heads"] * D * pairs}


def tolerance(case):
    # BF16 weights and outputs: 2.3e-3 from the 64-bit result for one
    # implementation, a little over 3e-3 between two.
    return {"rel": 1e-2}


# ---- inputs and calls --------------------------------------------------------
def _randn(shape, gen):
    return torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32).to(torch.bfloat16)


def _offsets(lens):
    total, out = 0, [0]
    for n in lens:
        total += n
        out.append(total)
    return out


def _int32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEVICE)


def _inputs(case, seed):
    """Q/K/V (N(0, 1) in BF16) and, for packed and paged cases, where the sequences lie."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    h, kvh = case["heads"], case["kv_heads"]
    seqs = _sequences(case)
    if case["op"] in ("forward", "splitkv"):
        b, sq, sk = case["batch"], case["sq"], case["sk"]
        if case.get("layout") == "bhsd":
            q, k, v = (_randn((b, n, s, D), gen).transpose(1, 2) for n, s in ((h, sq), (kvh, sk), (kvh, sk)))
        else:
            q, k, v = (_randn((b, s, n, D), gen) for n, s in ((h, sq), (kvh, sk), (kvh, sk)))
        return dict(q=q, k=k, v=v)
    cu_q = _offsets([sq for sq, _ in seqs])
    x = dict(q=_randn((cu_q[-1], h, D), gen), cu_q=_int32(cu_q), max_q=max(sq for sq, _ in seqs),
             max_k=max(sk for _, sk in seqs), total_k=sum(sk for _, sk in seqs))
    if case["op"] == "varlen":
        x.update(k=_randn((x["total_k"], kvh, D), gen), v=_randn((x["total_k"], kvh, D), gen), cu_k=x["cu_q"])
        return x
    # Paged caches: every sequence's pages lie anywhere in the pool.
    page = case["page_size"]
    pages = [-(-sk // page) for _, sk in seqs]
    order = torch.randperm(sum(pages), generator=gen, device=DEVICE, dtype=torch.int32)
    table = torch.zeros((len(seqs), max(pages)), dtype=torch.int32, device=DEVICE)
    for i, start in enumerate(_offsets(pages)[:-1]):
        table[i, :pages[i]] = order[start:start + pages[i]]
    x.update(k=_randn((sum(pages), page, kvh, D), gen), v=_randn((sum(pages), page, kvh, D), gen),
             seqlens=_int32([sk for _, sk in seqs]), table=table)
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    runner = __graft_entry__.import_package().Runner()
    q, h = x["q"], case["heads"]
    state = dict(case=case, runner=runner, o=torch.empty_like(q), lse=None, workspace=None, **x)
    if case["lse"]:
        shape = (case["batch"], h, case["sq"]) if q.dim() == 4 else (h, q.shape[0])
        state["lse"] = torch.empty(shape, dtype=torch.float32, device=DEVICE)
    # A serving loop keeps its split-KV workspace between steps.
    need = 0
    if case["op"] == "splitkv":
        need = runner.splitkv_workspace_size(case["batch"], h, case["sq"], case["sk"], case["mask"],
                                             kv_heads=case["kv_heads"])
    elif case["op"] == "paged":
        need = runner.splitkv_paged_workspace_size(case["seqs"], h, case["kv_heads"], x["max_q"], x["max_k"],
                                                   q.shape[0], x["total_k"], case["page_size"], x["table"].shape[1],
                                                   x["k"].shape[0], causal=case["mask"])
    if case["op"] in ("splitkv", "paged"):
        state["workspace"] = torch.empty(max(need, 1), dtype=torch.uint8, device=DEVICE)
    return state


def run(state):
    s, case = state, state["case"]
    runner, mask = s["runner"], case["mask"]
    if case["op"] == "forward":
        if case["layout"] == "bhsd":
            runner.call_strided(s["q"], s["k"], s["v"], s["o"], s["lse"], mask)
        elif case["kv_heads"] != case["heads"]:
            runner.call_gqa(s["q"], s["k"], s["v"], s["o"], s["lse"], mask)
        else:
            runner.call(s["q"], s["k"], s["v"], s["o"], s["lse"], mask)
    elif case["op"] == "splitkv":
        runner.call_splitkv(s["q"], s["k"], s["v"], s["o"], s["lse"], mask, workspace=s["workspace"])
    elif case["op"] == "varlen":
        runner.call_varlen(s["q"], s["k"], s["v"], s["o"], s["lse"], s["cu_q"], s["cu_k"], s["max_q"], s["max_k"],
                           mask)
    else:
        runner.call_splitkv_paged(s["q"], s["k"], s["v"], s["o"], s["lse"], s["cu_q"], s["seqlens"], s["table"],
                                  s["max_q"], s["max_k"], workspace=s["workspace"], total_k=s["total_k"],
                                  causal=mask)
    return (s["o"], s["lse"]) if s["lse"] is not None else s["o"]


# ---- the same in 64 bits -------------------------------------------------------
def _attend(q, k, v, mask):
    """One sequence and one K/V head: q [g, sq, D], k and v [sk, D] -> O [g, sq, D], LSE [g, sq] in float64."""
    g, sq, _ = q.shape
    sk = k.shape[0]
    k, v = k.double(), v.double()
    o = torch.empty((g, sq, D), dtype=torch.float64, device=q.device)
    lse = torch.empty((g, sq), dtype=torch.float64, device=q.device)
    step = max(1, (1 << 27) // sk)                       # rows per block: 1 GiB of scores
    shift = sk - sq if mask == BOTTOM_RIGHT else 0
    keys = torch.arange(sk, device=q.device)
    for i in range(g):
        for r in range(0, sq, step):
            s = (q[i, r:r + step].double() @ k.T) * SCALE
            if mask:
                rows = torch.arange(r, r + s.shape[0], device=q.device) + shift
                s.masked_fill_(keys[None, :] > rows[:, None], -math.inf)
            lse[i, r:r + step] = torch.logsumexp(s, dim=1)
            o[i, r:r + step] = torch.softmax(s, dim=1) @ v
    return o, lse


def exact(case, seed):
    x = _inputs(case, seed)
    h, kvh = case["heads"], case["kv_heads"]
    g = h // kvh
    q, seqs = x["q"], _sequences(case)
    batched = q.dim() == 4
    o = torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
    lse = torch.empty((q.shape[0], h, q.shape[1]) if batched else (h, q.shape[0]), dtype=torch.float64, device=DEVICE)
    cu_q = _offsets([sq for sq, _ in seqs])
    for b, (sq, sk) in enumerate(seqs):
        if batched:
            qb, kb, vb, ob, lb = q[b], x["k"][b], x["v"][b], o[b], lse[b]
        else:
            rows = slice(cu_q[b], cu_q[b + 1])
            qb, ob, lb = q[rows], o[rows], lse[:, rows]
            if case["op"] == "varlen":
                kb, vb = x["k"][rows], x["v"][rows]
            else:
                pages = x["table"][b, :-(-sk // case["page_size"])].long()
                kb, vb = (x[n][pages].reshape(-1, kvh, D)[:sk] for n in ("k", "v"))
        for j in range(kvh):
            heads = slice(j * g, (j + 1) * g)
            oj, lj = _attend(qb[:, heads].transpose(0, 1), kb[:, j], vb[:, j], case["mask"])
            ob[:, heads] = oj.transpose(0, 1)
            lb[heads] = lj
    return (o, lse) if case["lse"] else o
