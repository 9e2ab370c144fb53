"""GPU checks that a batch is not slower than the parts of it that bound it.

Each case compares two calls of this library on one box, timed in turn, by a
ratio with a wide margin on both sides of what was measured.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ratio(torch, slow, fast, calls=20, rounds=5):
    """Time of `slow` over time of `fast`: the median of the rounds' ratios."""
    def us(fn):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(calls):
            fn()
        b.record()
        torch.cuda.synchronize()
        return a.elapsed_time(b) * 1e3 / calls
    us(slow), us(fast)
    times = [(us(slow), us(fast)) for _ in range(rounds)]
    print("  us:", *("%.1f / %.1f" % t for t in times), flush=True)
    return float(np.median([s / f for s, f in times]))


def _paged(torch, runner, h, kvh, lens_q, lens_k, causal=0, ps=64, splits=0, total_k=True):
    """A paged call on its own buffers; returns the function that runs it."""
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(7)
    mk = lambda *s: torch.randn(s, device=dev, dtype=torch.float32, generator=g).to(torch.bfloat16)
    pages = [-(-n // ps) for n in lens_k]
    table = torch.zeros((len(pages), max(pages)), dtype=torch.int32)
    first = 0
    for i, n in enumerate(pages):
        table[i, :n] = torch.arange(first, first + n)
        first += n
    table = table.to(dev)
    cu_q = torch.tensor(np.concatenate([[0], np.cumsum(lens_q)]), dtype=torch.int32, device=dev)
    keys = torch.tensor(lens_k, dtype=torch.int32, device=dev)
    q, kc, vc = mk(sum(lens_q), h, 128), mk(first, ps, kvh, 128), mk(first, ps, kvh, 128)
    o = torch.empty_like(q)
    max_q, max_k = max(lens_q), max(lens_k)
    total = sum(lens_k) if total_k else max_k * len(lens_k)
    need = runner.splitkv_paged_workspace_size(len(lens_k), h, kvh, max_q, max_k, len(q), total, ps, table.shape[1],
                                               first, splits, causal=causal)
    ws = torch.empty(need, device=dev, dtype=torch.uint8)
    return lambda: runner.call_splitkv_paged(q, kc, vc, o, None, cu_q, keys, table, max_q, max_k, splits,
                                             workspace=ws, total_k=sum(lens_k) if total_k else None, causal=causal)


def test_short_sequences_beside_a_long_one(gpu_runner):
    """Decode: 63 sequences of 50 keys beside one of 200000 (H32 KVH8) cost a
    few percent of the long one (165 us against 155), not what a workgroup
    takes for 50 of them in a row (352 us)."""
    import torch
    print("  decode 63 x 50 keys + 200000", flush=True)
    both = _paged(torch, gpu_runner, 32, 8, [1] * 64, [50] * 63 + [200000])
    alone = _paged(torch, gpu_runner, 32, 8, [1], [200000])
    assert _ratio(torch, both, alone) < 1.6


def test_ragged_decode_of_several_q_tiles(gpu_runner):
    """Decode of 16 queries of 8 heads on one K/V head (four 32-row tiles, 41
    sequences of 24000-30000 keys): Auto's equal ranges are no slower than the
    chunks of its plan (the tiles of a range share its keys in one XCD's L2;
    spread over the XCDs they read them four times)."""
    import torch
    lens = [24000 + 157 * i for i in range(41)]
    print("  decode 41 x 16 queries H8 KVH1", flush=True)
    auto = _paged(torch, gpu_runner, 8, 1, [16] * 41, lens, causal=2)
    plan = gpu_runner.splitkv_paged_select(41, 8, 1, 16, max(lens), 41 * 16, sum(lens), 64, -(-max(lens) // 64),
                                           sum(-(-n // 64) for n in lens), causal=2)
    chunks = _paged(torch, gpu_runner, 8, 1, [16] * 41, lens, causal=2, splits=plan)
    assert _ratio(torch, auto, chunks) < 1.15


def test_ragged_decode_without_a_total(gpu_runner):
    """Decode of 105 sequences of 324-2545 keys (H12 KVH3) when the caller does
    not say how many keys there are: no slower than when it does."""
    import torch
    lens = np.random.default_rng(3).integers(324, 2546, size=105).tolist()
    print("  decode 105 ragged, no total", flush=True)
    unknown = _paged(torch, gpu_runner, 12, 3, [1] * 105, lens, total_k=False)
    known = _paged(torch, gpu_runner, 12, 3, [1] * 105, lens)
    assert _ratio(torch, unknown, known) < 1.12


def test_paged_prefill_of_few_queries(gpu_runner):
    """Prefill of 2 x 40 queries on 12288 keys (H8, 8 chunks of 24 tiles), K/V
    from memory (12 caches in turn): through pages about as fast as from
    contiguous K/V, two key tiles in flight in both (37.7 us and 34.6; with one
    in flight through pages 43.8)."""
    import torch
    print("  prefill 2 x 40 on 12288 keys, 12 caches", flush=True)
    paged, contiguous = [], []
    for _ in range(12):
        paged.append(_paged(torch, gpu_runner, 8, 8, [40, 40], [12288, 12288], splits=8))
        mk = lambda s: torch.randn((2, s, 8, 128), device="cuda").to(torch.bfloat16)
        q, k, v = mk(40), mk(12288), mk(12288)
        o = torch.empty_like(q)
        ws = torch.empty(gpu_runner.splitkv_workspace_size(2, 8, 40, 12288, False, 8), device="cuda",
                         dtype=torch.uint8)
        contiguous.append(lambda q=q, k=k, v=v, o=o, ws=ws: gpu_runner.call_splitkv(q, k, v, o, None, False, 8,
                                                                                   workspace=ws))
    all_of = lambda calls: lambda: [c() for c in calls]
    assert _ratio(torch, all_of(paged), all_of(contiguous), calls=3) < 1.18


# (heads, kv_heads, causal, total known, [(sq, sk), ...]) where a count that
# looked cheap was not: one query tile of every sequence counted as half a one;
# unknown lengths; the last q tile of a square bottom-right batch.
PREFILL = {
    "short_queries": (32, 8, 0, True, [(40 + 2 * i, 22000 + 300 * i) for i in range(11)]),
    "unknown_total": (4, 4, 2, False, [(24 + 5 * (i % 14), 6630 + 1100 * i) for i in range(43)]),
    "square": (8, 8, 2, True, [(4096, 4096)]),
}


@pytest.mark.parametrize("name", PREFILL)
def test_prefill_auto_against_its_plan(gpu_runner, name):
    """Auto prefill over paged caches is no slower than its plan's chunk count."""
    import torch
    h, kvh, causal, known, lens = PREFILL[name]
    lq, lk = [s for s, _ in lens], [s for _, s in lens]
    print(f"  paged prefill {name}", flush=True)
    auto = _paged(torch, gpu_runner, h, kvh, lq, lk, causal=causal, total_k=known)
    plan = gpu_runner.splitkv_paged_select(len(lens), h, kvh, max(lq), max(lk), sum(lq), sum(lk), 64,
                                           -(-max(lk) // 64), sum(-(-n // 64) for n in lk), causal=causal)
    chunks = _paged(torch, gpu_runner, h, kvh, lq, lk, causal=causal, splits=plan)
    assert _ratio(torch, auto, chunks) < 1.08


def test_short_packed_sequences(gpu_runner):
    """256 packed sequences of 16 tokens (H32 KVH8) take no longer than 257,
    which are too many for sorted item lists: there is nothing to sort."""
    import torch
    print("  packed 256 x 16 and 257 x 16", flush=True)
    calls = []
    for n in (256, 257):
        mk = lambda heads: torch.randn((n * 16, heads, 128), device="cuda").to(torch.bfloat16)
        q, k, v = mk(32), mk(8), mk(8)
        o = torch.empty_like(q)
        cu = torch.arange(n + 1, device="cuda", dtype=torch.int32) * 16
        calls.append(lambda q=q, k=k, v=v, o=o, cu=cu: gpu_runner.call_varlen(q, k, v, o, None, cu, cu, 16, 16, False))
    assert _ratio(torch, *calls, calls=50) < 1.035


def _packed(torch, runner, h, kvh, lens, causal):
    mk = lambda heads: torch.randn((sum(lens), heads, 128), device="cuda").to(torch.bfloat16)
    q, k, v = mk(h), mk(kvh), mk(kvh)
    o = torch.empty_like(q)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device="cuda")
    return lambda: runner.call_varlen(q, k, v, o, None, cu, cu, max(lens), max(lens), causal)


def test_packed_sequences_of_few_q_tiles(gpu_runner):
    """40 causal sequences of 300 tokens (H16, three 128-row q tiles each, 3.75
    rounds of workgroups) cost a tenth less than 44: the q tiles of a sequence
    run together in both."""
    import torch
    print("  packed causal 40 x 300 and 44 x 300", flush=True)
    calls = [_packed(torch, gpu_runner, 16, 16, [300] * n, True) for n in (40, 44)]
    assert _ratio(torch, *calls, calls=50) < 0.97


def test_packed_heads_in_no_xcd_shares(gpu_runner):
    """56 sequences of 148 tokens, dense, with 4 heads: as fast as 28 with 8,
    each sequence's full and short q tile on the same XCD in both."""
    import torch
    print("  packed dense 56 x 148 H4 and 28 x 148 H8", flush=True)
    calls = [_packed(torch, gpu_runner, h, h, [148] * n, False) for h, n in ((4, 56), (8, 28))]
    assert _ratio(torch, *calls, calls=50) < 1.1
