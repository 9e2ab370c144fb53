"""GPU checks of split-KV decode over paged K/V caches (fav4_bshd_forward_splitkv_paged) via the C ABI.

Each sequence's keys are scattered over randomly chosen pages of the caches;
the pages no sequence uses hold NaN, and block-table entries past a
sequence's pages hold out-of-range numbers (which the kernel clamps and never
reads through), so a wrong page, slot or head shows up.  Pins:
  * bitwise equality with fav4_bshd_forward_splitkv_varlen on the same keys
    stored contiguously, at the same explicit chunk count (same plan, chunk
    bounds and merge), for page sizes 32, 64 and 256 and MHA / GQA / MQA;
  * every sequence against the FP64 oracle at the reference harness's bar,
    Auto and explicit chunk counts, LSE on and off;
  * a sequence without queries writes nothing, one without keys gets O = 0
    and LSE = -inf, and rows after O / LSE are never written.
"""
import numpy as np
import pytest

from oracle import attention as orc
from tests.conftest import to_device, to_host_bits

pytestmark = pytest.mark.gpu

GUARD = 64
NAN_BF16 = 0x7FC0

# (heads, kv_heads, page_size, [(sq, sk), ...], explicit chunk count)
CASES = [
    (32, 8, 32, [(1, 4096), (1, 100), (1, 1), (1, 9000), (1, 33), (1, 2048)], 7),
    (8, 1, 64, [(16, 3000), (5, 1), (32, 700), (1, 5000)], 5),
    (4, 4, 256, [(3, 300), (32, 4096), (0, 50), (7, 0), (1, 20000)], 16),
    (6, 2, 32, [(32, 32), (31, 64), (17, 1025)], 2),
]


def _build(heads, kv_heads, page_size, lens, seed):
    """Packed Q, contiguous packed K/V, and paged caches holding the same keys."""
    rng = np.random.default_rng(seed)
    qs, ks, vs = [], [], []
    for i, (sq, sk) in enumerate(lens):
        q, _, _ = orc.make_inputs(1, heads, max(sq, 1), max(sk, 1), "normal", seed=seed + 2 * i)
        _, k, v = orc.make_inputs(1, kv_heads, max(sq, 1), max(sk, 1), "normal", seed=seed + 2 * i + 1)
        qs.append(q[0, :sq])
        ks.append(k[0, :sk])
        vs.append(v[0, :sk])
    npages = [-(-sk // page_size) for _, sk in lens]
    max_pages = max(max(npages), 1)
    num_pages = sum(npages) + 7                       # 7 pages nobody uses
    perm = rng.permutation(num_pages)
    kc = np.full((num_pages, page_size, kv_heads, 128), NAN_BF16, dtype=np.uint16)
    vc = np.full_like(kc, NAN_BF16)
    table = rng.choice([-3, num_pages, 1 << 30], size=(len(lens), max_pages)).astype(np.int32)
    nxt = 0
    for i, (_, sk) in enumerate(lens):
        for p in range(npages[i]):
            page = perm[nxt]
            nxt += 1
            table[i, p] = page
            rows = slice(p * page_size, min(sk, (p + 1) * page_size))
            n = rows.stop - rows.start
            kc[page, :n] = ks[i][rows]
            vc[page, :n] = vs[i][rows]
    cu_q = np.concatenate([[0], np.cumsum([s for s, _ in lens])]).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum([s for _, s in lens])]).astype(np.int32)
    seqlens_k = np.array([s for _, s in lens], dtype=np.int32)
    return (np.concatenate(qs), np.concatenate(ks), np.concatenate(vs), kc, vc, cu_q, cu_k, seqlens_k, table)


def _out(torch, dev, tq, h, with_lse):
    o_buf = torch.full((tq + GUARD, h, 128), float("nan"), device=dev, dtype=torch.bfloat16)
    l_buf = torch.full((h * tq + GUARD,), float("nan"), device=dev, dtype=torch.float32)
    return o_buf, l_buf, o_buf[:tq], (l_buf[:h * tq].view(h, tq) if with_lse else None)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "h%dkv%d_p%d_n%d" % (c[0], c[1], c[2], len(c[3])))
def test_splitkv_paged(gpu_runner, case):
    import torch
    h, kvh, ps, lens, splits = case
    q, k, v, kc, vc, cu_q, cu_k, seqlens_k, table = _build(h, kvh, ps, lens, seed=17)
    dev = torch.device("cuda:0")
    qd, kd, vd, kcd, vcd = (to_device(x, dev) for x in (q, k, v, kc, vc))
    cq, ck, sk_d, tb = (torch.from_numpy(x).to(dev) for x in (cu_q, cu_k, seqlens_k, table))
    max_q = max(s for s, _ in lens)
    max_k = max(s for _, s in lens)
    tq, group = len(q), h // kvh
    print(f"  splitkv paged H{h} KVH{kvh} page {ps} lens={lens} splits={splits}", flush=True)

    # bitwise against the contiguous packed split-KV at the same chunk count
    ob, lb, o, lse = _out(torch, dev, tq, h, True)
    gpu_runner.call_splitkv_paged(qd, kcd, vcd, o, lse, cq, sk_d, tb, max_q, max_k, splits, total_k=len(k))
    ob2, lb2, o2, lse2 = _out(torch, dev, tq, h, True)
    gpu_runner.call_splitkv_varlen(qd, kd, vd, o2, lse2, cq, ck, max_q, max_k, False, splits)
    torch.cuda.synchronize()
    assert torch.equal(o.view(torch.int16), o2.view(torch.int16))
    assert torch.equal(lse.view(torch.int32), lse2.view(torch.int32))
    assert torch.isnan(ob[tq:]).all().item() and torch.isnan(lb[h * tq:]).all().item()

    # Auto, LSE off, against the oracle (and the explicit run's empty rows)
    ob3, lb3, o3, _ = _out(torch, dev, tq, h, False)
    gpu_runner.call_splitkv_paged(qd, kcd, vcd, o3, None, cq, sk_d, tb, max_q, max_k, 0, total_k=len(k))
    torch.cuda.synchronize()
    assert torch.isnan(ob3[tq:]).all().item() and torch.isnan(lb3).all().item()
    for i, (sq, sk) in enumerate(lens):
        a, b = cu_q[i], cu_q[i + 1]
        c, d = cu_k[i], cu_k[i + 1]
        if sq == 0:
            continue
        if sk == 0:
            assert (o[a:b].float() == 0).all().item() and (o3[a:b].float() == 0).all().item(), i
            assert torch.isneginf(lse[:, a:b]).all().item(), i
            continue
        ke = np.repeat(k[c:d][None], group, axis=2)
        ve = np.repeat(v[c:d][None], group, axis=2)
        ref, ref_lse = orc.attention_fp64(q[a:b][None], ke, ve, orc.DEFAULT_SCALE, False)
        e = orc.errors(to_host_bits(o[a:b])[None], lse[:, a:b].cpu().numpy()[None], ref, ref_lse)
        assert orc.check_acceptance_tolerance(e) and orc.check_reference_tolerance(e), (i, sq, sk, e)
        e3 = orc.errors(to_host_bits(o3[a:b])[None], None, ref, None)
        assert orc.check_acceptance_tolerance(e3) and orc.check_reference_tolerance(e3), ("auto", i, e3)


def test_splitkv_paged_single_chunk_and_long_cache(gpu_runner):
    """One chunk (max_seqlen_k <= 64 key tiles: still the split kernels and the
    merge), and a cache long enough that the 64-tile chunk cap raises an
    explicit count of 2 (2188 key tiles -> 35 chunks)."""
    import torch
    h, kvh, ps = 16, 4, 128
    dev = torch.device("cuda:0")
    group = h // kvh
    for lens, max_k, splits, want in (([(2, 2048), (1, 700), (3, 0)], 2048, 1, 1),
                                      ([(2, 70000), (1, 5000)], 70000, 2, 35)):
        q, k, v, kc, vc, cu_q, cu_k, seqlens_k, table = _build(h, kvh, ps, lens, seed=23)
        qd, kcd, vcd = (to_device(x, dev) for x in (q, kc, vc))
        cq, sk_d, tb = (torch.from_numpy(x).to(dev) for x in (cu_q, seqlens_k, table))
        max_q = max(s for s, _ in lens)
        need = gpu_runner.splitkv_paged_workspace_size(len(lens), h, kvh, max_q, max_k, len(q), len(k), ps,
                                                       table.shape[1], len(kc), splits)
        assert need == want * len(lens) * h * max_q * 520, (lens, need)
        print(f"  splitkv paged lens={lens} splits={splits} -> {want} chunks", flush=True)
        ob, lb, o, lse = _out(torch, dev, len(q), h, True)
        gpu_runner.call_splitkv_paged(qd, kcd, vcd, o, lse, cq, sk_d, tb, max_q, max_k, splits)
        torch.cuda.synchronize()
        assert torch.isnan(ob[len(q):]).all().item() and torch.isnan(lb[h * len(q):]).all().item()
        for i, (sq, sk) in enumerate(lens):
            a, b = cu_q[i], cu_q[i + 1]
            c, d = cu_k[i], cu_k[i + 1]
            if sk == 0:
                assert (o[a:b].float() == 0).all().item() and torch.isneginf(lse[:, a:b]).all().item(), i
                continue
            ke = np.repeat(k[c:d][None], group, axis=2)
            ve = np.repeat(v[c:d][None], group, axis=2)
            ref, ref_lse = orc.attention_fp64(q[a:b][None], ke, ve, orc.DEFAULT_SCALE, False)
            e = orc.errors(to_host_bits(o[a:b])[None], lse[:, a:b].cpu().numpy()[None], ref, ref_lse)
            assert orc.check_acceptance_tolerance(e) and orc.check_reference_tolerance(e), (splits, i, e)


def _draw(rng):
    kvh = int(rng.choice([1, 2, 4]))
    group = int(rng.choice([1, 2, 4, 8]))
    b = int(rng.integers(1, 7))
    sq_max = int(rng.choice([1, 4, 32]))
    lens = [(int(rng.integers(0, sq_max + 1)), int(rng.integers(0, 6000))) for _ in range(b)]
    lens[0] = (max(lens[0][0], 1), max(lens[0][1], 40))        # at least one row with keys past one tile
    return dict(h=kvh * group, kvh=kvh, ps=int(rng.choice([32, 64, 128, 512])), lens=lens,
                splits=int(rng.choice([2, 3, 8, 33, 200])), lse=bool(rng.integers(0, 2)))


RANDOM = [_draw(np.random.default_rng(500 + i)) for i in range(12)]


@pytest.mark.parametrize("case", RANDOM, ids=lambda c: "h%dkv%d_p%d_b%d_s%d" % (c["h"], c["kvh"], c["ps"],
                                                                                len(c["lens"]), c["splits"]))
def test_splitkv_paged_random(gpu_runner, case):
    """Seeded random batches: bitwise the contiguous packed split-KV at the same
    explicit chunk count, and the FP64 oracle on every sequence."""
    import torch
    h, kvh, ps, lens, splits, with_lse = case["h"], case["kvh"], case["ps"], case["lens"], case["splits"], case["lse"]
    q, k, v, kc, vc, cu_q, cu_k, seqlens_k, table = _build(h, kvh, ps, lens, seed=31)
    dev = torch.device("cuda:0")
    qd, kd, vd, kcd, vcd = (to_device(x, dev) for x in (q, k, v, kc, vc))
    cq, ck, sk_d, tb = (torch.from_numpy(x).to(dev) for x in (cu_q, cu_k, seqlens_k, table))
    max_q = max(s for s, _ in lens)
    max_k = max(s for _, s in lens)
    tq, group = len(q), h // kvh
    print(f"  splitkv paged random H{h} KVH{kvh} page {ps} lens={lens} splits={splits}", flush=True)
    ob, lb, o, lse = _out(torch, dev, tq, h, with_lse)
    gpu_runner.call_splitkv_paged(qd, kcd, vcd, o, lse, cq, sk_d, tb, max_q, max_k, splits, total_k=len(k))
    torch.cuda.synchronize()
    assert torch.isnan(ob[tq:]).all().item() and torch.isnan(lb[h * tq:]).all().item()
    # Same plan (the paged one caps chunks at 64 key tiles, which only ever
    # raises the count): same workspace size.
    ws_v = gpu_runner.splitkv_varlen_workspace_size(len(lens), h, kvh, max_q, max_k, tq, len(k), False, splits)
    ws_p = gpu_runner.splitkv_paged_workspace_size(len(lens), h, kvh, max_q, max_k, tq, len(k), ps, table.shape[1],
                                                   len(kc), splits)
    if ws_v == ws_p:
        _, _, o2, lse2 = _out(torch, dev, tq, h, with_lse)
        gpu_runner.call_splitkv_varlen(qd, kd, vd, o2, lse2, cq, ck, max_q, max_k, False, splits)
        torch.cuda.synchronize()
        assert torch.equal(o.view(torch.int16), o2.view(torch.int16))
        if with_lse:
            assert torch.equal(lse.view(torch.int32), lse2.view(torch.int32))
    for i, (sq, sk) in enumerate(lens):
        a, b = cu_q[i], cu_q[i + 1]
        c, d = cu_k[i], cu_k[i + 1]
        if sq == 0:
            continue
        if sk == 0:
            assert (o[a:b].float() == 0).all().item(), i
            continue
        ke = np.repeat(k[c:d][None], group, axis=2)
        ve = np.repeat(v[c:d][None], group, axis=2)
        ref, ref_lse = orc.attention_fp64(q[a:b][None], ke, ve, orc.DEFAULT_SCALE, False)
        got_lse = lse[:, a:b].cpu().numpy()[None] if with_lse else None
        e = orc.errors(to_host_bits(o[a:b])[None], got_lse, ref, ref_lse if with_lse else None)
        assert orc.check_acceptance_tolerance(e) and orc.check_reference_tolerance(e), (i, sq, sk, e)


def _bottom_right_ref(q, k, v, group):
    """FP64 bottom-right causal (query i sees keys j <= sk - sq + i) from the
    top-left oracle: queries padded in front to sk rows when sq <= sk, else
    the rows that see keys are the last sk, top-left against all keys."""
    sq, sk = len(q), len(k)
    ke = np.repeat(k[None], group, axis=2)
    ve = np.repeat(v[None], group, axis=2)
    h = q.shape[1]
    o = np.zeros((1, sq, h, 128))
    lse = np.full((1, h, sq), -np.inf)
    if sk == 0:
        return o, lse
    if sq <= sk:
        qp = np.concatenate([np.zeros((sk - sq,) + q.shape[1:], dtype=q.dtype), q])[None]
        return orc.attention_fp64(qp, ke, ve, orc.DEFAULT_SCALE, True, rows=np.arange(sk - sq, sk))
    ref, ref_lse = orc.attention_fp64(q[sq - sk:][None], ke, ve, orc.DEFAULT_SCALE, True)
    o[:, sq - sk:] = ref
    lse[:, :, sq - sk:] = ref_lse
    return o, lse


@pytest.mark.parametrize("ps", [32, 128])
def test_splitkv_bottom_right_causal(gpu_runner, ps):
    """causal = 2 on the packed and the paged decode calls: the FP64 oracle
    (bottom-right, including sequences with more queries than keys, whose
    first rows see no key), and paged bitwise the packed call at the same
    chunk count."""
    import torch
    h, kvh = 8, 2
    lens = [(4, 3000), (1, 700), (32, 5000), (17, 17), (20, 9), (5, 0), (0, 40), (32, 65)]
    q, k, v, kc, vc, cu_q, cu_k, seqlens_k, table = _build(h, kvh, ps, lens, seed=41)
    dev = torch.device("cuda:0")
    qd, kd, vd, kcd, vcd = (to_device(x, dev) for x in (q, k, v, kc, vc))
    cq, ck, sk_d, tb = (torch.from_numpy(x).to(dev) for x in (cu_q, cu_k, seqlens_k, table))
    max_q, max_k, tq, group = 32, 5000, len(q), h // kvh
    for splits in (0, 1, 6):
        print(f"  bottom-right causal page {ps} splits={splits}", flush=True)
        ob, lb, o, lse = _out(torch, dev, tq, h, True)
        gpu_runner.call_splitkv_varlen(qd, kd, vd, o, lse, cq, ck, max_q, max_k, 2, splits)
        ob2, lb2, o2, lse2 = _out(torch, dev, tq, h, True)
        gpu_runner.call_splitkv_paged(qd, kcd, vcd, o2, lse2, cq, sk_d, tb, max_q, max_k, splits, total_k=len(k),
                                      causal=2)
        torch.cuda.synchronize()
        assert torch.isnan(ob[tq:]).all().item() and torch.isnan(lb[h * tq:]).all().item()
        assert torch.isnan(ob2[tq:]).all().item() and torch.isnan(lb2[h * tq:]).all().item()
        ws_v = gpu_runner.splitkv_varlen_workspace_size(len(lens), h, kvh, max_q, max_k, tq, len(k), 2, splits)
        ws_p = gpu_runner.splitkv_paged_workspace_size(len(lens), h, kvh, max_q, max_k, tq, len(k), ps,
                                                       table.shape[1], len(kc), splits, causal=2)
        if ws_v == ws_p:      # same plan (one explicit chunk over 157 key tiles: the paged cap makes 3)
            assert torch.equal(o.view(torch.int16), o2.view(torch.int16)), splits
            assert torch.equal(lse.view(torch.int32), lse2.view(torch.int32)), splits
        for out_o, out_lse in ((o, lse), (o2, lse2)):
            _check_bottom_right(out_o, out_lse, q, k, v, cu_q, cu_k, lens, group, splits)


def _check_bottom_right(o, lse, q, k, v, cu_q, cu_k, lens, group, splits):
    """Every sequence of a bottom-right causal output against the FP64 reference."""
    for i, (sq, sk) in enumerate(lens):
        a, b = cu_q[i], cu_q[i + 1]
        c, d = cu_k[i], cu_k[i + 1]
        if sq == 0:
            continue
        ref, ref_lse = _bottom_right_ref(q[a:b], k[c:d], v[c:d], group)
        got, got_lse = to_host_bits(o[a:b])[None], lse[:, a:b].cpu().numpy()[None]
        seen = np.isfinite(ref_lse[0, 0])                       # rows that see at least one key
        assert (got_lse[:, :, ~seen] == -np.inf).all() and (orc.bf16_to_f32(got[:, ~seen]) == 0).all(), i
        if seen.any():
            e = orc.errors(got[:, seen], got_lse[:, :, seen], ref[:, seen], ref_lse[:, :, seen])
            assert orc.check_acceptance_tolerance(e) and orc.check_reference_tolerance(e), (splits, i, e)


def _check_dense(o, lse, q, k, v, cu_q, cu_k, lens, group):
    """Every sequence of a dense output against the FP64 oracle."""
    for i, (sq, sk) in enumerate(lens):
        a, b = cu_q[i], cu_q[i + 1]
        c, d = cu_k[i], cu_k[i + 1]
        if sq == 0:
            continue
        got, got_lse = to_host_bits(o[a:b])[None], lse[:, a:b].cpu().numpy()[None]
        if sk == 0:
            assert (orc.bf16_to_f32(got) == 0).all() and (got_lse == -np.inf).all(), i
            continue
        ke, ve = (np.repeat(x[c:d][None], group, axis=2) for x in (k, v))
        ref, ref_lse = orc.attention_fp64(q[a:b][None], ke, ve, orc.DEFAULT_SCALE, False)
        e = orc.errors(got, got_lse, ref, ref_lse)
        assert orc.check_acceptance_tolerance(e) and orc.check_reference_tolerance(e), (i, sq, sk, e)


@pytest.mark.parametrize("ps", [64, 256])
def test_splitkv_paged_prefill(gpu_runner, ps):
    """Queries longer than 32 over paged caches: dense and
    bottom-right causal against the FP64 oracle on ragged batches (several q
    tiles, q tiles past short sequences, sq > sk), and a uniform batch bitwise
    the contiguous split-KV at the same chunk count."""
    import torch
    h, kvh = 8, 2
    group = h // kvh
    dev = torch.device("cuda:0")
    lens = [(600, 3000), (33, 700), (300, 300), (64, 20), (0, 100), (1, 4100)]
    q, k, v, kc, vc, cu_q, cu_k, seqlens_k, table = _build(h, kvh, ps, lens, seed=61)
    qd, kcd, vcd = (to_device(x, dev) for x in (q, kc, vc))
    cq, sk_d, tb = (torch.from_numpy(x).to(dev) for x in (cu_q, seqlens_k, table))
    max_q, max_k, tq = 600, 4100, len(q)
    for causal, splits in ((0, 0), (0, 5), (2, 0), (2, 3)):
        print(f"  paged prefill page {ps} causal={causal} splits={splits}", flush=True)
        ob, lb, o, lse = _out(torch, dev, tq, h, True)
        gpu_runner.call_splitkv_paged(qd, kcd, vcd, o, lse, cq, sk_d, tb, max_q, max_k, splits, total_k=len(k),
                                      causal=causal)
        torch.cuda.synchronize()
        assert torch.isnan(ob[tq:]).all().item() and torch.isnan(lb[h * tq:]).all().item()
        if causal == 2:
            _check_bottom_right(o, lse, q, k, v, cu_q, cu_k, lens, group, splits)
            # the contiguous packed call: the same rows, bitwise when the plans agree
            kd, vd = to_device(k, dev), to_device(v, dev)
            _, _, o2, lse2 = _out(torch, dev, tq, h, True)
            gpu_runner.call_splitkv_varlen(qd, kd, vd, o2, lse2, cq, torch.from_numpy(cu_k).to(dev), max_q, max_k,
                                           2, splits)
            torch.cuda.synchronize()
            _check_bottom_right(o2, lse2, q, k, v, cu_q, cu_k, lens, group, splits)
            ws_v = gpu_runner.splitkv_varlen_workspace_size(len(lens), h, kvh, max_q, max_k, tq, len(k), 2, splits)
            ws_p = gpu_runner.splitkv_paged_workspace_size(len(lens), h, kvh, max_q, max_k, tq, len(k), ps,
                                                           table.shape[1], len(kc), splits, causal=2)
            if ws_v == ws_p:
                assert torch.equal(o.view(torch.int16), o2.view(torch.int16)), splits
                assert torch.equal(lse.view(torch.int32), lse2.view(torch.int32)), splits
            continue
        for i, (sq, sk) in enumerate(lens):
            a, b = cu_q[i], cu_q[i + 1]
            c, d = cu_k[i], cu_k[i + 1]
            if sq == 0:
                continue
            ke = np.repeat(k[c:d][None], group, axis=2)
            ve = np.repeat(v[c:d][None], group, axis=2)
            ref, ref_lse = orc.attention_fp64(q[a:b][None], ke, ve, orc.DEFAULT_SCALE, False)
            e = orc.errors(to_host_bits(o[a:b])[None], lse[:, a:b].cpu().numpy()[None], ref, ref_lse)
            assert orc.check_acceptance_tolerance(e) and orc.check_reference_tolerance(e), (splits, i, e)

    # uniform batch: bitwise the contiguous (BSHD) split-KV at the same chunk count
    b, sq, sk, splits = 3, 300, 2500, 4
    q, k, v, kc, vc, cu_q, cu_k, seqlens_k, table = _build(h, kvh, ps, [(sq, sk)] * b, seed=62)
    qd, kd, vd, kcd, vcd = (to_device(x, dev) for x in (q, k, v, kc, vc))
    cq, sk_d, tb = (torch.from_numpy(x).to(dev) for x in (cu_q, seqlens_k, table))
    _, _, o, lse = _out(torch, dev, b * sq, h, True)
    gpu_runner.call_splitkv_paged(qd, kcd, vcd, o, lse, cq, sk_d, tb, sq, sk, splits, total_k=b * sk)
    oc = torch.full((b, sq, h, 128), float("nan"), device=dev, dtype=torch.bfloat16)
    lc = torch.full((b, h, sq), float("nan"), device=dev, dtype=torch.float32)
    gpu_runner.call_splitkv(qd.view(b, sq, h, 128), kd.view(b, sk, kvh, 128), vd.view(b, sk, kvh, 128), oc, lc,
                            False, splits)
    torch.cuda.synchronize()
    assert torch.equal(o.view(torch.int16), oc.view(-1, h, 128).view(torch.int16))
    assert torch.equal(lse.view(torch.int32), lc.permute(1, 0, 2).reshape(h, b * sq).view(torch.int32))


def test_splitkv_paged_presized_workspace_bottom_right(gpu_runner):
    """A caller that sizes the workspace with the helper for the mask it will
    use (as for graph capture) and passes exactly that buffer: the bottom-right
    plan of B1 H8 Sq=Sk=4096 has more chunks than the dense one, so a
    dense-sized buffer would be rejected.  The call succeeds and matches the
    call that allocates its own workspace, bitwise."""
    import torch
    h, kvh, ps = 8, 8, 64
    dev = torch.device("cuda:0")
    lens = [(4096, 4096)]
    q, k, v, kc, vc, cu_q, cu_k, seqlens_k, table = _build(h, kvh, ps, lens, seed=71)
    qd, kcd, vcd = (to_device(x, dev) for x in (q, kc, vc))
    cq, sk_d, tb = (torch.from_numpy(x).to(dev) for x in (cu_q, seqlens_k, table))
    args = (1, h, kvh, 4096, 4096, len(q), len(k), ps, table.shape[1], len(kc))
    need_dense = gpu_runner.splitkv_paged_workspace_size(*args, 0, causal=0)
    need_br = gpu_runner.splitkv_paged_workspace_size(*args, 0, causal=2)
    print(f"  workspace dense {need_dense} B, bottom-right {need_br} B", flush=True)
    ws = torch.empty(need_br, device=dev, dtype=torch.uint8)
    _, _, o, lse = _out(torch, dev, len(q), h, True)
    gpu_runner.call_splitkv_paged(qd, kcd, vcd, o, lse, cq, sk_d, tb, 4096, 4096, 0, workspace=ws, total_k=len(k),
                                  causal=2)
    _, _, o2, lse2 = _out(torch, dev, len(q), h, True)
    gpu_runner.call_splitkv_paged(qd, kcd, vcd, o2, lse2, cq, sk_d, tb, 4096, 4096, 0, total_k=len(k), causal=2)
    torch.cuda.synchronize()
    assert torch.equal(o.view(torch.int16), o2.view(torch.int16))
    assert torch.equal(lse.view(torch.int32), lse2.view(torch.int32))


def _check_close(o, ref, cu_q, case):
    """Each sequence's O against another call's, RMS-relative.  Both round to
    BF16 and round their weights to BF16 against bases of their own; each is
    0.0020-0.0024 from the FP64 result, so they are up to 0.0034 apart."""
    for a, b in zip(cu_q[:-1], cu_q[1:]):
        x, y = o[a:b].double(), ref[a:b].double()
        if b > a and y.any().item():
            rel = ((x - y).norm() / y.norm()).item()
            assert rel <= 0.005, (case, int(a), rel)


# (heads, kv_heads, page_size, [(sq, sk), ...]): q tiles that end in one chunk
# beside q tiles that are merged, sizes at the edges of the 64-key and 128- /
# 256-row tiles, queries without a visible key, few sequences (sorted item
# lists) and more than 256 (plain grid), and a grid that Auto fills with one
# chunk of more than 64 pages per q tile.
PREFILL_CASES = [
    (4, 2, 64, [(200, 9001), (129, 64), (33, 65), (255, 4097)]),
    (8, 8, 64, [(257, 700), (256, 256), (128, 128), (1, 6000), (0, 500), (130, 0), (300, 90)]),
    (8, 2, 128, [(1 + 37 * i % 70, 1 + 61 * i % 400) for i in range(260)]),
    (32, 2, 64, [(256, 4500 + i) for i in range(8)]),
]


@pytest.mark.parametrize("case", PREFILL_CASES, ids=lambda c: "h%dkv%d_p%d_n%d" % (c[0], c[1], c[2], len(c[3])))
def test_paged_prefill_chunks(gpu_runner, case):
    """Bottom-right prefill over paged caches: in one chunk O is bitwise the
    unsplit packed forward's (a q tile of one chunk writes its own O); with
    more chunks it is within the reference bar (0.01 + 0.01 |ref|) of it and
    close to it relative to each sequence's own size, and bitwise the packed
    K/V call's where the plans agree; nothing is written past O and LSE."""
    import torch
    h, kvh, ps, lens = case
    q, k, v, kc, vc, cu_q, cu_k, seqlens_k, table = _build(h, kvh, ps, lens, seed=97)
    dev = torch.device("cuda:0")
    qd, kd, vd, kcd, vcd = (to_device(x, dev) for x in (q, k, v, kc, vc))
    cq, ck, sk_d, tb = (torch.from_numpy(x).to(dev) for x in (cu_q, cu_k, seqlens_k, table))
    max_q, max_k, tq = max(s for s, _ in lens), max(s for _, s in lens), len(q)
    whole_buf, _, whole, whole_lse = _out(torch, dev, tq, h, True)
    gpu_runner.call_varlen(qd, kd, vd, whole, whole_lse, cq, ck, max_q, max_k, 2)
    for splits in (1, 2, 5, 0):
        print(f"  paged prefill h{h} kv{kvh} n{len(lens)} splits {splits}", flush=True)
        ob, lb, o, lse = _out(torch, dev, tq, h, True)
        gpu_runner.call_splitkv_paged(qd, kcd, vcd, o, lse, cq, sk_d, tb, max_q, max_k, splits, total_k=len(k),
                                      causal=2)
        ob2, _, o2, _ = _out(torch, dev, tq, h, False)
        gpu_runner.call_splitkv_paged(qd, kcd, vcd, o2, None, cq, sk_d, tb, max_q, max_k, splits, total_k=len(k),
                                      causal=2)
        ob3, lb3, o3, lse3 = _out(torch, dev, tq, h, True)
        gpu_runner.call_splitkv_varlen(qd, kd, vd, o3, lse3, cq, ck, max_q, max_k, 2, splits)
        torch.cuda.synchronize()
        for guard in (ob[tq:], ob2[tq:], ob3[tq:], lb[h * tq:], lb3[h * tq:]):
            assert torch.isnan(guard).all().item(), splits
        assert torch.equal(o.view(torch.int16), o2.view(torch.int16)), splits
        sizes = (len(lens), h, kvh, max_q, max_k, tq, len(k))
        ws_p = gpu_runner.splitkv_paged_workspace_size(*sizes, ps, table.shape[1], len(kc), splits, causal=2)
        if ws_p == gpu_runner.splitkv_varlen_workspace_size(*sizes, 2, splits):
            assert torch.equal(o.view(torch.int16), o3.view(torch.int16)), splits
        if ws_p == len(lens) * h * max_q * 520:               # one chunk
            assert torch.equal(o.view(torch.int16), whole.view(torch.int16))
        else:
            assert ((o.float() - whole.float()).abs() <= 0.01 + 0.01 * whole.float().abs()).all().item(), splits
            _check_close(o, whole, cu_q, splits)
        seen = torch.isfinite(whole_lse)
        assert torch.equal(torch.isfinite(lse), seen) and torch.equal(torch.isfinite(lse3), seen)
        assert (lse[seen] - whole_lse[seen]).abs().max().item() <= 2e-4, splits


# (heads, kv_heads, page_size, [(sq, sk), ...], splits): chunks of 12 key tiles
# and more under at most 128 queries (three LDS stages; 11 tiles and 129 queries
# have two), with chunks of one and two tiles, queries without keys, keys without
# queries, and more pages than a wave's lanes.
FEW_QUERY_CASES = [
    (2, 1, 64, [(33, 5000), (128, 4097), (1, 768), (100, 0), (0, 300), (40, 30), (7, 65)], 6),
    (3, 3, 64, [(128, 64 * 24), (127, 64 * 24 - 63), (90, 64 * 12), (64, 64 * 12 + 1)], 2),
    (3, 3, 64, [(128, 64 * 22), (33, 64 * 11 + 1)], 2),
    (3, 3, 64, [(129, 64 * 24), (33, 64 * 12 + 1)], 2),
    (1, 1, 64, [(97, 9000), (34, 700)], 1),
    (2, 2, 128, [(61, 6001), (128, 3333), (90, 90)], 0),
]


@pytest.mark.parametrize("case", FEW_QUERY_CASES, ids=lambda c: "h%dkv%d_p%d_n%d_s%d" % (*c[:3], len(c[3]), c[4]))
def test_prefill_of_few_queries(gpu_runner, case):
    """Paged prefill, dense and bottom-right, and packed bottom-right, against
    the FP64 oracle, on a workspace full of NaN; nothing is written past O, LSE
    and the workspace."""
    import torch
    h, kvh, ps, lens, splits = case
    q, k, v, kc, vc, cu_q, cu_k, seqlens_k, table = _build(h, kvh, ps, lens, seed=211)
    dev = torch.device("cuda:0")
    group = h // kvh
    qd, kd, vd, kcd, vcd = (to_device(x, dev) for x in (q, k, v, kc, vc))
    cq, ck, sk_d, tb = (torch.from_numpy(x).to(dev) for x in (cu_q, cu_k, seqlens_k, table))
    max_q, max_k, tq = max(s for s, _ in lens), max(s for _, s in lens), len(q)
    sizes = (len(lens), h, kvh, max_q, max_k, tq, len(k))
    for paged, causal in ((True, 0), (True, 2), (False, 2)):
        print(f"  few queries h{h} kv{kvh} n{len(lens)} splits {splits} paged {paged} causal {causal}", flush=True)
        need = gpu_runner.splitkv_paged_workspace_size(*sizes, ps, table.shape[1], len(kc), splits, causal=causal) \
            if paged else gpu_runner.splitkv_varlen_workspace_size(*sizes, causal, splits)
        ws = torch.full((need // 4 + GUARD,), float("nan"), device=dev, dtype=torch.float32)
        ob, lb, o, lse = _out(torch, dev, tq, h, True)
        if paged:
            gpu_runner.call_splitkv_paged(qd, kcd, vcd, o, lse, cq, sk_d, tb, max_q, max_k, splits, workspace=ws,
                                          total_k=len(k), causal=causal)
        else:
            gpu_runner.call_splitkv_varlen(qd, kd, vd, o, lse, cq, ck, max_q, max_k, causal, splits, workspace=ws)
        torch.cuda.synchronize()
        for guard in (ob[tq:], lb[h * tq:], ws[need // 4:]):
            assert torch.isnan(guard).all().item(), (paged, causal)
        if causal == 2:
            _check_bottom_right(o, lse, q, k, v, cu_q, cu_k, lens, group, splits)
        else:
            _check_dense(o, lse, q, k, v, cu_q, cu_k, lens, group)


# (heads, kv_heads, page_size, [(sq, sk), ...], causal): ragged decode batches
# whose Auto takes equal ranges of the batch's keys (8 key tiles or more for
# each of 512 workgroups): ranges that cross sequences of one key tile, none,
# without queries and at the tile edges; more sequences than a wave's lanes;
# bottom-right rows without a visible key; two 32-row q tiles; a range over
# more than 64 pages.
RANGE_CASES = [
    (8, 8, 32, [(1, 9000), (1, 33), (0, 500), (1, 0), (1, 32), (1, 5000), (1, 31), (1, 1), (1, 2100)], 0),
    (16, 4, 64, [(1, 37 + 997 * i % 1200) for i in range(150)], 0),
    (32, 8, 64, [(4, 3), (4, 6001), (1, 64), (3, 0), (4, 4095), (2, 1), (4, 4097), (0, 0), (4, 3000)], 2),
    (32, 2, 128, [(4, 30000), (2, 20001), (4, 2), (1, 12900), (4, 8200)], 2),
    (16, 1, 32, [(1, 100), (8, 200000), (8, 8), (5, 90001)], 0),
]


@pytest.mark.parametrize("case", RANGE_CASES, ids=lambda c: "h%dkv%d_p%d_n%d_m%d" % (*c[:3], len(c[3]), c[4]))
def test_ragged_decode_ranges(gpu_runner, case):
    """Auto decode of ragged batches, paged and packed, on a workspace full of
    NaN: within the reference bar (0.01 + 0.01 |ref|, LSE 2e-4) of the same
    call with an explicit chunk count and close to it relative to each
    sequence's own size, rows without a key O = 0 and LSE = -inf, nothing
    written past O, LSE and the workspace.  Two query heads of the first and of
    the last K/V head against the FP64 oracle."""
    import torch
    h, kvh, ps, lens, causal = case
    q, k, v, kc, vc, cu_q, cu_k, seqlens_k, table = _build(h, kvh, ps, lens, seed=131)
    dev = torch.device("cuda:0")
    qd, kd, vd, kcd, vcd = (to_device(x, dev) for x in (q, k, v, kc, vc))
    cq, ck, sk_d, tb = (torch.from_numpy(x).to(dev) for x in (cu_q, cu_k, seqlens_k, table))
    max_q, max_k, tq = max(s for s, _ in lens), max(s for _, s in lens), len(q)
    sizes = (len(lens), h, kvh, max_q, max_k, tq, len(k))
    print(f"  ragged decode h{h} kv{kvh} n{len(lens)} causal {causal}", flush=True)
    _, _, ref, ref_lse = _out(torch, dev, tq, h, True)
    gpu_runner.call_splitkv_paged(qd, kcd, vcd, ref, ref_lse, cq, sk_d, tb, max_q, max_k, 5, total_k=len(k),
                                  causal=causal)
    for paged in (True, False):
        need = gpu_runner.splitkv_paged_workspace_size(*sizes, ps, table.shape[1], len(kc), 0, causal=causal) \
            if paged else gpu_runner.splitkv_varlen_workspace_size(*sizes, causal, 0)
        ws = torch.full((need // 4 + GUARD,), float("nan"), device=dev, dtype=torch.float32)
        for with_lse in (True, False):
            ob, lb, o, lse = _out(torch, dev, tq, h, with_lse)
            if paged:
                gpu_runner.call_splitkv_paged(qd, kcd, vcd, o, lse, cq, sk_d, tb, max_q, max_k, 0, workspace=ws,
                                              total_k=len(k), causal=causal)
            else:
                gpu_runner.call_splitkv_varlen(qd, kd, vd, o, lse, cq, ck, max_q, max_k, causal, 0, workspace=ws)
            torch.cuda.synchronize()
            assert torch.isnan(ob[tq:]).all().item() and torch.isnan(lb[h * tq if with_lse else 0:]).all().item()
            assert torch.isnan(ws[need // 4:]).all().item()
            assert ((o.float() - ref.float()).abs() <= 0.01 + 0.01 * ref.float().abs()).all().item(), (paged, with_lse)
            _check_close(o, ref, cu_q, (paged, with_lse))
            if with_lse:
                for kh in sorted({0, kvh - 1}):
                    first, n = kh * (h // kvh), min(2, h // kvh)
                    check = _check_bottom_right if causal == 2 else _check_dense
                    check(o[:, first:first + n], lse[first:first + n], q[:, first:first + n], k[:, kh:kh + 1],
                          v[:, kh:kh + 1], cu_q, cu_k, lens, n, *([paged] if causal == 2 else []))
                seen = torch.isfinite(ref_lse)
                assert torch.equal(torch.isfinite(lse), seen) and torch.isneginf(lse[~seen]).all().item()
                assert (lse[seen] - ref_lse[seen]).abs().max().item() <= 2e-4, paged
            empty = torch.isneginf(ref_lse).T
            assert (o[empty].float() == 0).all().item()


@pytest.mark.parametrize("case", RANGE_CASES, ids=lambda c: "h%dkv%d_p%d_n%d_m%d" % (*c[:3], len(c[3]), c[4]))
def test_ragged_decode_with_a_wrong_total(gpu_runner, case):
    """total_k only steers Auto: too small, too large and the most possible, it
    gives a result close to the explicit chunks' and no write past the workspace
    that the same total asks for."""
    import torch
    h, kvh, ps, lens, causal = case
    q, k, v, kc, vc, cu_q, cu_k, seqlens_k, table = _build(h, kvh, ps, lens, seed=137)
    dev = torch.device("cuda:0")
    qd, kcd, vcd = (to_device(x, dev) for x in (q, kc, vc))
    cq, sk_d, tb = (torch.from_numpy(x).to(dev) for x in (cu_q, seqlens_k, table))
    max_q, max_k, tq = max(s for s, _ in lens), max(s for _, s in lens), len(q)
    most = len(lens) * max_k
    _, _, ref, ref_lse = _out(torch, dev, tq, h, True)
    gpu_runner.call_splitkv_paged(qd, kcd, vcd, ref, ref_lse, cq, sk_d, tb, max_q, max_k, 5, total_k=len(k),
                                  causal=causal)
    for total in (0, len(k) // 7, len(k) // 2, (len(k) + most) // 2, most - 1, most):
        print(f"  ragged decode h{h} kv{kvh} n{len(lens)} total {total} of {len(k)}", flush=True)
        need = gpu_runner.splitkv_paged_workspace_size(len(lens), h, kvh, max_q, max_k, tq, total, ps, table.shape[1],
                                                       len(kc), 0, causal=causal)
        ws = torch.full((need // 4 + GUARD,), float("nan"), device=dev, dtype=torch.float32)
        ob, lb, o, lse = _out(torch, dev, tq, h, True)
        gpu_runner.call_splitkv_paged(qd, kcd, vcd, o, lse, cq, sk_d, tb, max_q, max_k, 0, workspace=ws[:need // 4],
                                      total_k=total, causal=causal)
        torch.cuda.synchronize()
        for guard in (ob[tq:], lb[h * tq:], ws[need // 4:]):
            assert torch.isnan(guard).all().item(), total
        _check_close(o, ref, cu_q, total)
        seen = torch.isfinite(ref_lse)
        assert torch.equal(torch.isfinite(lse), seen)
        assert (lse[seen] - ref_lse[seen]).abs().max().item() <= 2e-4, total


def test_paged_decode_keeps_64_tiles_a_chunk(gpu_runner):
    """Equal lengths whose resident workgroups would take more than 64 key tiles
    a chunk (B32 H8 Sk10208, 319 tiles, page 32: three chunks): Auto keeps to
    64, a chunk's page numbers in a wave's lanes, and is bitwise five chunks."""
    import torch
    b, h, sk, ps = 32, 8, 10208, 32
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(3)
    mk = lambda *s: torch.randn(s, device=dev, dtype=torch.float32, generator=g).to(torch.bfloat16)
    q, kc, vc = mk(b, h, 128), mk(b * sk // ps, ps, h, 128), mk(b * sk // ps, ps, h, 128)
    table = torch.randperm(b * sk // ps, device=dev, generator=g).to(torch.int32).view(b, -1)
    cq = torch.arange(b + 1, device=dev, dtype=torch.int32)
    keys = torch.full((b,), sk, device=dev, dtype=torch.int32)
    outs = []
    for splits in (0, 5):
        o = torch.full_like(q, float("nan"))
        lse = torch.full((h, b), float("nan"), device=dev, dtype=torch.float32)
        gpu_runner.call_splitkv_paged(q, kc, vc, o, lse, cq, keys, table, 1, sk, splits, total_k=b * sk)
        torch.cuda.synchronize()
        outs.append((o.view(torch.int16), lse.view(torch.int32)))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    rows = [0, 17, 31]
    pick = lambda c: to_host_bits(c[table[rows].long()].reshape(len(rows), sk, h, 128))
    ref, ref_lse = orc.attention_fp64(to_host_bits(q[rows])[:, None], pick(kc), pick(vc), orc.DEFAULT_SCALE, False)
    got = to_host_bits(outs[0][0].view(torch.bfloat16)[rows])[:, None]
    e = orc.errors(got, outs[0][1].view(torch.float32)[:, rows].T.cpu().numpy()[:, :, None], ref, ref_lse)
    assert orc.check_acceptance_tolerance(e) and orc.check_reference_tolerance(e), e


def _prefill_tile(h, lens, br, splits, cus=256):
    """The q tile (128 or 256 rows) that an explicit chunk count of a paged
    prefill runs with, from the library's cost model."""
    n, max_q, max_k = len(lens), max(s for s, _ in lens), max(s for _, s in lens)
    total_q, total_k, ktiles = sum(s for s, _ in lens), sum(s for _, s in lens), -(-max_k // 64)
    tps = min(64, -(-ktiles // min(splits, ktiles)))
    mean_q, mean_k = total_q / n, total_k / n
    uniform = 4 * mean_k >= 3 * max_k
    mean = max(1.0, mean_k / 64 + 0.5 - (0.5 * mean_q / 64 if br else 0.0))

    def predict(bm):
        slots = cus if bm == 256 else 2 * cus
        qtiles = h * n * min(-(-max_q // bm), max(1.0, mean_q / bm + 0.5))
        chunks = max(1.0, np.ceil(mean / tps - 0.25) if uniform else mean / tps + 0.4)
        items, rounds = qtiles * chunks, qtiles * chunks / slots
        alone = 1.1 if bm == 128 else 1.0 if max_q <= 128 else 1.45
        shared = bm == 128 and items > cus
        per_tile = 1.5 if shared else alone
        chunk = 7 + per_tile * min(tps, mean)
        if rounds <= 1:
            t = 7 + (chunk - 7) * (1.1 if shared else 1.0)
        elif uniform:
            t = chunk * (2.0 if rounds <= 2.02 else rounds + 0.5)
        else:
            t = qtiles * (chunks * 7 + per_tile * mean) / slots + 0.2 * (7 + per_tile * min(tps, ktiles))
        return max(t, 7 + alone * min(tps, ktiles))

    return 256 if predict(256) <= predict(128) else 128


# (heads, kv_heads, page_size, [(sq, sk), ...], {chunk count: q tile}): both
# tiles with several q tiles a sequence, more queries than keys, sequences
# without keys or queries, q tiles of one chunk beside merged ones; one and four
# sequences a lane in the sorted lists, and more than those hold.
TILE_CASES = [
    (8, 2, 64, [(512, 1500), (512, 900), (512, 40), (512, 512), (0, 100), (512, 0), (500, 700), (257, 1400)],
     {1: 128, 2: 128, 3: 256, 5: 256}),
] + [(4, 2, 64, [(200 + 37 * i % 57 if i % 9 else 0, 1 + 61 * i % 500 if i % 7 else 0) for i in range(n)], tiles)
     for n, tiles in ((64, {1: 128, 3: 256}), (65, {1: 128, 3: 256}), (255, {2: 256}), (256, {2: 256}), (257, {2: 256}))
] + [(4, 2, 64, [(1 + 37 * i % 140, 1 + 61 * i % 500) for i in range(n)], {2: 128}) for n in (65, 256)]


@pytest.mark.parametrize("case", TILE_CASES, ids=lambda c: "h%dkv%d_n%d" % (c[0], c[1], len(c[3])))
def test_prefill_tiles(gpu_runner, case):
    """Paged prefill, dense and bottom-right, with the q tile that the chunk
    count takes, against the FP64 oracle."""
    import torch
    h, kvh, ps, lens, tiles = case
    q, k, v, kc, vc, cu_q, cu_k, seqlens_k, table = _build(h, kvh, ps, lens, seed=151)
    dev = torch.device("cuda:0")
    qd, kcd, vcd = (to_device(x, dev) for x in (q, kc, vc))
    cq, sk_d, tb = (torch.from_numpy(x).to(dev) for x in (cu_q, seqlens_k, table))
    max_q, max_k, tq = max(s for s, _ in lens), max(s for _, s in lens), len(q)
    for splits, tile in tiles.items():
        for causal in (2, 0):
            print(f"  prefill tiles h{h} kv{kvh} n{len(lens)} splits {splits} causal {causal}", flush=True)
            if causal:
                assert _prefill_tile(h, lens, True, splits) == tile, splits
            ob, lb, o, lse = _out(torch, dev, tq, h, True)
            gpu_runner.call_splitkv_paged(qd, kcd, vcd, o, lse, cq, sk_d, tb, max_q, max_k, splits, total_k=len(k),
                                          causal=causal)
            torch.cuda.synchronize()
            assert torch.isnan(ob[tq:]).all().item() and torch.isnan(lb[h * tq:]).all().item()
            if causal:
                _check_bottom_right(o, lse, q, k, v, cu_q, cu_k, lens, h // kvh, splits)
            else:
                _check_dense(o, lse, q, k, v, cu_q, cu_k, lens, h // kvh)
