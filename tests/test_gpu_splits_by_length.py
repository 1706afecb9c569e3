"""GPU parity: decode attention whose splits are dealt to the sequences of a
batch by their device lengths (KVQ_SPLIT_BY_LENGTH, for batches of 2 to 64
sequences over large caches, where the caller asks for it) against the same
launch with equal splits per sequence and against float64 attention.

Both plans run the same tile code and differ in where a sequence is cut and
in the merge's order: outputs agree within two bf16 / fp16 roundings of the
output (2e-2 is the repository's bar; outputs here average hundreds of random
values, so 4e-3 is asked, and 2e-2 where a sequence has few keys). Codes and
scales that a step appends are equal byte for byte. Replayed in a HIP graph
with lengths that change between replays, the launch follows them.

Lengths: one long among short ones, all alike, zero, one, around a split's
256-key minimum, negative and past the capacity (nothing written), batches of
2, 7, 33 and 64, GQA 1, 4 and 8, both types, pages with a missing block.
"""

from __future__ import annotations

import pytest
import torch

from kvint4 import _native as nat
from kvint4 import ops

DEV = torch.device("cuda:0")
BY_LENGTH = 1 << 30  # KVQ_SPLIT_BY_LENGTH
TDT = {"bf16": torch.bfloat16, "f16": torch.float16}


def _dequant64(p, s, G):
    n = torch.stack((p & 15, p >> 4), -1).flatten(-2).double() - 8
    return n * s.double().repeat_interleave(G, -1)


def _want(q, k, v, n, scale):
    """One sequence: q [Hq, D], k and v [Hkv, S, D] float64, its first n keys."""
    r = q.shape[0] // k.shape[0]
    out = torch.zeros(q.shape, dtype=torch.float64, device=q.device)
    if n > 0:
        for h in range(q.shape[0]):
            p = torch.softmax(k[h // r, :n] @ q[h].double() * scale, 0)
            out[h] = p @ v[h // r, :n]
    return out


def _cache(B, Hkv, cap, G, dtype, g):
    out = []
    for _ in range(2):
        p, s = ops.quantize(torch.randn(B, Hkv, cap, 128, generator=g, device=DEV).to(TDT[dtype]), G, TDT[dtype])
        out += [p, s]
    return out


def _lengths(kind, B, cap, g):
    if kind == "equal":
        return torch.full((B,), cap - 5, dtype=torch.int32, device=DEV)
    if kind == "one_long":
        lens = torch.randint(1, 200, (B,), generator=g, device=DEV, dtype=torch.int32)
        lens[B // 2] = cap - 1
        return lens
    lens = (cap ** torch.rand(B, generator=g, device=DEV)).int()
    odd = [0, 1, 255, 256, 257, -3, cap, cap + 9][:B - 1]
    lens[: len(odd)] = torch.tensor(odd, dtype=torch.int32, device=DEV)
    return lens


CASES = [(2, 32, 8, 4096, "one_long", "bf16", 32), (7, 8, 8, 4100, "mixed", "f16", 64), (33, 32, 8, 4500, "mixed", "bf16", 32),
         (64, 64, 8, 4096, "one_long", "bf16", 128), (12, 64, 8, 5000, "equal", "f16", 32), (20, 16, 4, 5000, "mixed", "bf16", 32)]


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,cap,kind,dtype,G", CASES)
def test_step_and_attention_by_length(B, Hq, Hkv, cap, kind, dtype, G):
    g = torch.Generator(device=DEV).manual_seed(B * cap)
    t = TDT[dtype]
    code = nat.DTYPE_CODE[t]  # the shape has such a plan (of any size, from 64K rows on)
    assert nat.lib().kvq_decode_attn_by_length_workspace_bytes(B, Hq, Hkv, 1, 128, 65536, code, code) > 0
    bufs = _cache(B, Hkv, cap, G, dtype, g)
    lens = _lengths(kind, B, cap, g)
    q = torch.randn(B, Hq, 1, 128, generator=g, device=DEV).to(t)
    kn, vn = (torch.randn(B, Hkv, 1, 128, generator=g, device=DEV).to(t) for _ in range(2))
    kw = dict(n_kv_heads=Hkv, group_size=G, sm_scale=128 ** -0.5)
    # attention over the cached rows
    a = ops.fused_decode_attention(q, *bufs, is_causal=False, seq_lens=lens, n_split=BY_LENGTH, **kw)
    b = ops.fused_decode_attention(q, *bufs, is_causal=False, seq_lens=lens, n_split=2, **kw)
    # the step, on its own copy of the cache
    one, two = [x.clone() for x in bufs], [x.clone() for x in bufs]
    sa = ops.decode_step(q, kn, vn, *one, lens, n_split=BY_LENGTH, **kw)
    sb = ops.decode_step(q, kn, vn, *two, lens, n_split=2, **kw)
    for x, y in zip(one, two):
        assert torch.equal(x, y)
    k64, v64 = _dequant64(one[0], one[1], G), _dequant64(one[2], one[3], G)
    for i, n in enumerate(lens.tolist()):
        bar = 4e-3 if n >= 200 else 2e-2
        assert (a[i].float() - b[i].float()).abs().max().item() <= bar, (i, n)
        assert (sa[i].float() - sb[i].float()).abs().max().item() <= bar, (i, n)
        m = min(max(n, 0), cap)
        assert (a[i, :, 0].double() - _want(q[i, :, 0], k64[i], v64[i], m, 128 ** -0.5)).abs().max().item() <= 2e-2
        m = m + 1 if 0 <= n < cap else m
        assert (sa[i, :, 0].double() - _want(q[i, :, 0], k64[i], v64[i], m, 128 ** -0.5)).abs().max().item() <= 2e-2


@pytest.mark.gpu
def test_paged_step_by_length_and_graph_replays():
    """A paged batch: equal to the equal-splits plan; then captured, and replayed while the lengths change."""
    B, Hq, Hkv, P, cols, G = 6, 32, 8, 64, 64, 32
    g = torch.Generator(device=DEV).manual_seed(4)
    nb = B * cols + 1
    pools = [x[0] for x in _cache(1, Hkv, nb * P, G, "bf16", g)]
    table = torch.randperm(nb, generator=torch.Generator().manual_seed(1))[: B * cols].view(B, cols).to(DEV, torch.int32)
    table[4, 7] = -1  # sequence 4 ends before that page
    pt = ops.PageTable(table, P, nb)
    lens = torch.tensor([2500, 3, 700, 0, 447, 64], dtype=torch.int32, device=DEV)
    q = torch.randn(B, Hq, 1, 128, generator=g, device=DEV).bfloat16()
    kn, vn = (torch.randn(B, Hkv, 1, 128, generator=g, device=DEV).bfloat16() for _ in range(2))
    kw = dict(n_kv_heads=Hkv, group_size=G, sm_scale=128 ** -0.5)

    def both():
        one, two = [x.clone() for x in pools], [x.clone() for x in pools]
        a = ops.decode_step_paged(q, kn, vn, *one, pt, lens, n_split=BY_LENGTH, **kw)
        b = ops.decode_step_paged(q, kn, vn, *two, pt, lens, n_split=2, **kw)
        for x, y in zip(one, two):
            assert torch.equal(x, y)
        assert (a.float() - b.float()).abs().max().item() <= 2e-2
        return a

    both()
    out, own = torch.empty_like(q), [x.clone() for x in pools]
    ws = torch.zeros(ops.decode_workspace_bytes(B, Hq, Hkv, 128, q.dtype, q.dtype), dtype=torch.uint8, device=DEV)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with ops.using_workspace(ws):
        with torch.cuda.graph(graph, stream=side):
            ops.decode_step_paged(q, kn, vn, *own, pt, lens, out=out, n_split=BY_LENGTH, **kw)
    for new in ([2500, 3, 700, 0, 447, 64], [10, 2000, 1, 300, 64, 2559], [5, 5, 5, 5, 5, 5], [2500, 3, 700, 0, 447, 64]):
        lens.copy_(torch.tensor(new, dtype=torch.int32))
        for x, y in zip(own, pools):
            x.copy_(y)
        graph.replay()
        torch.cuda.synchronize()
        if new[4] < 448:  # with the missing page's keys in range, the two plans still agree
            assert torch.equal(out, both())


@pytest.mark.gpu
def test_plan_rule_and_workspace_bound():
    """Which calls are planned by length, and that a workspace sized for 64 equal splits covers them."""
    lib, bf = nat.lib(), nat.KVQ_BF16

    def plan(B, s_max, Hq=32, Hkv=8, Sq=1, D=128, qd=bf, sd=bf):
        return lib.kvq_decode_attn_by_length_workspace_bytes(B, Hq, Hkv, Sq, D, s_max, qd, sd)

    assert plan(8, 8192) > 0 and plan(16, 4096) > 0 and plan(4, 16384) > 0 and plan(32, 8192) > 0
    assert plan(1, 1 << 20) == 0 and plan(65, 16384) == 0 and plan(8, 4096) == 0 and plan(32, 4096) == 0
    assert plan(8, 8192, Sq=2) == 0 and plan(8, 8192, D=64) == 0 and plan(8, 8192, qd=nat.KVQ_F32) == 0
    assert plan(8, 8192, sd=nat.KVQ_F16) == 0
    for B in (2, 3, 8, 20, 33, 64):
        for Hq, Hkv in ((32, 8), (8, 1), (64, 8), (4, 4), (16, 2)):
            n = plan(B, 1 << 17, Hq, Hkv)
            assert n <= lib.kvq_decode_attn_workspace_bytes(B, Hq, Hkv, 1, 128, bf, bf, 64)


@pytest.mark.gpu
def test_workspace_of_the_equal_splits_is_still_enough():
    """A workspace that the caller sized for the library's equal splits: the
    call takes them, with the bytes of by_length = False."""
    B, Hq, Hkv, cap, G = 32, 32, 8, 8192, 32
    g = torch.Generator(device=DEV).manual_seed(32)
    n = nat.lib().kvq_decode_attn_num_splits(B, Hq, Hkv, 1, 128, cap, nat.KVQ_BF16, nat.KVQ_BF16, ops._num_cus(DEV))
    size = ops.decode_workspace_bytes(B, Hq, Hkv, 128, torch.bfloat16, torch.bfloat16, n_split=n)
    assert size < nat.lib().kvq_decode_attn_by_length_workspace_bytes(B, Hq, Hkv, 1, 128, cap, nat.KVQ_BF16, nat.KVQ_BF16)
    cache = _cache(B, Hkv, cap, G, "bf16", g)
    pos = _lengths("mixed", B, cap - 10, g).clamp(min=0)
    q = torch.randn(B, Hq, 1, 128, generator=g, device=DEV).bfloat16()
    k, v = (torch.randn(B, Hkv, 1, 128, generator=g, device=DEV).bfloat16() for _ in range(2))
    kw = dict(n_kv_heads=Hkv, group_size=G, sm_scale=0.0884)
    want = ops.decode_step(q, k, v, *cache, pos, by_length=False, **kw)
    with ops.using_workspace(torch.zeros(max(size, 16), dtype=torch.uint8, device=DEV)):
        got = ops.decode_step(q, k, v, *cache, pos, **kw)
    assert torch.equal(got, want)


@pytest.mark.gpu
def test_operators_split_equally_unless_asked():
    """The operators' defaults over device lengths: equal splits, whose bits they have; by_length = True takes the
    lengths' own, in every operator that has device lengths."""
    B, Hq, Hkv, cap, G, P = 6, 32, 8, 16384, 32, 128
    g = torch.Generator(device=DEV).manual_seed(17)
    bufs = _cache(B, Hkv, cap, G, "bf16", g)
    lens = _lengths("one_long", B, cap, g)
    q = torch.randn(B, Hq, 1, 128, generator=g, device=DEV).bfloat16()
    k, v = (torch.randn(B, Hkv, 1, 128, generator=g, device=DEV).bfloat16() for _ in range(2))
    kw = dict(n_kv_heads=Hkv, group_size=G, sm_scale=128 ** -0.5)
    n = nat.lib().kvq_decode_attn_num_splits(B, Hq, Hkv, 1, 128, cap, nat.KVQ_BF16, nat.KVQ_BF16, ops._num_cus(DEV))
    pools = [t.transpose(0, 1).reshape(Hkv, B * cap, -1).contiguous() for t in bufs]
    pt = ops.PageTable(torch.arange(B * cap // P, dtype=torch.int32, device=DEV).view(B, -1), P, B * cap // P)
    calls = {
        "step": lambda **o: ops.decode_step(q, k, v, *bufs, lens, **kw, **o),
        "paged step": lambda **o: ops.decode_step_paged(q, k, v, *pools, pt, lens, **kw, **o),
        "attention": lambda **o: ops.fused_decode_attention(q, *bufs, is_causal=False, seq_lens=lens, **kw, **o),
        "paged attention": lambda **o: ops.fused_decode_attention_paged(q, *pools, pt, is_causal=False, seq_lens=lens,
                                                                        **kw, **o),
    }
    for name, call in calls.items():
        equal, dealt = call(n_split=n), call(n_split=BY_LENGTH)
        assert not torch.equal(equal, dealt), name  # (the long sequence's sums are in another order)
        assert torch.equal(call(), equal), name
        assert torch.equal(call(by_length=True), dealt), name


@pytest.mark.gpu
@pytest.mark.parametrize("n_split", [(1 << 30) + 1, (1 << 31) - 1, 1 << 40])
def test_other_large_split_counts_are_equal_splits(n_split):
    """A split count past the cap means the cap, 64 equal splits; only KVQ_SPLIT_BY_LENGTH itself asks for the list."""
    B, Hq, Hkv, cap, G = 3, 32, 8, 16384, 32
    g = torch.Generator(device=DEV).manual_seed(18)
    bufs = _cache(B, Hkv, cap, G, "bf16", g)
    lens = _lengths("one_long", B, cap, g)
    q = torch.randn(B, Hq, 1, 128, generator=g, device=DEV).bfloat16()
    kw = dict(n_kv_heads=Hkv, group_size=G, sm_scale=128 ** -0.5, is_causal=False, seq_lens=lens)
    want = ops.fused_decode_attention(q, *bufs, n_split=64, **kw)
    assert torch.equal(ops.fused_decode_attention(q, *bufs, n_split=n_split, **kw), want)


def test_when_splits_by_length_pay():
    """The caches' rule: never for lengths alike, for few sequences' small spread, or where the kernel has no such
    plan; for one long sequence among short ones."""
    def pays(lens, cap, Hq=32, Hkv=8, D=128, dt=torch.bfloat16, sd=None):
        return ops.by_length_pays(len(lens), Hq, Hkv, D, dt, sd or dt, cap, sum(lens), max(lens), 256)

    for B in (1, 2, 8, 32, 64):
        for cap in (4096, 16384, 32768):
            for n in (0, 100, cap // 4, cap - 1):
                assert not pays([n] * B, cap)
    long32 = [16383] + [256] * 31
    assert pays(long32, 16384) and pays(long32, 16384, dt=torch.float16) and pays([16000] + [300] * 7, 16384)
    assert not pays(long32, 16384, D=64) and not pays(long32, 16384, dt=torch.float32)
    assert not pays(long32, 16384, sd=torch.float16)
    assert not pays([2047] + [128] * 31, 8192)          # 12.9 us equal, 19.1 by length
    assert not pays([16383, 9000] * 16, 16384)          # half as long
    assert not pays([16383] + [256] * 64, 16384)        # more sequences than the plan takes
    assert not pays(long32, 16384, Hq=4, Hkv=8)


def test_host_lengths_of_a_ragged_layer():
    from kvint4.cache_base import _lag

    assert _lag(torch.tensor([5, 9, 0]), 9) == (13, 0)
    assert _lag(torch.tensor([5, 4, -3]), 9) == (18, 4)


@pytest.mark.gpu
@pytest.mark.parametrize("paged", [False, True])
def test_caches_choose_by_their_lengths(monkeypatch, paged):
    """Caches whose host knows the lengths ask for splits by length where the rule says so, and no longer after an
    edit that leaves them unknown."""
    from kvint4.llama3.kv_cache import QuantizedKVCache
    from kvint4.paged_cache import PagedQuantizedKVCache

    B, Hkv, S, D, G = 8, 8, 16000, 128, 32
    g = torch.Generator(device=DEV).manual_seed(3)
    k, v = (torch.randn(B, Hkv, S, D, generator=g, device=DEV).bfloat16() for _ in range(2))
    q = torch.randn(B, 32, 1, D, generator=g, device=DEV).bfloat16()
    kn, vn = k[:, :, :1].contiguous(), v[:, :, :1].contiguous()
    name = "decode_step_paged" if paged else "decode_step"
    real, seen = getattr(ops, name), []
    monkeypatch.setattr(ops, name, lambda *a, **kw: (seen.append(kw["by_length"]), real(*a, **kw))[1])

    def step(cache):
        assert cache.append_and_attend(q, kn, vn, 0, n_kv_heads=Hkv, scale=D ** -0.5) is not None
        return seen[-1]

    def make(lens):
        cache = PagedQuantizedKVCache(group_size=G, page_size=128) if paged else QuantizedKVCache(group_size=G)
        cache.load_ragged(k, v, 0, lens)
        return cache

    spread = torch.tensor([S] + [300] * 7, dtype=torch.int32)
    cache = make(spread)
    assert step(cache) and step(cache)
    cache.crop(-1)
    assert step(cache)
    if paged:
        cache.crop(400)
        assert not step(cache)
    else:
        cache.crop(15990)
        assert not step(cache)
        assert not step(make(spread.to(DEV)))  # lengths that only the device knows
    assert not step(make(torch.tensor([S, S - 900] * 4, dtype=torch.int32)))
    assert not step(make(torch.full((B,), S, dtype=torch.int32)))
