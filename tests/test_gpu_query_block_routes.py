"""Query blocks of a batch on both sides of the lines at which units x rows x keys sends them to the prefill kernel
instead of the fused decode kernel: either route meets the float64 oracle's bar (2e-2), on the contiguous and the paged
cache, and the rule never takes a block away from the prefill kernel that a single unit's rows and keys already give it."""

from __future__ import annotations

import pytest
import torch

from kvint4 import ops
from kvint4.paged_cache import PagedQuantizedKVCache


def test_rule_only_adds():
    for rows in (1, 31, 32, 47, 48, 63, 64, 100, 1024, 70000):
        for Sk in (0, 64, 1000, 4096, 16384, 65536):
            for units in (1, 8, 128):
                got = ops.use_prefill_kernel(rows, Sk, units)
                assert got or not ops.use_prefill_kernel(rows, Sk)
                assert not got or rows >= 32


def _want(q, cache, G, n_kv):
    """float64 attention over the cache's dequantized rows, causal from the bottom right."""
    kp, ks, vp, vs = cache

    def deq(p, s):
        n = torch.stack((p & 15, p >> 4), -1).flatten(-2).double() - 8
        return n * s.double().repeat_interleave(G, -1)

    k, v = deq(kp, ks), deq(vp, vs)
    B, Hq, Sq, D = q.shape
    Sk = k.shape[2]
    lim = Sk - Sq + torch.arange(Sq, device=q.device)[:, None]
    mask = torch.arange(Sk, device=q.device)[None] > lim
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for b in range(B):
        for h in range(Hq):
            s = q[b, h].double() @ k[b, h * n_kv // Hq].T.contiguous() * D ** -0.5
            out[b, h] = torch.softmax(s.masked_fill(mask, float("-inf")), -1) @ v[b, h * n_kv // Hq]
    return out


CASES = [
    # B, Hq, Hkv, Sq, Sk, D, dtype, prefill route
    (4, 8, 2, 16, 8192, 128, torch.bfloat16, True),    # 64 rows: 2^22 exactly
    (4, 8, 2, 16, 8191, 128, torch.bfloat16, False),   # one key short of it
    (8, 12, 12, 47, 1100, 64, torch.float16, False),   # 47 rows: the line is 2^24
    (8, 12, 12, 48, 1100, 64, torch.float16, True),    # 48 rows: past 2^22
    (4, 8, 8, 32, 16384, 64, torch.bfloat16, True),    # 32 rows: 2^24 exactly
    (4, 8, 8, 31, 17000, 64, torch.bfloat16, False),   # 31 rows: past 2^24, never
]


@pytest.mark.gpu
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,dtype,prefill", CASES)
def test_blocks_at_the_lines(monkeypatch, B, Hq, Hkv, Sq, Sk, D, dtype, prefill, paged):
    dev, G = torch.device("cuda:0"), 32
    g = torch.Generator(device=dev).manual_seed(Sk + Sq)
    q, k, v = (torch.randn(B, h, s, D, generator=g, device=dev).to(dtype) for h, s in ((Hq, Sq), (Hkv, Sk), (Hkv, Sk)))
    dense = (*ops.quantize(k, G, dtype), *ops.quantize(v, G, dtype))
    taken = []
    for name in ("prefill_attention", "prefill_attention_paged"):
        real = getattr(ops, name)
        monkeypatch.setattr(ops, name, lambda *a, _f=real, **kw: (taken.append(1), _f(*a, **kw))[1])
    kw = dict(n_kv_heads=Hkv, group_size=G, is_causal=True, sm_scale=D ** -0.5)
    if paged:
        cache = PagedQuantizedKVCache(group_size=G, page_size=128)
        cache.append(k, v, 0)
        out = cache.attend(q, 0, n_kv_heads=Hkv, is_causal=True, scale=D ** -0.5)
    else:
        out = ops.attention_over_quantized(q, *dense, **kw)
    assert bool(taken) == prefill
    assert (out.double() - _want(q, dense, G, Hkv)).abs().max().item() <= 2e-2
