"""Query blocks that the fused decode kernel takes (fewer than 64 rows per KV head, or rows x keys below the prefill
kernel's line) keep its precision whatever the batch: K and V codes stay exact there and their scales are fp32, where
the prefill kernel rounds dequantized K and V to 16 bits.

Bars, relative to the outputs' norm against float64 attention over the cache: 3e-3 for bf16 and 4e-4 for fp16. What the
fused kernel narrows is the weight p * v_scale and the output (2^-9 each in bf16, 2^-12 and 2^-12 in fp16: measured
2.0e-3 and 2.3e-4); the prefill kernel's roundings of K and V measure 6e-3 and 8.5e-4 on keys with outlier channels."""

from __future__ import annotations

import pytest
import torch

from kvint4 import ops
from kvint4.paged_cache import PagedQuantizedKVCache

BARS = {torch.bfloat16: 3e-3, torch.float16: 4e-4}


def test_more_kv_heads_than_query_heads_is_refused():
    """The library's own refusal, as for any other shape it does not take (without a GPU: that there is none)."""
    q = torch.zeros(1, 4, 8, 64, dtype=torch.float16)
    p = torch.zeros(1, 8, 16, 32, dtype=torch.uint8)
    s = torch.zeros(1, 8, 16, 2, dtype=torch.float16)
    with pytest.raises((ValueError, RuntimeError)):
        ops.attention_over_quantized(q, p, s, p, s, n_kv_heads=8, group_size=32, is_causal=True, sm_scale=0.1)


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
    # B, Hq, Hkv, Sq, Sk, D, dtype
    (1, 32, 8, 8, 8200, 128, torch.bfloat16),    # 32 rows, one sequence
    (16, 32, 8, 8, 4096, 128, torch.bfloat16),   # 32 rows, a batch
    (16, 32, 8, 12, 2100, 128, torch.float16),   # 48 rows
    (16, 32, 8, 16, 1000, 128, torch.bfloat16),  # 64 rows below the prefill kernel's rows x keys
    (8, 12, 12, 48, 1100, 64, torch.float16),    # MHA, D = 64
    (8, 12, 12, 63, 1100, 64, torch.bfloat16),
]


@pytest.mark.gpu
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,dtype", CASES)
def test_blocks_keep_the_fused_kernels_precision(B, Hq, Hkv, Sq, Sk, D, dtype, paged):
    dev, G = torch.device("cuda:0"), 32
    g = torch.Generator(device=dev).manual_seed(Sk + Sq)
    q, k, v = (torch.randn(B, h, s, D, generator=g, device=dev) for h, s in ((Hq, Sq), (Hkv, Sk), (Hkv, Sk)))
    k[..., [(5 + 13 * i) % D for i in range(8)]] *= 8.0  # outlier channels, as trained models' keys have them
    q, k, v = q.to(dtype), k.to(dtype), v.to(dtype)
    dense = (*ops.quantize(k, G, dtype), *ops.quantize(v, G, dtype))
    if paged:
        cache = PagedQuantizedKVCache(group_size=G, page_size=128)
        cache.append(k, v, 0)
        out = cache.attend(q, 0, n_kv_heads=Hkv, is_causal=True, scale=D ** -0.5)
    else:
        out = ops.attention_over_quantized(q, *dense, n_kv_heads=Hkv, group_size=G, is_causal=True, sm_scale=D ** -0.5)
    want = _want(q, dense, G, Hkv)
    err = ((out.double() - want).norm() / want.norm()).item()
    print(f"rows {Hq // Hkv * Sq} keys {Sk} batch {B} {dtype}: relative error {err:.2e}", flush=True)
    assert err <= BARS[dtype]
