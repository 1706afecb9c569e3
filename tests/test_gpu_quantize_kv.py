"""GPU parity: K and V quantized in one launch (kvq_quantize_kv, contiguous
and paged) write the bytes of two kvq_quantize calls, and leave every other
byte of the destinations alone.

Strided K beside contiguous V, one tensor aligned for the vector path and the
other not, a head dim outside it for both, device positions with rows past the
capacity, both row counts per lane, an empty append, and pairs that do not
match (different dtypes or capacities), which take two launches.
"""

from __future__ import annotations

import pytest
import torch

from kvint4 import ops

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TDT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _buffers(B, H, cap, D, G, sd):
    w, ng = ops.packed_width(D, G), ops.num_groups(D, G)
    g = torch.Generator(device=DEV).manual_seed(cap)
    out = []
    for _ in range(2):
        out.append(torch.randint(0, 256, (B, H, cap, w), dtype=torch.uint8, device=DEV, generator=g))
        out.append(torch.randn(B, H, cap, ng, device=DEV, generator=g).to(sd))
    return out


def _both(k, v, bufs, G, pos):
    one, two = [t.clone() for t in bufs], [t.clone() for t in bufs]
    ops.quantize_kv_into(k, v, one[0], one[1], one[2], one[3], G, pos)
    ops.quantize_into(k, two[0], two[1], G, pos)
    ops.quantize_into(v, two[2], two[3], G, pos)
    for a, b in zip(one, two):
        assert torch.equal(a, b)


@pytest.mark.parametrize("B,H,S,D,G,dtype", [
    (1, 8, 1, 128, 32, "bf16"), (2, 12, 5, 64, 32, "f32"), (1, 3, 33, 80, 32, "f16"), (2, 2, 7, 50, 33, "bf16"),
    (1, 8, 2100, 128, 64, "bf16"), (3, 5, 1001, 128, 32, "f16"), (1, 2, 0, 128, 32, "bf16"),
])
def test_pair_equals_two_calls(B, H, S, D, G, dtype):
    g = torch.Generator(device=DEV).manual_seed(S + D)
    t = TDT[dtype]
    k = torch.randn(B, S, H, D, generator=g, device=DEV).to(t).transpose(1, 2)  # as a projection leaves it
    v = torch.randn(B, H, S, D, generator=g, device=DEV).to(t)
    bufs = _buffers(B, H, S + 9, D, G, torch.float16 if dtype == "f32" else t)
    _both(k, v, bufs, G, 4)
    odd = torch.randn(B, H, S, D + 1, generator=g, device=DEV).to(t)[..., 1:]  # not aligned for 16-byte loads
    _both(k, odd, bufs, G, 0)
    _both(odd, k, bufs, G, 0)
    pos = torch.tensor([(7 * b + 3) % 13 for b in range(B)], dtype=torch.int32, device=DEV)  # some rows past the end
    _both(k, v, bufs, G, pos)


def test_pair_mismatches_take_two_launches():
    k = torch.randn(1, 4, 6, 64, device=DEV)
    bufs = _buffers(1, 4, 16, 64, 32, torch.float16)
    _both(k, k.half(), bufs, 32, 2)
    short = _buffers(1, 4, 10, 64, 32, torch.float16)
    _both(k, k, bufs[:2] + short[2:], 32, 2)
    with pytest.raises(ValueError):
        ops.quantize_kv_into(k, k, *bufs, 32, 11)


def test_pair_paged_equals_two_calls():
    B, H, S, D, G, P = 3, 4, 150, 128, 32, 64
    g = torch.Generator(device=DEV).manual_seed(2)
    k, v = (torch.randn(B, H, S, D, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    cols, nb = 3, 12
    table = torch.randperm(nb, generator=torch.Generator().manual_seed(1))[: B * cols].view(B, cols).to(DEV, torch.int32)
    table[1, 1] = -1
    pt = ops.PageTable(table, P, nb)
    pools = [t[0] for t in _buffers(1, H, nb * P, D, G, torch.bfloat16)]
    pos = torch.tensor([0, 20, 60], dtype=torch.int32, device=DEV)
    one, two = [t.clone() for t in pools], [t.clone() for t in pools]
    ops.quantize_kv_into_paged(k, v, *one, pt, G, pos)
    ops.quantize_into_paged(k, two[0], two[1], pt, G, pos)
    ops.quantize_into_paged(v, two[2], two[3], pt, G, pos)
    for a, b in zip(one, two):
        assert torch.equal(a, b)
