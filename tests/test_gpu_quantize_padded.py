"""GPU parity: rows whose last group the head dim only partly fills, on the
vector quantize / dequantize kernels (8-element chunks; the padding's chunks
are zeros). Codes and scales equal the CPU oracle's byte
for byte, the dequantized values its narrowed products exactly.

Head dims of one chunk, one chunk short of and past a group, and several
groups; every group size the path takes; both row counts per lane (a launch
of more than 256K chunks takes four rows per lane, with a remainder); a view
with spare columns; d_head inside the last group.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from kvint4 import ops
from oracle import kvq_oracle as O

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TDT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _check(x, dtype, G, d_outs):
    D = x.shape[-1]
    p, s = ops.quantize(x, G, TDT[dtype])
    op, osc = O.quantize_int4(x.float().cpu().numpy(), G, dtype)
    assert np.array_equal(p.cpu().numpy(), op)
    assert np.array_equal(s.float().cpu().numpy(), osc)
    n = torch.stack((p & 15, p >> 4), -1).flatten(-2).float() - 8
    want = (n * s.float().repeat_interleave(G, -1)).to(TDT[dtype])
    for d in d_outs:
        got = ops.dequantize(p, s, G, d, TDT[dtype])
        assert got.shape[-1] == d and torch.equal(got, want[..., :d]), d


@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("D,G", [(8, 16), (8, 128), (24, 32), (40, 32), (56, 64), (72, 64), (80, 32), (120, 128),
                                 (136, 128), (200, 16), (88, 8)])
def test_padded_rows(D, G, dtype):
    g = torch.Generator().manual_seed(D * G)
    x = torch.randn(2, 3, 37, D, generator=g).to(TDT[dtype]).to(DEV)
    x[0, 0, 5] = 0  # all-zero groups next to the padding
    ng = -(-D // G)
    _check(x, dtype, G, sorted({D, ng * G, max(8, D - 8)}))


def test_padded_rows_four_per_lane_and_view():
    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn(3, 7, 1301, 96, generator=g, device=DEV).to(torch.bfloat16)[..., :80]
    assert 3 * 7 * 1301 * 12 > 256 * 1024 and 3 * 7 * 1301 % 4
    _check(x, "bf16", 32, [80])
