"""The prefill route's scratch where the device has no room for the staged
kernels' operand images: the call falls back to the unstaged kernel's scratch
(none for a whole prompt, the partials of a split over keys for a chunk)."""

from __future__ import annotations

import pytest
import torch

from kvint4 import _native as nat
from kvint4 import ops


@pytest.mark.parametrize("Sq,Sk", [(16384, 16384), (512, 4096), (64, 1024)])
def test_no_room_for_images_takes_the_unstaged_scratch(monkeypatch, Sq, Sk):
    q = torch.empty(1, 32, Sq, 128, dtype=torch.bfloat16, device="meta")
    staged = nat.lib().kvq_prefill_attn_staged_workspace_bytes(1, 32, 8, Sq, 128, Sk)
    unstaged = nat.lib().kvq_prefill_attn_workspace_bytes(1, 32, 8, Sq, 128, Sk)
    real, asked = torch.empty, []

    def empty(n, dtype, device):
        asked.append(n)
        if staged != unstaged and n == staged:
            raise torch.cuda.OutOfMemoryError("no room")
        return real(n, dtype=dtype)

    monkeypatch.setattr(ops.torch, "empty", empty)
    ws, ptr, n = ops._prefill_ws(q, 8, Sk)
    assert n == unstaged and asked[0] == staged
    assert (ws is None and ptr is None) if n == 0 else (ws.numel() == n and ptr == ws.data_ptr())


@pytest.mark.parametrize("units,rows,Sk,D,staged", [
    (8, 2048, 1024, 128, True),       # 2^24 of units x rows x keys
    (8, 2047, 1024, 128, False),
    (31, 256, 4096, 128, True),       # 256 rows, 512 at D = 64
    (64, 255, 4096, 128, False),
    (32, 512, 4096, 64, True),
    (64, 511, 4096, 64, False),
    (32, 4096, 1023, 128, False),     # 1024 keys ...
    (32, 8192, 1023, 128, True),      # ... or 8192 rows
    (32, 8192, 511, 64, False),
    (127, 512, 2048, 128, True),      # a full device of the unstaged kernel's 256-row blocks: from 1024 rows
    (128, 512, 2048, 128, False),
    (128, 1024, 2048, 128, True),
    (32, 256, 4096, 128, False),      # 64 MiB of images: from 512 rows
    (32, 512, 4096, 128, True),
    (40, 2047, 16448, 128, False),    # more than 256 MiB: from 2048 rows, 1024 at D = 64
    (40, 2048, 16448, 128, True),
    (80, 1023, 16448, 64, False),
    (80, 1024, 16448, 64, True),
    (75, 1024, 1024, 64, False),      # 300 workgroups on 256 CUs
    (80, 1024, 1024, 64, True),       # 320: the second round a quarter full
])
def test_where_staging_pays(units, rows, Sk, D, staged):
    """Both sides of each line of the staged route's rule, as the workspace sizes show them."""
    shape = (units, 1, 1, rows, D, Sk)
    got = nat.lib().kvq_prefill_attn_staged_workspace_bytes(*shape) != nat.lib().kvq_prefill_attn_workspace_bytes(*shape)
    assert got == staged
