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
