"""Every operand of the attention operators is asked for its device before a native call: a host pointer that reached a
kernel would fault the GPU. (CPU: the check itself is replaced by a recorder that ends the call.)"""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from kvint4 import ops


class _Seen(Exception):
    pass


def _operands(paged):
    q = torch.zeros(1, 4, 1, 64, dtype=torch.float16)
    n = torch.zeros(1, 2, 1, 64, dtype=torch.float16)
    lead = (2, 64) if paged else (1, 2, 64)
    kv = [torch.zeros(*lead, w, dtype=t) for w, t in ((32, torch.uint8), (2, torch.float16)) * 2]
    return q, n, n.clone(), kv, torch.zeros_like(q)


@pytest.mark.parametrize("name", ["fused_decode_attention", "prefill_attention", "decode_step",
                                  "fused_decode_attention_paged", "prefill_attention_paged", "decode_step_paged"])
def test_every_operand_is_checked(monkeypatch, name):
    paged = name.endswith("paged")
    q, kn, vn, kv, out = _operands(paged)
    seen = []

    def check(*ts, what):
        seen.extend(ts)
        raise _Seen

    kw = dict(n_kv_heads=2, group_size=32, sm_scale=0.1, out=out)
    # (a PageTable refuses a host table by itself)
    table = SimpleNamespace(table=torch.zeros(1, 1, dtype=torch.int32), page_size=64, num_blocks=1, capacity=64)
    pt = (table,) if paged else ()
    if name.startswith("decode_step"):
        args, want = (q, kn, vn, *kv, *pt, 3), [q, kn, vn, *kv, out]
    else:
        kw["is_causal"] = True
        args = (q, *kv, *pt, *((64,) if name == "prefill_attention_paged" else ()))
        want = [q, *kv, out]
        if name == "fused_decode_attention_paged":
            kw["seq_len"] = 64
    want += [table.table] if paged else []
    monkeypatch.setattr(ops, "_check_cuda", check)
    with pytest.raises(_Seen):
        getattr(ops, name)(*args, **kw)
    for t in want:
        assert any(t is u for u in seen)


@pytest.mark.parametrize("name", ["fused_decode_attention", "prefill_attention", "decode_step"])
def test_host_tensors_are_refused(name):
    q, kn, vn, kv, _ = _operands(False)
    kw = dict(n_kv_heads=2, group_size=32, sm_scale=0.1)
    with pytest.raises(ValueError, match="GPU tensors"):
        if name == "decode_step":
            ops.decode_step(q, kn, vn, *kv, 3, **kw)
        else:
            getattr(ops, name)(q, *kv, is_causal=True, **kw)
