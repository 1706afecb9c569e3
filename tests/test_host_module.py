"""CPU tests of the CPython module over the native library (_kvq_host):
argument counts and types are refused before any call, a null tensor reaches
the entry point's own checks, strides come from tensors or (pointer, strides)
tuples, and its plan equals the C planning functions."""

from __future__ import annotations

import pytest
import torch

from kvint4 import _native as nat


def test_argument_counts_and_types():
    h = nat.host()
    for name in ("quantize", "quantize_kv", "quantize_paged", "quantize_kv_paged", "dequantize", "dequantize_paged",
                 "plan", "decode_attn", "decode_attn_paged", "decode_step", "decode_step_paged", "prefill_attn",
                 "prefill_attn_paged"):
        with pytest.raises(TypeError):
            getattr(h, name)()
        with pytest.raises(TypeError):
            getattr(h, name)(*[1] * 40)
    x = torch.zeros(1, 1, 1, 32)
    with pytest.raises(AttributeError):  # not a tensor
        h.quantize(object(), 0, 1, 1, 1, 32, 32, None, None, 0, None, 0, 1, None)
    with pytest.raises(TypeError):       # not an integer
        h.quantize(None, 0, 1, 1, "1", 32, 32, None, None, 0, None, 0, 1, None)
    with pytest.raises(ValueError):      # too few strides
        h.quantize(x[0], 0, 1, 1, 1, 32, 32, None, None, 0, None, 0, 1, None)
    with pytest.raises(ValueError):
        h.quantize((0, (1, 1)), 0, 1, 1, 1, 32, 32, None, None, 0, None, 0, 1, None)
    with pytest.raises(ValueError):      # a table has five arguments
        h.quantize_paged(None, 0, 1, 1, 1, 32, 32, None, None, 0, (None, 1), None, 0, None)


def test_null_tensors_reach_the_entry_points_checks():
    h = nat.host()
    assert h.quantize(None, nat.KVQ_BF16, 1, 1, 1, 32, 32, None, None, nat.KVQ_BF16, None, 0, 1, None) == nat.KVQ_EINVAL
    assert "null" in nat.last_error()
    assert h.quantize(None, nat.KVQ_BF16, 1, 1, 1, 32, 0, None, None, nat.KVQ_BF16, None, 0, 1, None) == nat.KVQ_EINVAL
    assert "group_size" in nat.last_error()
    # nothing to do: no pointer is read
    assert h.quantize((None, (0, 0, 0, 1)), nat.KVQ_BF16, 0, 1, 1, 32, 32, None, None, nat.KVQ_BF16, None, 0, 1, None) == 0


@pytest.mark.parametrize("shape", [(1, 32, 8, 1, 128, 16385), (8, 64, 8, 1, 128, 32769), (2, 12, 12, 5, 64, 1024)])
def test_plan_equals_the_planning_functions(shape):
    lib = nat.lib()
    for qd, sd in ((0, 0), (1, 1), (2, 1)):
        n = lib.kvq_decode_attn_num_splits(*shape, qd, sd, 256)
        w = lib.kvq_decode_attn_workspace_bytes(*shape[:5], qd, sd, n)
        assert nat.host().plan(*shape, qd, sd, 256, 0, 0) == (n, w)
        assert nat.host().plan(*shape, qd, sd, 256, 3, 0)[0] == 3
    assert nat.host().plan(1, 3, 2, 1, 128, 10, 0, 0, 256, 0, 0)[0] == nat.KVQ_EINVAL
