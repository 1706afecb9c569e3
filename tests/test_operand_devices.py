"""No operator passes the pointer of a tensor in host memory to a kernel, where the first read would fault the GPU: the
module below the operators refuses such a tensor in every place where it takes one (CPU test)."""

from __future__ import annotations

import pytest
import torch

from kvint4 import _native as nat

# positions of the tensor arguments of each function of the host module, and its number of arguments
TENSORS = {
    "quantize": ((0, 7, 8), 14),
    "quantize_kv": ((0, 1, 8, 9, 10, 11), 17),
    "quantize_paged": ((0, 7, 8), 14),
    "quantize_kv_paged": ((0, 1, 8, 9, 10, 11), 17),
    "dequantize": ((0, 1, 8), 12),
    "dequantize_paged": ((0, 1, 9), 13),
    "decode_attn": ((0, 2, 3, 4, 5, 7), 22),
    "decode_attn_paged": ((0, 2, 3, 4, 5, 8), 23),
    "decode_step": ((0, 2, 3, 4, 5, 6, 7, 9), 23),
    "decode_step_paged": ((0, 2, 3, 4, 5, 6, 7, 10), 23),
    "prefill_attn": ((0, 2, 3, 4, 5, 7), 20),
    "prefill_attn_paged": ((0, 2, 3, 4, 5, 8), 21),
}
TABLES = {"quantize_paged": 10, "quantize_kv_paged": 13, "dequantize_paged": 3, "decode_attn_paged": 7,
          "decode_step_paged": 9, "prefill_attn_paged": 7}


@pytest.mark.parametrize("name", TENSORS)
def test_host_tensors_are_refused(name):
    places, n = TENSORS[name]
    fn, t = getattr(nat.host(), name), torch.zeros(1, 1, 1, 1)
    for at in places:
        args = [None if i in places else 0 for i in range(n)]
        if name in TABLES:
            args[TABLES[name]] = (None, 0, 0, 0, 0)
        args[at] = t
        with pytest.raises(ValueError, match="host memory"):
            fn(*args)
