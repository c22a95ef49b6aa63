"""Offsets and lengths that already lie on the GPU as int32 are read where they are, and refused
like any others before anything is launched."""
import pytest
import torch

import dashmag_amd as dm
from dashmag_amd import _lib
from dashmag_amd.contract import Unsupported

pytestmark = pytest.mark.gpu


def i32(*x):
    return torch.tensor(x, dtype=torch.int32, device="cuda")


def _calls():
    q = torch.zeros(1, 10, 2, 64, device="cuda", dtype=torch.bfloat16)
    g = torch.zeros(1, 10, 2, device="cuda")
    one = torch.zeros(2, 2, 64, device="cuda", dtype=torch.bfloat16)
    x, w = torch.zeros(1, 10, 16, device="cuda"), torch.zeros(16, 4, device="cuda")
    cache = torch.zeros(2, 5, 2, 64, device="cuda", dtype=torch.bfloat16)
    lse = torch.zeros(1, 10, 2, device="cuda")
    row, gate = torch.zeros(10, 2, 64, device="cuda", dtype=torch.bfloat16), torch.zeros(10, 2, device="cuda")
    state = torch.zeros(2, 2, 64, 64, device="cuda")
    return {
        "attention": lambda cu: dm.attention(q, q, q, dm.AttentionMask.packed(cu, cu)),
        "attention_k": lambda cu: dm.attention(q, q, q, dm.AttentionMask.packed(i32(0, 4, 10), cu)),
        "chunk": lambda cu: dm.chunk_gated_delta_rule(q, q, q, g, g, None, cu),
        "conv1d": lambda cu: dm.causal_conv1d(x, w, cu_seqlens=cu),
        "attention backward": lambda cu: dm.attention_backward(q, q, q, q, lse, q, dm.AttentionMask.packed(cu, cu)),
        "chunk backward": lambda cu: dm.chunk_gated_delta_rule_backward(q, q, q, g, g, None, cu, q),
        "conv1d backward": lambda cu: dm.causal_conv1d_backward(x, w, None, None, cu, x),
        "step": lambda cu: dm.gated_delta_step(row, row, row, gate, gate, state, cu),
        "step backward": lambda cu: dm.gated_delta_step_backward(row, row, row, gate, gate, state, cu, row, state),
        "packed decode": lambda cu: dm.attention_decode_packed(one, q[0], q[0], cu),
        "decode": lambda n: dm.attention_decode(one, cache, cache, n),
        "paged decode": lambda n: dm.attention_decode_paged(one, cache, cache, i32(0, 1).reshape(2, 1), n),
    }


@pytest.mark.parametrize("name", ["attention", "attention_k", "chunk", "conv1d", "packed decode",
                                  "decode", "paged decode", "attention backward", "chunk backward",
                                  "conv1d backward", "step", "step backward"])
def test_refused_before_any_launch(name):
    call = _calls()[name]
    bad = [i32(3, -1)] if "decode" in name and "packed" not in name else [i32(0, 11, 10), i32(0, 4, 11)]
    for value in bad:
        _lib.probe_reset()
        with pytest.raises(Unsupported):
            call(value)
        assert not any(_lib.probe_counts().values())
    call(i32(3, 0) if len(bad) == 1 else i32(0, 4, 10))
    assert any(_lib.probe_counts().values())
