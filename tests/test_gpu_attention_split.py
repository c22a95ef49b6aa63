"""The 16-bit forward split along the keys (calls of fewer work items than compute units) against
the f64 oracle: segments that divide the key tiles unevenly, query tiles of one segment beside
tiles of several, rows that see no key, windows, key padding, cross lengths, a batch, packed
sequences, and few queries against many keys; and the same call in one piece, through the C ABI
without a workspace. Bounds as test_gpu_attention_sweep.py."""
import ctypes

import numpy as np
import pytest
import torch

import dashmag_amd as dm
import oracle
from conformance import BF16, F16
from dashmag_amd import _lib, ops
from fixtures import errors
from test_gpu_attention_sweep import U, _build, host

pytestmark = pytest.mark.gpu

# (name, B, Tq, Tk, Hq, Hkv, mask spec, causal, window, scale)
CASES = [
    ("causal_1300", 1, 1300, 1300, 2, 1, None, True, None, None),
    ("none_16x3000", 1, 16, 3000, 4, 2, None, False, None, None),
    ("causal_cross_700x2100_b2", 2, 700, 2100, 2, 1, None, True, None, 0.2),
    ("causal_empty_rows_1800x1500", 1, 1800, 1500, 2, 2, None, True, None, None),
    ("window_1800", 1, 1800, 1800, 2, 1, None, True, (1000, U), None),
    ("padding_1700_b3", 3, 1700, 1700, 1, 1, "padding", False, None, None),
    ("packed_3200", 1, None, None, 2, 1, ("packed", [3000, 200], [3000, 200], 30), True, None,
     None),
    ("packed_1900_1300", 1, None, None, 2, 1, ("packed", [1900, 1300], [1900, 1300], 0), True, None, None),
    ("packed_200_2300_window", 1, None, None, 2, 1, ("packed", [200, 2300], [300, 2500], 0), True, (1500, U), None),
]


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.bfloat16, 128), (torch.float16, 128),
                                     (torch.bfloat16, 256)])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_split_matches_oracle(case, dtype, d):
    print(f"case {case[0]} {dtype} D={d}", flush=True)
    (q, k, v, _), mask, opts, mk = _build(case, dtype, d, 9000 + 17 * CASES.index(case) + d)
    desc = ops._attention_desc("attention", q, k, v, mask, opts, keep := [])
    lib = _lib.lib()
    assert lib.dm_attention_fwd_workspace(ctypes.byref(desc)) > 0, "the call is not split"
    _lib.probe_reset()
    o, lse = dm.attention_with_lse(q, k, v, mask, opts)
    o1, lse1 = torch.empty_like(o), torch.empty_like(lse)
    rc = lib.dm_attention_fwd(ctypes.byref(desc), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                              o1.data_ptr(), lse1.data_ptr(), None, 0,
                              torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    torch.cuda.synchronize()
    assert _lib.probe_counts()["attn_fwd_mfma"] == 2
    eo, el = oracle.attention_fwd(mk(host(q), host(k), host(v)), "f64")
    bounds = (BF16 if dtype == torch.bfloat16 else F16).masks
    for go, gl in ((o, lse), (o1, lse1)):
        ro, rl = errors(host(go), eo)[1], errors(host(gl), el)[1]
        print(f"  o {ro:.2e} lse {rl:.2e}")
        assert ro <= 2 * bounds[0] and rl <= 2 * bounds[1] * max(1.0, np.sqrt(k.shape[1] / 64))
        assert np.all(host(go)[el == -np.inf] == 0.0)


def test_more_than_two_workgroups_a_unit():
    """759 workgroups, taken in rounds: the results of the whole call, each within its bound of the exact
    ones."""
    d, hq, tq, tk = 64, 11, 1800, 9000
    q, k, v = (torch.randn(1, t, h, d, device="cuda", dtype=torch.bfloat16, generator=torch.Generator("cuda").manual_seed(t + h))
               for t, h in ((tq, hq), (tk, 1), (tk, 1)))
    opts = dm.AttentionOptions(causal=True)
    desc = ops._attention_desc("attention", q, k, v, dm.AttentionMask.none(), opts, [])
    lib = _lib.lib()
    assert lib.dm_attention_fwd_workspace(ctypes.byref(desc)) > 512 * 256 * (4 * d + 8)
    o, lse = dm.attention_with_lse(q, k, v, None, opts)
    o1, lse1 = torch.empty_like(o), torch.empty_like(lse)
    assert lib.dm_attention_fwd(ctypes.byref(desc), q.data_ptr(), k.data_ptr(), v.data_ptr(), o1.data_ptr(),
                                lse1.data_ptr(), None, 0, torch.cuda.current_stream().cuda_stream) == 0
    assert errors(host(o), host(o1))[1] <= 4 * BF16.masks[0]
    assert errors(host(lse), host(lse1))[1] <= 4 * BF16.masks[1] * np.sqrt(tk / 64)


# (name, B, Tq, Tk, Hq, Hkv, mask spec, causal, window, scale): at width 64, calls of work items
# enough for two workgroups a compute unit (768, or 257 of one length), whole
PAIRED = [
    ("causal_768", 96, 70, 200, 8, 4, None, True, None, None),
    ("window_768", 48, 300, 300, 8, 2, None, True, (100, U), 0.1),
    ("padding_768", 96, 90, 130, 8, 1, "padding", False, None, None),  # (three rounds: one at a time)
    ("padding_1024", 128, 90, 130, 8, 1, "padding", True, None, None),
    ("padding_equal_272", 17, 70, 500, 16, 2, "padding", False, None, None),
    ("equal_272", 17, 70, 500, 16, 2, None, False, None, None),
    ("packed_768", 1, None, None, 256, 16, ("packed", [300, 40, 260], [300, 90, 260], 5), True, None, None),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", PAIRED, ids=[c[0] for c in PAIRED])
def test_paired_workgroups_match_oracle(case, dtype):
    print(f"case {case[0]} {dtype}", flush=True)
    (q, k, v, _), mask, opts, mk = _build(case, dtype, 64, 9900 + 17 * PAIRED.index(case))
    desc = ops._attention_desc("attention", q, k, v, mask, opts, [])
    items = -(-q.shape[1] // 256) * q.shape[0] * q.shape[2]
    assert items >= 768 or ("equal" in case[0] and items > 256)
    assert _lib.lib().dm_attention_fwd_workspace(ctypes.byref(desc)) == 0, "the call is split"
    _lib.probe_reset()
    o, lse = dm.attention_with_lse(q, k, v, mask, opts)
    torch.cuda.synchronize()
    assert _lib.probe_counts()["attn_fwd_mfma"] == 1
    eo, el = oracle.attention_fwd(mk(host(q), host(k), host(v)), "f64")
    bounds = (BF16 if dtype == torch.bfloat16 else F16).masks
    ro, rl = errors(host(o), eo)[1], errors(host(lse), el)[1]
    print(f"  o {ro:.2e} lse {rl:.2e}")
    assert ro <= 2 * bounds[0] and rl <= 2 * bounds[1] * max(1.0, np.sqrt(k.shape[1] / 64))
    assert np.all(host(o)[el == -np.inf] == 0.0)
