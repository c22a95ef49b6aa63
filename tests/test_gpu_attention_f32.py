"""The f32 attention kernels (f32 inputs, and 16-bit ones of widths the 16-bit MFMA kernels do not
take) against the f64 oracle over the mask kinds of test_gpu_attention_sweep.py, whose lengths cut
the 16-row tiles, at every padded width, at widths that are not multiples of 16 or of 4 (element
loads instead of 16-byte ones), and on views at odd strides.

Bounds, of the largest difference over the largest value: dash-conformance's f32 ones for the
fixtures' 40 keys (1e-6; lse 2e-7), doubled for the sums over up to 700 keys and widths up to 256,
lse's further by sqrt(Tk / 64), and not below a dot product's own rounding: D terms whose sums are of
unit size carry sqrt(D) 2^-24 (a lone key's lse is such a product, and may be small); 16-bit inputs at twice dash-conformance's 16-bit bounds."""
import numpy as np
import pytest
import torch

import dashmag_amd as dm
import oracle
from conformance import AUTOTUNE_F32, BF16, F16
from dashmag_amd import _lib, synthetic as syn
from fixtures import errors
from test_gpu_attention_sweep import CASES, PARTS, _build, host

pytestmark = pytest.mark.gpu
FEW = [c for c in CASES if c[0] in ("causal_1", "causal_127_scale", "causal_tq127_tk33_empty_rows",
                                    "window_both_300", "key_padding_causal_133", "packed_cross",
                                    "packed_tiles_tail")]
RUNS = [(torch.float32, 64, c) for c in CASES if c[0] != "causal_4097"]
RUNS += [(dt, d, c) for dt, d in ((torch.float32, 128), (torch.float32, 256), (torch.float32, 20),
                                  (torch.float32, 13), (torch.float32, 200), (torch.bfloat16, 80),
                                  (torch.float16, 200)) for c in FEW]


@pytest.mark.parametrize("dtype,d,case", RUNS, ids=[f"{r[0]}-{r[1]}-{r[2][0]}" for r in RUNS])
def test_matches_oracle(dtype, d, case):
    print(f"case {case[0]} {dtype} D={d}", flush=True)
    (q, k, v, do), mask, opts, mk = _build(case, dtype, d, 5000 + 17 * CASES.index(case) + d)
    _lib.probe_reset()
    o, lse = dm.attention_with_lse(q, k, v, mask, opts)
    dq, dk, dv = dm.attention_backward(q, k, v, o, lse, do, mask, opts)
    torch.cuda.synchronize()
    pc = _lib.probe_counts()
    assert pc["attn_fwd_generic"] > 0 and pc["attn_bwd_generic"] > 0, pc
    call = mk(host(q), host(k), host(v))
    eo, el = oracle.attention_fwd(call, "f64")
    gq, gk, gv = oracle.attention_bwd(call, host(o), host(lse), host(do), "f64")
    bounds = {torch.float32: AUTOTUNE_F32, torch.bfloat16: BF16, torch.float16: F16}[dtype].masks
    got = [host(o), host(lse), host(dq), host(dk), host(dv)]
    for name, a, e, bound in zip(PARTS, got, [eo, el, gq, gk, gv], bounds):
        ab, err = errors(a, e)
        if name != "lse" and np.max(np.abs(e[np.isfinite(e)]), initial=0.0) < 1e-3:
            err = ab
        tol = 2 * bound
        if name == "lse":
            tol = max(tol * max(1.0, np.sqrt(k.shape[1] / 64)),
                      np.sqrt(d) * 2.0 ** -24 / np.max(np.abs(e[np.isfinite(e)]), initial=1e-3))
        print(f"  {name}: rel {err:.2e} (bound {tol:.1e})")
        assert err <= tol, (case[0], name, err)
    empty = el == -np.inf
    if empty.any():
        assert np.all(got[0][empty] == 0.0) and np.all(got[2][empty] == 0.0)


def test_odd_strides_and_unread_keys():
    """Views whose rows are not 16-byte aligned give the contiguous call's values (the same
    arithmetic in the same order: to the bit), and keys left out by the padding mask may hold
    anything."""
    b, t, hq, hkv, d = 2, 77, 4, 2, 64
    wide = [syn.normal(s, (b, t, h, d + 3), "cuda") for s, h in ((1, hq), (2, hkv), (3, hkv), (4, hq))]
    pad = torch.zeros(b, t, dtype=torch.bool, device="cuda")
    pad[0, 5:9] = pad[1, 60:] = True
    for x in wide[1:3]:
        x[pad] = float("nan")
    mask, opts = dm.AttentionMask.key_padding(pad), dm.AttentionOptions(causal=True)
    out = []
    for f in (lambda x: x[..., 1:d + 1], lambda x: x[..., 1:d + 1].contiguous()):
        q, k, v, do = (f(x) for x in wide)
        o, lse = dm.attention_with_lse(q, k, v, mask, opts)
        out.append((o, lse) + tuple(dm.attention_backward(q, k, v, o, lse, do, mask, opts)))
    for a, e in zip(*out):
        assert torch.isfinite(a[~pad] if a.shape[2] == hkv and a.shape[:2] == pad.shape else a).all()
        assert torch.equal(a, e)
    assert all((g[pad] == 0).all() for g in out[0][3:])


def _step(x, mask, opts):
    q, k, v, do = x
    o, lse = dm.attention_with_lse(q, k, v, mask, opts)
    return (o, lse) + tuple(dm.attention_backward(q, k, v, o, lse, do, mask, opts))


@pytest.mark.parametrize("dtype,d", [(torch.float32, 64), (torch.float32, 128), (torch.float32, 256),
                                     (torch.float32, 13), (torch.bfloat16, 80), (torch.float16, 200)])
@pytest.mark.parametrize("case", ["tail", "neighbours", "later_keys", "earlier_queries", "window", "empty_rows"])
def test_unseen_rows_may_hold_anything(case, dtype, d):
    """Rows that a query (or a key) does not see reach none of its results, infinite and NaN ones
    included: what has no such row in sight is, to the bit, what it is with finite values there. But
    for dq: a query whose own results are NaN has a log-sum-exp of -inf and takes no part in the keys
    its tile walks over, so another row's sum of at most 167 terms may start at another key. In f32
    two orders of it are within 2 sqrt(167) 2^-24 = 1.6e-6 of the largest value, and a 16-bit result
    within one unit in the last place."""
    print(f"case {case} {dtype} D={d}", flush=True)
    t, hq, hkv = 167, 4, 2
    b, bad, mask, opts = 1, {}, None, dm.AttentionOptions(causal=True)
    idx = torch.arange(t, device="cuda")
    clean_q = clean_k = idx < 0  # the rows whose results must not change
    if case == "tail":  # positions past the last offset belong to no sequence
        cu = torch.tensor([0, 37, 100], dtype=torch.int32, device="cuda")
        mask, opts = dm.AttentionMask.packed(cu, cu), dm.AttentionOptions()
        rows = dict.fromkeys("qkvg", range(100, t))
        clean_q = clean_k = idx >= 0
    elif case == "neighbours":
        cu = torch.tensor([0, 37, 90, t], dtype=torch.int32, device="cuda")
        mask = dm.AttentionMask.packed(cu, cu)
        rows = dict.fromkeys("qkvg", (37, 60, 89))
        clean_q = clean_k = (idx < 37) | (idx >= 90)
    elif case == "later_keys":
        rows = dict(k=(75, 110), v=(70, 130))
        clean_q = idx < 70
    elif case == "earlier_queries":
        rows = dict(q=(60, 61), g=(62,))
        clean_q, clean_k = (idx < 60) | (idx > 62), idx > 62
    elif case == "window":  # a query sees itself and the 20 before
        opts = opts.with_window(20, 0)
        rows = dict.fromkeys("qkvg", (60, 75))
        clean_q, clean_k = (idx < 60) | (idx > 95), (idx < 40) | (idx > 95)
    else:  # every key of the second batch row is left out, 16 of the first
        b, opts = 2, dm.AttentionOptions()
        pad = torch.zeros(b, t, dtype=torch.bool, device="cuda")
        pad[1], pad[0, 40:56] = True, True
        mask = dm.AttentionMask.key_padding(pad)
        rows = {}
        clean_q = clean_k = idx >= 0
    shapes = ((b, t, hq, d), (b, t, hkv, d), (b, t, hkv, d), (b, t, hq, d))
    x = [syn.normal(900 + i, s, "cuda").to(dtype) for i, s in enumerate(shapes)]
    y = [z.clone() for z in x]
    for name, z in zip("qkvg", y):
        for i, r in enumerate(rows.get(name, ())):
            z[:, r] = (float("nan"), float("inf"), float("-inf"))[i % 3]
    if case == "empty_rows":
        for z in y:
            z[1] = float("nan")
        for z in y[1:3]:
            z[0, 40:56] = float("inf")
    assert clean_q.any()
    want, got = _step(x, mask, opts), _step(y, mask, opts)
    torch.cuda.synchronize()
    for name, e, a in zip(("o", "lse", "dq", "dk", "dv"), want, got):
        keep = clean_k if name in ("dk", "dv") else clean_q
        assert torch.isfinite(e[:, keep]).logical_or(e[:, keep] == -float("inf")).all()
        if name != "dq":
            assert torch.equal(a[:, keep], e[:, keep]), name
        else:
            a, e = a[:, keep].float(), e[:, keep].float()
            ulp = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]
            assert torch.isfinite(a).all() and ((a - e).abs() <= 1.6e-6 * e.abs().max() + ulp * e.abs()).all()
    if case == "empty_rows":
        assert all((z[1] == 0).all() for z in (got[0], got[2], got[3], got[4]))
        assert all((z[0, 40:56] == 0).all() for z in got[3:])


def test_seen_infinities_arrive():
    """A value that is not finite reaches the rows that see it, its own element only."""
    t, h, d = 70, 2, 64
    q, k, v, do = (syn.normal(950 + i, (1, t, h, d), "cuda") for i in range(4))
    opts, at = dm.AttentionOptions(causal=True), 37
    clean, _ = dm.attention_with_lse(q, k, v, None, opts)
    v[0, at, 1, 5], v[0, at + 9, 0, 60] = float("inf"), float("-inf")
    o, _ = dm.attention_with_lse(q, k, v, None, opts)
    clean[0, at:, 1, 5], clean[0, at + 9:, 0, 60] = float("inf"), float("-inf")
    assert torch.equal(o, clean)
