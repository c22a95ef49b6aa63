"""The f32 chunked gated delta rule (f32 inputs, and 16-bit ones of widths the 16-bit MFMA kernels
do not take) against the f64 oracle: widths that are not multiples of the kernels' 64 columns,
every padded width up to 256, chunks of 1, 63, 64 and 65 tokens, an empty sequence, a batch
without offsets, and calls with few and with many (sequence, head) pairs (the state pass takes 16
columns a workgroup below 256 workgroups of 32, else 32).

Bounds, of the largest difference over the largest value. f32: sums of up to 256 products round to
sqrt(256) 2^-24 = 1e-6, and up to four such products feed one another: 4e-6. 16-bit inputs: the
outputs' rounding (half a unit in the last place, 2^-8 of a value's power of two for bf16) with
the sums in f32: 4e-3."""
import numpy as np
import pytest
import torch

import dashmag_amd as dm
import oracle
from dashmag_amd import _lib, synthetic as syn
from fixtures import errors

pytestmark = pytest.mark.gpu


def host(x):
    return x.detach().float().cpu().numpy()


@pytest.mark.parametrize("dtype,dk,dv,lens,h,l2norm,states", [
    (torch.float32, 128, 128, [65, 0, 1, 63, 64], 3, True, True),
    (torch.float32, 20, 36, [130], 2, False, False),
    (torch.float32, 192, 64, [70, 3], 2, True, True),
    (torch.float32, 256, 256, [100], 1, True, True),
    (torch.float32, 64, 128, [90, 64, 20], 24, False, True),
    (torch.float32, 128, 256, [65, 30], 20, True, True),
    (torch.float32, 160, 256, [65, 30], 20, True, False),
    (torch.float32, 256, 256, [65, 30], 17, False, True),
    (torch.float32, 128, 96, 3, 2, True, True),
    (torch.bfloat16, 20, 30, [64, 33], 2, True, True),
    (torch.float16, 136, 72, [129], 2, False, True),
])
def test_matches_oracle(dtype, dk, dv, lens, h, l2norm, states):
    if isinstance(lens, int):  # a batch of sequences of 100 tokens
        B, T, S, cu = lens, 100, lens, None
    else:
        B, T, S = 1, sum(lens), len(lens)
        cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32)
    seed = 500 + 3 * dk + dv + T
    q = syn.normal(seed, (B, T, h, dk), "cuda")
    k = syn.normal(seed + 1, (B, T, h, dk), "cuda")
    if not l2norm:
        q, k = syn.l2norm(q), syn.l2norm(k)
    v = syn.normal(seed + 2, (B, T, h, dv), "cuda")
    g = -torch.nn.functional.softplus(syn.normal(seed + 3, (B, T, h), "cuda"))
    beta = torch.sigmoid(syn.normal(seed + 4, (B, T, h), "cuda"))
    h0 = syn.normal(seed + 5, (S, h, dk, dv), "cuda", std=0.1) if states else None
    do = syn.normal(seed + 6, (B, T, h, dv), "cuda").to(dtype)
    dfin = syn.normal(seed + 7, (S, h, dk, dv), "cuda", std=0.1) if states else None
    q, k, v = q.to(dtype), k.to(dtype), v.to(dtype)
    print(f"case {dtype} {dk}x{dv} lens {lens} h {h}", flush=True)
    _lib.probe_reset()
    opts = dm.ChunkGatedDeltaOptions(qk_l2norm=l2norm, output_final_state=True)
    cud = None if cu is None else cu.cuda()
    got = list(dm.chunk_gated_delta_rule(q, k, v, g, beta, h0, cud, opts))
    got += dm.chunk_gated_delta_rule_backward(q, k, v, g, beta, h0, cud, do, dfin, opts)
    torch.cuda.synchronize()
    pc = _lib.probe_counts()
    assert pc["gdr_chunk_fwd"] > 0 and pc["gdr_chunk_bwd"] > 0, pc
    a = (host(q), host(k), host(v), host(g), host(beta), None if h0 is None else host(h0))
    cun = None if cu is None else cu.numpy()
    want = list(oracle.gdr_chunk_fwd(*a, cun, l2norm, precision="f64"))
    want += oracle.gdr_chunk_bwd(*a, host(do), None if dfin is None else host(dfin), cun, l2norm,
                                 precision="f64")
    tol = 4e-6 if dtype == torch.float32 else 4e-3
    for name, x, e in zip(["out", "final", "dq", "dk", "dv", "dg", "dbeta", "dh0"], got, want):
        if x is None:
            assert name == "dh0" and h0 is None
            continue
        rel = errors(host(x), e)[1]
        print(f"  {name}: rel {rel:.2e}")
        assert rel <= tol, name


@pytest.mark.parametrize("dtype,dk,dv", [(torch.float32, 128, 128), (torch.float32, 20, 36),
                                         (torch.bfloat16, 136, 72)])
@pytest.mark.parametrize("what", ["q", "k", "v", "beta", "g", "do"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_tokens_depend_on_earlier_ones_alone(what, dtype, dk, dv, value):
    """A token's value that is not finite does not reach the results that do not depend on it, within
    its chunk either: forward, the outputs of the tokens before it (of every other token for a query);
    backward, with a gradient or query at fault, dv of the tokens after it and dq of every other; with
    a value, dq of the tokens before it, dv and the initial state's gradient. Bounds as above (such a
    chunk's sums run in another order)."""
    T, H, x = 150, 2, 90
    print(f"case {what} {value} {dtype} {dk}x{dv}", flush=True)
    q = syn.l2norm(syn.normal(71, (1, T, H, dk), "cuda")).to(dtype)
    k = syn.l2norm(syn.normal(72, (1, T, H, dk), "cuda")).to(dtype)
    v, do = (syn.normal(s, (1, T, H, dv), "cuda").to(dtype) for s in (73, 74))
    g = -torch.nn.functional.softplus(syn.normal(75, (1, T, H), "cuda"))
    beta = torch.sigmoid(syn.normal(76, (1, T, H), "cuda"))
    h0 = syn.normal(77, (1, H, dk, dv), "cuda", std=0.1)
    opts = dm.ChunkGatedDeltaOptions(output_final_state=True)
    bad = dict(q=q.clone(), k=k.clone(), v=v.clone(), g=g.clone(), beta=beta.clone(), do=do.clone())
    bad[what][0, x, 0] = value

    def step(q, k, v, g, beta, do):
        out, fin = dm.chunk_gated_delta_rule(q, k, v, g, beta, h0, None, opts)
        gr = dm.chunk_gated_delta_rule_backward(q, k, v, g, beta, h0, None, do, None, opts)
        return dict(out=out, fin=fin, dq=gr[0], dv=gr[2], dh0=gr[5])
    want, got = step(q, k, v, g, beta, do), step(**bad)
    before, after = slice(0, x), slice(x + 1, T)
    same = {"q": dict(out=(before, after), fin=(slice(None),), dq=(before, after), dv=(after,)),
            "k": dict(out=(before,)), "beta": dict(out=(before,)), "g": dict(out=(before,)),
            "v": dict(out=(before,), dq=(before,), dv=(slice(None),), dh0=(slice(None),)),
            "do": dict(out=(slice(None),), fin=(slice(None),), dq=(before, after), dv=(after,))}[what]
    tol = 4e-6 if dtype == torch.float32 else 4e-3
    for name, parts in same.items():
        for part in parts:
            a, e = host(got[name][:, part]), host(want[name][:, part])
            assert np.isfinite(a).all(), (name, part)
            assert errors(a, e)[1] <= tol, (name, part)
    for name in want:  # the other head
        h = 1 if name in ("fin", "dh0") else 2
        assert torch.equal(got[name].select(h, 1), want[name].select(h, 1)), name
