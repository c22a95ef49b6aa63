"""What a program that trains or serves with this framework calls, as measurable cases.

Every case is one pass through the public operations of ``dashmag_amd``: an attention layer's
forward and backward, a prefill, a decoding step against a key-value cache, the gated delta rule
in chunks and one token at a time, the causal conv1d in front of it, and the loss over the
vocabulary. Inputs are on the GPU, with the distributions of the benchmark's synthetic data
(q, k, v, gradients N(0, 1); gates g = -softplus(N(0, 1)); beta = sigmoid(N(0, 1)); states
N(0, 0.1)). Offsets and lengths are int32 tensors on the GPU, as the program's batching leaves them.
"""
import math
import random

import torch
import torch.nn.functional as F

import dashmag_amd as dm

DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZE = {"bf16": 2, "f16": 2, "f32": 4}


# ------------------------------------------------------------------------------------------
# The cases
# ------------------------------------------------------------------------------------------

def listed():
    return [
        # A grouped-query attention layer's training step over a packed batch of documents: the
        # benchmark's headline batch.
        dict(name="attn_train_packed_d128", kind="attn", train=True, dtype="bf16", b=1, t=16384,
             hq=32, hkv=8, d=128, mask="packed", causal=True, window=0,
             lens="307,2954,3945,952,3616,2791,1819"),
        # The same step with wide heads over one sequence: the attention layers of a hybrid
        # Gated DeltaNet model.
        dict(name="attn_train_d256", kind="attn", train=True, dtype="bf16", b=1, t=6144, hq=8,
             hkv=2, d=256, mask="none", causal=True, window=0, lens=""),
        # A prompt's prefill with narrow heads.
        dict(name="attn_prefill_d64", kind="attn", train=False, dtype="bf16", b=1, t=6144, hq=8,
             hkv=2, d=64, mask="none", causal=True, window=0, lens=""),
        # A training step in single precision on a short sequence: the smallest attention call.
        dict(name="attn_train_f32", kind="attn", train=True, dtype="f32", b=1, t=256, hq=4,
             hkv=4, d=64, mask="none", causal=True, window=0, lens=""),
        # Serving: one token for each of 64 requests, 512 to 8192 cached keys each, the cache
        # packed.
        dict(name="decode_packed_d128", kind="decode", dtype="bf16", cache="packed", b=64, s=8192,
             lo=512, hq=32, hkv=8, d=128, window=0, page=0, lseed=3),
        # Serving at a small batch with a sliding window over a full cache of wide heads: a call
        # of microseconds.
        dict(name="decode_window_d256", kind="decode", dtype="bf16", cache="dense", b=8, s=6144,
             lo=6144, hq=8, hkv=2, d=256, window=1024, page=0, lseed=0),
        # A Gated DeltaNet layer's training step over a packed batch.
        dict(name="gdr_train_d128", kind="gdr", train=True, dtype="bf16", h=16, dk=128, dv=128,
             lens="2729,1502,4152,2700,880,3748,5957,11100", l2norm=False, initial=True,
             final=False),
        # The same layer's prefill of one prompt, handing its state to decoding.
        dict(name="gdr_prefill_d128", kind="gdr", train=False, dtype="bf16", h=16, dk=128, dv=128,
             lens="6144", l2norm=True, initial=False, final=True),
        # The layer's training step in single precision, ragged sequences.
        dict(name="gdr_train_f32", kind="gdr", train=True, dtype="f32", h=8, dk=128, dv=128,
             lens="700,1001,347", l2norm=True, initial=True, final=True),
        # Serving: one token of the recurrent rule for each of 128 requests.
        dict(name="gdr_step_b128", kind="step", dtype="bf16", b=128, h=16, dk=128, dv=128,
             l2norm=True),
        # The causal convolution in front of the gated delta rule, forward and backward, over
        # the packed batch.
        dict(name="conv1d_train", kind="conv", train=True, dtype="bf16", c=6144, k=4, silu=True,
             bias=False, state=True, lens="2729,1502,4152,2700,880,3748,5957,11100"),
        # The loss over the vocabulary with both gradients: the largest call.
        dict(name="loss_train", kind="loss", dtype="bf16", n=4096, d=4096, v=151936,
             smoothing=0.1, z_loss=1e-4),
    ]


def _log(rng, lo, hi, step=1):
    """A whole number from lo to hi, uniform in its logarithm, a multiple of ``step``."""
    x = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step
    return max(lo, min(hi, x))


def _cut(rng, total, n):
    """``total`` tokens in ``n`` sequences of random lengths, as text."""
    n = min(n, total)
    at = [0] + sorted(rng.sample(range(1, total), n - 1)) + [total]
    return ",".join(str(y - x) for x, y in zip(at, at[1:]))


def draw(rng):
    kind = rng.choice(["attn", "attn", "attn32", "decode", "decode", "gdr", "gdr", "gdr32",
                       "step", "conv", "loss"])
    half = rng.choice(["bf16", "bf16", "f16"])
    if kind in ("attn", "attn32"):
        f32 = kind == "attn32"
        d = rng.choice([64, 128] if f32 else [64, 128, 256])
        hkv = rng.choice([1, 2, 4] if f32 else [1, 2, 4, 8])
        mask = rng.choice(["none", "none", "packed", "padding"])
        t = _log(rng, 64, 1024) if f32 else _log(rng, 256, 16384 if mask == "packed" else 6144)
        return dict(kind="attn", train=rng.random() < 0.7, dtype="f32" if f32 else half,
                    b=rng.choice([2, 3]) if mask == "padding" and t <= 2048 else 1, t=t,
                    hq=hkv * rng.choice([1, 2, 4]), hkv=hkv, d=d, mask=mask,
                    causal=rng.random() < 0.8, window=rng.choice([0, 0, 0, 128, 1024]),
                    lens=_cut(rng, t, max(2, t // 1500)) if mask == "packed" else "")
    if kind == "decode":
        hkv = rng.choice([1, 2, 4, 8])
        s = _log(rng, 512, 8192)
        cache = rng.choice(["dense", "packed", "paged"])
        return dict(kind="decode", dtype=half, cache=cache, b=_log(rng, 1, 64), s=s,
                    lo=max(1, s // 16), hq=hkv * rng.choice([1, 4, 8]), hkv=hkv,
                    d=rng.choice([64, 128, 256]), window=rng.choice([0, 0, 1024]),
                    page=rng.choice([16, 64]) if cache == "paged" else 0,
                    lseed=rng.randrange(1 << 30))
    if kind in ("gdr", "gdr32"):
        f32 = kind == "gdr32"
        t = _log(rng, 64, 2048 if f32 else 32768)
        dk, dv = rng.choice([(128, 128), (128, 128), (64, 64), (64, 128), (96, 64)])
        return dict(kind="gdr", train=rng.random() < 0.6, dtype="f32" if f32 else half,
                    h=rng.choice([2, 4, 8] if f32 else [4, 8, 16]), dk=dk, dv=dv,
                    lens=_cut(rng, t, rng.choice([1, 2, 8])), l2norm=rng.random() < 0.5,
                    initial=rng.random() < 0.5, final=rng.random() < 0.5)
    if kind == "step":
        return dict(kind="step", dtype=rng.choice(["bf16", "bf16", "f16", "f32"]),
                    b=_log(rng, 1, 256), h=rng.choice([4, 8, 16, 32]),
                    dk=rng.choice([64, 128, 128]), dv=rng.choice([64, 128, 128]),
                    l2norm=rng.random() < 0.5)
    if kind == "conv":
        t = _log(rng, 64, 32768)
        return dict(kind="conv", train=rng.random() < 0.7, dtype=rng.choice([half, half, "f32"]),
                    c=_log(rng, 512, 6144, 8), k=rng.choice([2, 3, 4, 4]),
                    silu=rng.random() < 0.7, bias=rng.random() < 0.5, state=rng.random() < 0.5,
                    lens=_cut(rng, t, rng.choice([1, 2, 8])))
    return dict(kind="loss", dtype=half, n=_log(rng, 64, 4096), d=_log(rng, 512, 4096, 8),
                v=_log(rng, 2000, 151936), smoothing=rng.choice([0.0, 0.1]),
                z_loss=rng.choice([0.0, 1e-4]))


# ------------------------------------------------------------------------------------------
# Inputs
# ------------------------------------------------------------------------------------------

def _lens(case):
    return [int(x) for x in case["lens"].split(",")]


def _offsets(lens):
    at = [0]
    for n in lens:
        at.append(at[-1] + n)
    return at


def _cache_lens(case):
    r = random.Random(case["lseed"])
    return [r.randint(case["lo"], case["s"]) for _ in range(case["b"])]


def _pads(case):
    """Keys left out at each row's end of a padded batch (the batch's longest row has none)."""
    return [0] + [case["t"] // (3 + i) for i in range(case["b"] - 1)]


class _Draw:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(1000003 * seed + 17)

    def normal(self, shape, dtype=torch.float32, std=1.0):
        x = torch.randn(shape, generator=self.g, device="cuda")
        return (x if std == 1.0 else x * std).to(dtype)

    def unit(self, shape, dtype):
        x = self.normal(shape)
        return (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)).to(dtype)


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, _Draw(seed))


def _attn_mask(case):
    if case["mask"] == "packed":
        cu = _i32(_offsets(_lens(case)))
        return dm.AttentionMask.packed(cu, cu)
    if case["mask"] == "padding":
        pad = torch.zeros(case["b"], case["t"], dtype=torch.bool)
        for i, n in enumerate(_pads(case)):
            if n:
                pad[i, case["t"] - n:] = True
        return dm.AttentionMask.key_padding(pad.cuda())
    return dm.AttentionMask.none()


def _attn_prepare(case, r):
    dt, b, t, d = DT[case["dtype"]], case["b"], case["t"], case["d"]
    options = dm.AttentionOptions(causal=case["causal"])
    if case["window"]:
        options = options.with_window(case["window"] - 1, case["window"] - 1)
    st = dict(kind="attn", train=case["train"], q=r.normal((b, t, case["hq"], d), dt),
              k=r.normal((b, t, case["hkv"], d), dt), v=r.normal((b, t, case["hkv"], d), dt),
              mask=_attn_mask(case), options=options)
    if case["train"]:
        st["do"] = r.normal((b, t, case["hq"], d), dt)
    return st


def _decode_prepare(case, r):
    dt, b, s, hkv, d = DT[case["dtype"]], case["b"], case["s"], case["hkv"], case["d"]
    lens = _cache_lens(case)
    options = dm.AttentionOptions()
    if case["window"]:
        options = options.with_window(case["window"] - 1, 0)
    st = dict(kind="decode", cache=case["cache"], q=r.normal((b, case["hq"], d), dt),
              options=options, lengths=None)
    if case["cache"] == "packed":
        shape = (sum(lens), hkv, d)
        st["cu"] = _i32(_offsets(lens))
    elif case["cache"] == "paged":
        per = -(-s // case["page"])
        shape = (b * per, case["page"], hkv, d)
        pages = list(range(b * per))
        random.Random(case["lseed"] + 1).shuffle(pages)
        st["table"] = _i32(pages).reshape(b, per)
        st["lengths"] = _i32(lens)
    else:
        shape = (b, s, hkv, d)
        st["lengths"] = _i32(lens) if case["lo"] < s else None
    st["k"], st["v"] = r.normal(shape, dt), r.normal(shape, dt)
    return st


def _gdr_prepare(case, r):
    dt, h, dk, dv, lens = DT[case["dtype"]], case["h"], case["dk"], case["dv"], _lens(case)
    t = sum(lens)
    qk = r.normal if case["l2norm"] else r.unit
    st = dict(kind="gdr", train=case["train"], q=qk((1, t, h, dk), dt), k=qk((1, t, h, dk), dt),
              v=r.normal((1, t, h, dv), dt), g=-F.softplus(r.normal((1, t, h))),
              beta=torch.sigmoid(r.normal((1, t, h))).to(dt), h0=None, dfin=None,
              cu=_i32(_offsets(lens)) if len(lens) > 1 else None,
              options=dm.ChunkGatedDeltaOptions(qk_l2norm=case["l2norm"],
                                                output_final_state=case["final"]))
    if case["initial"]:
        st["h0"] = r.normal((len(lens), h, dk, dv), std=0.1)
    if case["train"]:
        st["do"] = r.normal((1, t, h, dv), dt)
        if case["final"]:
            st["dfin"] = r.normal((len(lens), h, dk, dv), std=0.1)
    return st


def _step_prepare(case, r):
    dt, b, h, dk, dv = DT[case["dtype"]], case["b"], case["h"], case["dk"], case["dv"]
    qk = r.normal if case["l2norm"] else r.unit
    return dict(kind="step", q=qk((b, h, dk), dt), k=qk((b, h, dk), dt),
                v=r.normal((b, h, dv), dt), g=-F.softplus(r.normal((b, h))),
                beta=torch.sigmoid(r.normal((b, h))).to(dt),
                state=r.normal((b, h, dk, dv), std=0.1),
                options=dm.GatedDeltaStepOptions(qk_l2norm=case["l2norm"]))


def _conv_prepare(case, r):
    dt, c, k, lens = DT[case["dtype"]], case["c"], case["k"], _lens(case)
    t, n = sum(lens), len(lens)
    st = dict(kind="conv", train=case["train"], x=r.normal((1, t, c), dt),
              weight=r.normal((c, k), dt, std=0.5),
              bias=r.normal((c,), dt, std=0.1) if case["bias"] else None,
              h0=r.normal((n, k - 1, c)) if case["state"] else None,
              cu=_i32(_offsets(lens)) if n > 1 else None, gfin=None,
              options=dm.CausalConv1dOptions(
                  activation=dm.Activation.SILU if case["silu"] else dm.Activation.NONE,
                  output_final_state=case["state"]))
    if case["train"]:
        st["go"] = r.normal((1, t, c), dt)
        if case["state"]:
            st["gfin"] = r.normal((n, k - 1, c))
    return st


def _loss_prepare(case, r):
    dt, n, v = DT[case["dtype"]], case["n"], case["v"]
    targets = torch.randint(0, v, (n,), generator=r.g, device="cuda")
    ignored = torch.arange(n, device="cuda") % 16 == 5  # a prompt's tokens carry no loss
    targets[ignored] = -100
    upstream = torch.zeros(3, n, device="cuda")
    upstream[0] = 1.0 / (n - len(range(5, n, 16)))
    return dict(kind="loss", hidden=r.normal((n, case["d"]), dt),
                weight=r.normal((v, case["d"]), dt, std=0.02), targets=targets,
                upstream=upstream,
                options=dm.CrossEntropyOptions(label_smoothing=case["smoothing"],
                                               z_loss=case["z_loss"]))


_PREPARE = dict(attn=_attn_prepare, decode=_decode_prepare, gdr=_gdr_prepare, step=_step_prepare,
                conv=_conv_prepare, loss=_loss_prepare)


# ------------------------------------------------------------------------------------------
# One pass
# ------------------------------------------------------------------------------------------

def run(st):
    kind = st["kind"]
    if kind == "attn":
        out, lse = dm.attention_with_lse(st["q"], st["k"], st["v"], st["mask"], st["options"])
        if not st["train"]:
            return out, lse
        return (out, lse) + tuple(dm.attention_backward(
            st["q"], st["k"], st["v"], out, lse, st["do"], st["mask"], st["options"]))
    if kind == "decode":
        if st["cache"] == "packed":
            return dm.attention_decode_packed(st["q"], st["k"], st["v"], st["cu"],
                                              options=st["options"])
        if st["cache"] == "paged":
            return dm.attention_decode_paged(st["q"], st["k"], st["v"], st["table"],
                                             st["lengths"], st["options"])
        return dm.attention_decode(st["q"], st["k"], st["v"], st["lengths"], st["options"])
    if kind == "gdr":
        args = (st["q"], st["k"], st["v"], st["g"], st["beta"], st["h0"], st["cu"])
        out = tuple(dm.chunk_gated_delta_rule(*args, st["options"]))
        if st["train"]:
            out += tuple(dm.chunk_gated_delta_rule_backward(*args, st["do"], st["dfin"],
                                                            st["options"]))
        return out
    if kind == "step":
        return dm.gated_delta_step(st["q"], st["k"], st["v"], st["g"], st["beta"], st["state"],
                                   options=st["options"])
    if kind == "conv":
        args = (st["x"], st["weight"], st["bias"], st["h0"], st["cu"])
        out = tuple(dm.causal_conv1d(*args, st["options"]))
        if st["train"]:
            out += tuple(dm.causal_conv1d_backward(*args, st["go"], st["gfin"], st["options"]))
        return out
    loss, logprob, _, rows = dm.linear_cross_entropy(st["hidden"], st["weight"], st["targets"],
                                                     st["options"])
    return (loss, logprob) + tuple(dm.linear_cross_entropy_backward(
        st["hidden"], st["weight"], st["targets"], rows, st["upstream"], st["options"]))


# ------------------------------------------------------------------------------------------
# What a pass cannot do without
# ------------------------------------------------------------------------------------------

def _pairs(case):
    """Visible (query, key) pairs of one query head."""
    w = case["window"] or case["t"] + 1
    total = 0
    for i, n in enumerate(_lens(case) if case["mask"] == "packed" else [case["t"]] * case["b"]):
        pad = _pads(case)[i] if case["mask"] == "padding" else 0
        r = torch.arange(n, dtype=torch.int64)
        lo = (r - (w - 1)).clamp(min=0)
        hi = r if case["causal"] else (r + (w - 1)).clamp(max=n - 1)
        hi = hi.clamp(max=n - 1 - pad)
        total += int((hi - lo + 1).clamp(min=0).sum())
    return total


def work(case):
    kind, e = case["kind"], SIZE[case["dtype"]]
    if kind == "attn":
        bt, d = case["b"] * case["t"], case["d"]
        q, kv, row = bt * case["hq"] * d * e, bt * case["hkv"] * d * e, bt * case["hq"] * 4
        p = _pairs(case) * case["hq"] * d
        if not case["train"]:
            return dict(bytes=2 * q + 2 * kv + row, flops=4 * p)
        # forward and backward each read their inputs
        return dict(bytes=6 * q + 6 * kv + 2 * row, flops=14 * p)
    if kind == "decode":
        seen = sum(min(n, case["window"] or n) for n in _cache_lens(case))
        return dict(bytes=2 * seen * case["hkv"] * case["d"] * e
                    + 2 * case["b"] * case["hq"] * case["d"] * e,
                    flops=4 * seen * case["hq"] * case["d"])
    if kind == "gdr":
        lens, h, dk, dv = _lens(case), case["h"], case["dk"], case["dv"]
        rows = sum(lens) * h
        ins = rows * ((2 * dk + dv) * e + 4 + e)
        state = len(lens) * h * dk * dv * 4
        b = ins + rows * dv * e + state * (case["initial"] + case["final"])
        n = rows / 64  # chunks of 64 tokens and heads
        intra = 2 * 64 * 64 * (3 * dk + dv) + 64 ** 3 * 2 / 3
        fl = n * (intra + 2 * 64 * 64 * dv + 6 * 64 * dk * dv)
        if case["train"]:
            b += ins + rows * dv * e + ins + state * (2 * case["initial"] + case["final"])
            fl += n * (2 * intra + 4 * 64 * 64 * (dk + dv) + 14 * 64 * dk * dv)
        return dict(bytes=b, flops=fl)
    if kind == "step":
        bh, dk, dv = case["b"] * case["h"], case["dk"], case["dv"]
        return dict(bytes=bh * (8 * dk * dv + (2 * dk + 2 * dv) * e + 4 + e), flops=bh * 7 * dk * dv)
    if kind == "conv":
        lens, c, k = _lens(case), case["c"], case["k"]
        tc, state = sum(lens) * c, case["state"] * len(lens) * (k - 1) * c * 4
        if not case["train"]:
            return dict(bytes=2 * tc * e + 2 * state, flops=2 * k * tc)
        return dict(bytes=5 * tc * e + 5 * state, flops=6 * k * tc)
    n, d, v = case["n"], case["d"], case["v"]
    # forward: hidden and weight read; backward: read again, both gradients written
    return dict(bytes=3 * (n + v) * d * e + 8 * n, flops=8 * n * d * v)


# ------------------------------------------------------------------------------------------
# How far another correct implementation may be off
# ------------------------------------------------------------------------------------------

def tolerance(case):
    # about four times the errors measured against exact(): 16-bit inputs and products' operands
    # in 16 bits with sums in 32, or 32 bits throughout
    if case["dtype"] == "f32":
        return {"rel": 1e-5}
    return {"rel": {"attn": 0.01, "decode": 0.01, "gdr": 0.016, "step": 0.007, "conv": 0.007,
                    "loss": 0.008}[case["kind"]]}


# ------------------------------------------------------------------------------------------
# The same results in 64 bits
# ------------------------------------------------------------------------------------------

def exact(case, seed):
    return _EXACT[case["kind"]](case, prepare(case, seed))


def _attn_exact(case, st):
    b, t, hq, hkv, d = (case[x] for x in ("b", "t", "hq", "hkv", "d"))
    q, k, v = (st[x].double() for x in ("q", "k", "v"))
    do = st["do"].double() if case["train"] else None
    out, lse = torch.zeros_like(q), torch.zeros(b, t, hq, dtype=torch.float64, device="cuda")
    dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
    scale = 1 / math.sqrt(d)
    spans = ([(0, a, z) for a, z in zip(*(lambda o: (o[:-1], o[1:]))(_offsets(_lens(case))))]
             if case["mask"] == "packed" else [(i, 0, t) for i in range(b)])
    for i, a, z in spans:
        n = z - a
        r = torch.arange(n, device="cuda")
        gap = r[:, None] - r[None, :]  # query's position less the key's
        hide = torch.zeros(n, n, dtype=torch.bool, device="cuda")
        if case["causal"]:
            hide |= gap < 0
        if case["window"]:
            hide |= gap.abs() > case["window"] - 1
        if case["mask"] == "padding":
            hide |= (r >= n - _pads(case)[i])[None, :]
        for h in range(hq):
            kh = h // (hq // hkv)
            qh, kk, vh = q[i, a:z, h], k[i, a:z, kh], v[i, a:z, kh]
            s = (qh @ kk.T).mul_(scale).masked_fill_(hide, -math.inf)
            ls = torch.logsumexp(s, 1)
            # a query that sees no key has zeros
            p = torch.exp(s - ls.masked_fill(ls == -math.inf, 0.0)[:, None])
            del s
            out[i, a:z, h], lse[i, a:z, h] = p @ vh, ls
            if do is not None:
                g = do[i, a:z, h]
                dv[i, a:z, kh] += p.T @ g
                ds = g @ vh.T
                ds -= (g * out[i, a:z, h]).sum(1, keepdim=True)
                ds.mul_(p).mul_(scale)
                dq[i, a:z, h] = ds @ kk
                dk[i, a:z, kh] += ds.T @ qh
    return (out, lse, dq, dk, dv) if case["train"] else (out, lse)


def _decode_exact(case, st):
    b, hq, hkv, d = (case[x] for x in ("b", "hq", "hkv", "d"))
    lens = _cache_lens(case)
    off = _offsets(lens)
    out = torch.empty(b, hq, d, dtype=torch.float64, device="cuda")
    for i, n in enumerate(lens):
        a = max(0, n - case["window"]) if case["window"] else 0
        if case["cache"] == "packed":
            k, v = st["k"][off[i] + a:off[i] + n], st["v"][off[i] + a:off[i] + n]
        elif case["cache"] == "paged":
            pages = st["table"][i].long()
            k, v = (x[pages].reshape(-1, hkv, d)[a:n] for x in (st["k"], st["v"]))
        else:
            k, v = st["k"][i, a:n], st["v"][i, a:n]
        k, v, q = k.double(), v.double(), st["q"][i].double().reshape(hkv, hq // hkv, d)
        for h in range(hkv):
            p = torch.softmax((q[h] @ k[:, h].T) / math.sqrt(d), 1)
            out[i, h * (hq // hkv):(h + 1) * (hq // hkv)] = p @ v[:, h]
    return out


def _l2(x):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def _gdr_chunked(q, k, v, g, beta, s, live):
    """The rule over [N, T, ...] rows (N = sequences x heads), 64 tokens at a time, from the states
    ``s``; tokens past a row's end have k = v = beta = g = 0 and leave the state alone."""
    n, t, dk = q.shape
    eye = torch.eye(64, dtype=torch.float64, device="cuda")
    low = torch.tril(torch.ones(64, 64, dtype=torch.bool, device="cuda"))
    outs = []
    for c in range(0, t, 64):
        m = live[c // 64]  # the rows, longest first, that have tokens in this chunk
        qc, kc, vc, bc = q[:m, c:c + 64], k[:m, c:c + 64], v[:m, c:c + 64], beta[:m, c:c + 64, None]
        gc = torch.cumsum(g[:m, c:c + 64], 1)
        decay = torch.exp((gc[:, :, None] - gc[:, None, :]).masked_fill(~low, -math.inf))
        kt = kc.transpose(1, 2).contiguous()
        a = -(bc * torch.bmm(kc, kt) * decay).masked_fill(eye.bool(), 0.0)
        inv, power = eye + a, a
        for _ in range(5):  # (1 - a)^-1 = (1 + a)(1 + a^2)(1 + a^4) ...: a^64 = 0
            power = torch.bmm(power, power)
            inv = inv + torch.bmm(inv, power)
        gam = torch.exp(gc)[..., None]
        w, u = torch.bmm(inv, bc * gam * kc), torch.bmm(inv, bc * vc)
        sc = s[:m]
        new = u - torch.bmm(w, sc)
        outs.append(torch.bmm(gam * qc, sc) + torch.bmm(torch.bmm(qc, kt) * decay, new))
        last = gc[:, -1:]
        kd = (torch.exp(last - gc)[..., None] * kc).transpose(1, 2).contiguous()
        sc = torch.exp(last)[..., None] * sc + torch.bmm(kd, new)
        s = torch.cat([sc, s[m:]]) if m < n else sc
    return outs, s


def _gdr_exact(case, st):
    lens, h, dk, dv = _lens(case), case["h"], case["dk"], case["dv"]
    if case["train"] and (max(lens) > 12000 or sum(lens) * h > 600000):
        return None  # the states of every chunk would take the time and the memory
    off = _offsets(lens)
    order = sorted(range(len(lens)), key=lambda i: -lens[i])
    most = -(-max(lens) // 64) * 64
    leaf = {x: st[x].double().requires_grad_(case["train"]) for x in ("q", "k", "v", "g", "beta")}
    h0 = (st["h0"].double() if st["h0"] is not None
          else torch.zeros(len(lens), h, dk, dv, dtype=torch.float64, device="cuda"))
    h0.requires_grad_(case["train"])
    with torch.set_grad_enabled(case["train"]):
        q, k = leaf["q"], leaf["k"]
        if case["l2norm"]:
            q, k = _l2(q), _l2(k)
        q = q / math.sqrt(dk)

        def rows(x):  # [1, T, H, ...] to [S H, most, ...]
            parts = [F.pad(x[0, off[i]:off[i + 1]].transpose(0, 1),
                           [0, 0] * (x.dim() - 3) + [0, most - lens[i]]) for i in order]
            return torch.cat(parts).contiguous()

        live = [h * sum(n > c for n in lens) for c in range(0, most, 64)]
        outs, s = _gdr_chunked(rows(q), rows(k), rows(leaf["v"]), rows(leaf["g"]),
                               rows(leaf["beta"]), h0[order].reshape(-1, dk, dv), live)
        full = torch.cat([F.pad(o, [0, 0, 0, 0, 0, len(order) * h - o.shape[0]]) for o in outs], 1)
        back = [order.index(i) for i in range(len(lens))]
        out = torch.cat([full[j * h:(j + 1) * h, :lens[i]].transpose(0, 1)
                         for i, j in enumerate(back)])[None]
        fin = s.reshape(len(lens), h, dk, dv)[back]
        answer = [out.detach(), fin.detach() if case["final"] else None]
        if case["train"]:
            total = (out * st["do"].double()).sum()
            if st["dfin"] is not None:
                total = total + (fin * st["dfin"].double()).sum()
            total.backward()
            answer += [leaf[x].grad for x in ("q", "k", "v", "g", "beta")]
            answer.append(h0.grad if case["initial"] else None)
    return tuple(answer)


def _step_exact(case, st):
    q, k, v, g, beta, s = (st[x].double() for x in ("q", "k", "v", "g", "beta", "state"))
    if case["l2norm"]:
        q, k = _l2(q), _l2(k)
    q = q / math.sqrt(case["dk"])
    s = s * torch.exp(g)[..., None, None]
    delta = beta[..., None] * (v - (s * k[..., None]).sum(-2))
    s = s + k[..., None] * delta[..., None, :]
    return (s * q[..., None]).sum(-2), s


def _conv_exact(case, st):
    lens, k, c = _lens(case), case["k"], case["c"]
    off = _offsets(lens)
    train = case["train"]
    x = st["x"].double().requires_grad_(train)
    w = st["weight"].double().requires_grad_(train)
    bias = st["bias"].double().requires_grad_(train) if case["bias"] else None
    h0 = st["h0"].double().requires_grad_(train) if case["state"] else None
    outs, fins = [], []
    with torch.set_grad_enabled(train):
        for i in range(len(lens)):
            head = h0[i] if h0 is not None else torch.zeros(k - 1, c, dtype=torch.float64,
                                                            device="cuda")
            rows = torch.cat([head, x[0, off[i]:off[i + 1]]])
            y = sum(rows[j:j + lens[i]] * w[:, j] for j in range(k))
            y = y + bias if bias is not None else y
            outs.append(F.silu(y) if case["silu"] else y)
            fins.append(rows[rows.shape[0] - (k - 1):])
        out, fin = torch.cat(outs)[None], torch.stack(fins)
        answer = [out.detach(), fin.detach() if case["state"] else None]
        if train:
            total = (out * st["go"].double()).sum()
            if st["gfin"] is not None:
                total = total + (fin * st["gfin"].double()).sum()
            total.backward()
            answer += [x.grad, w.grad, bias.grad if bias is not None else None,
                       h0.grad if h0 is not None else None]
    return tuple(answer)


def _loss_exact(case, st):
    n, v, eps, z = case["n"], case["v"], case["smoothing"], case["z_loss"]
    hidden, weight, targets = st["hidden"].double(), st["weight"].double(), st["targets"]
    counted = targets != -100
    up = st["upstream"][0].double()
    loss = torch.zeros(n, dtype=torch.float64, device="cuda")
    logprob = torch.zeros_like(loss)
    gh, gw = torch.zeros_like(hidden), torch.zeros_like(weight)
    for a in range(0, n, 512):
        r = slice(a, min(a + 512, n))
        logits = hidden[r] @ weight.T
        lse = torch.logsumexp(logits, 1)
        t = targets[r].clamp(min=0)
        zt = logits.gather(1, t[:, None])[:, 0]
        live = counted[r]
        logprob[r] = torch.where(live, zt - lse, torch.zeros_like(lse))
        loss[r] = torch.where(live, (1 - eps) * (lse - zt) + eps * (lse - logits.mean(1))
                              + z * lse * lse, torch.zeros_like(lse))
        dz = torch.exp(logits - lse[:, None]) * (1 + 2 * z * lse)[:, None] - eps / v
        dz[torch.arange(len(t), device="cuda"), t] -= 1 - eps
        dz *= (up[r] * live)[:, None]
        gh[r] = dz @ weight
        gw += dz.T @ hidden[r]
    return (loss.sum() / counted.sum()).reshape(1), logprob, gh, gw


_EXACT = dict(attn=_attn_exact, decode=_decode_exact, gdr=_gdr_exact, step=_step_exact,
              conv=_conv_exact, loss=_loss_exact)
