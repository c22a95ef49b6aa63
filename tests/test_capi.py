"""The C ABI without a GPU: the library loads, exports every symbol include/dashmi.h declares,
and its host-side visibility intervals equal the oracle's element-wise mask, to the bit."""
import ctypes
import os
import re

import numpy as np
import pytest

import oracle
from dashmag_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "dashmi.h")).read()
    return sorted(set(re.findall(r"\b(dm_[a-z0-9_]+)\s*\(", text)))


def test_header_and_bindings_agree():
    assert declared_symbols() == sorted(_lib.SIGNATURES)


def test_library_exports_every_declared_symbol():
    lb = _lib.lib()
    for name in declared_symbols():
        assert hasattr(lb, name), name


def _desc(tq, tk, causal, left, right, kind, cu_q=None, cu_k=None):
    d = _lib.AttentionDesc(b=1, tq=tq, tk=tk, hq=1, hkv=1, d=8, dtype=_lib.DM_F32,
                           mask_kind=kind)
    d.options.causal = int(causal)
    if left is not None or right is not None:
        d.options.has_window = 1
        d.options.window_left = _lib.DM_UNBOUNDED if left is None else left
        d.options.window_right = _lib.DM_UNBOUNDED if right is None else right
    keep = []
    if kind == _lib.DM_MASK_PACKED:
        cq = np.ascontiguousarray(cu_q, np.int32)
        ck = np.ascontiguousarray(cu_k, np.int32)
        keep = [cq, ck]
        d.cu_seqlens_q, d.cu_seqlens_k = cq.ctypes.data, ck.ctypes.data
        d.nseq = len(cq) - 1
    return d, keep


@pytest.mark.parametrize("case", range(60))
def test_row_bounds_equal_the_oracle_mask(case):
    rng = np.random.default_rng(1000 + case)
    tq, tk = int(rng.integers(1, 24)), int(rng.integers(1, 24))
    causal = bool(rng.integers(0, 2))
    left = None if rng.random() < 0.4 else int(rng.integers(0, 9))
    right = None if rng.random() < 0.4 else int(rng.integers(0, 9))
    packed = case % 2 == 1
    cu_q = cu_k = None
    if packed:
        s = int(rng.integers(1, 5))
        cu_q = np.concatenate([[0], np.sort(rng.integers(0, tq + 1, s))])
        cu_k = np.concatenate([[0], np.sort(rng.integers(0, tk + 1, s))])
    d, keep = _desc(tq, tk, causal, left, right,
                    _lib.DM_MASK_PACKED if packed else _lib.DM_MASK_NONE, cu_q, cu_k)
    q = np.zeros((1, tq, 1, 8), np.float32)
    k = np.zeros((1, tk, 1, 8), np.float32)
    call = oracle.AttentionCall(q, k, k, ("packed", cu_q, cu_k) if packed else None, causal,
                                None, left, right)
    want = call.visible_matrix(0)
    lo, hi = ctypes.c_int64(), ctypes.c_int64()
    for i in range(tq):
        assert _lib.lib().dm_attention_row_bounds(ctypes.byref(d), 0, i, ctypes.byref(lo),
                                                  ctypes.byref(hi)) == 0
        got = np.zeros(tk, bool)
        got[lo.value:hi.value] = True
        assert np.array_equal(got, want[i]), (i, lo.value, hi.value, want[i])


def test_refusal_names_the_operation():
    d, _ = _desc(4, 4, False, None, None, _lib.DM_MASK_NONE)
    d.hq, d.hkv = 3, 2
    rc = _lib.lib().dm_attention_fwd(ctypes.byref(d), None, None, None, None, None, None, 0, None)
    assert rc == _lib.DM_ERR_REFUSED
    assert _lib.last_error().startswith("attention: the query heads (3)")


def test_paged_decode_refusals():
    """The paged decode refuses before any launch: capacity and page size disagree, a packed
    offset array instead of a block table, a missing block table."""
    lb = _lib.lib()
    d, _ = _desc(1, 64, False, None, None, _lib.DM_MASK_NONE)
    d.dtype = _lib.DM_BF16
    call = lambda ps, bt, mp: lb.dm_attention_decode_paged(  # noqa: E731
        ctypes.byref(d), None, None, None, 4, ps, bt, mp, None, None, None, 0, None)
    assert call(16, None, 3) == _lib.DM_ERR_REFUSED
    assert _lib.last_error().startswith("attention_decode_paged: desc->tk (64)")
    assert call(0, None, 4) == _lib.DM_ERR_REFUSED
    assert "page_size must be positive" in _lib.last_error()
    assert call(16, None, 4) == _lib.DM_ERR_REFUSED
    assert "block table" in _lib.last_error()
    ck = np.zeros(2, np.int32)
    d.cu_seqlens_k = ck.ctypes.data
    assert call(16, None, 4) == _lib.DM_ERR_REFUSED
    assert "not cu_seqlens_k" in _lib.last_error()


def test_packed_decode_refuses_a_wrong_sequence_count():
    d, _ = _desc(1, 8, False, None, None, _lib.DM_MASK_NONE)
    ck = np.zeros(3, np.int32)
    d.cu_seqlens_k, d.nseq = ck.ctypes.data, 2
    rc = _lib.lib().dm_attention_decode(ctypes.byref(d), None, None, None, None, None, None, 0,
                                        None)
    assert rc == _lib.DM_ERR_REFUSED
    assert _lib.last_error().startswith("attention_decode: a packed cache")


def test_logprob_refusals():
    """The log-probability refuses before any launch: a masked id outside the vocabulary, every
    token masked, an f16 operand, a zero row_chunk."""
    lb = _lib.lib()
    d = _lib.LogprobDesc(n=4, v=5, d=8, hidden_dtype=_lib.DM_BF16, weight_dtype=_lib.DM_BF16,
                         vocab_chunk=0, row_chunk=3072)

    def call(ids):
        arr = (ctypes.c_uint32 * max(len(ids), 1))(*ids)
        return lb.dm_chosen_logprob(ctypes.byref(d), None, None, None,
                                    ctypes.cast(arr, ctypes.c_void_p), len(ids), None, None,
                                    None, None, 0, None)

    assert call([7]) == _lib.DM_ERR_REFUSED
    assert _lib.last_error() == ("chosen_logprob: masked token id 7 is not below the "
                                 "vocabulary size 5")
    assert call([4, 3, 2, 1, 0, 0]) == _lib.DM_ERR_REFUSED
    assert _lib.last_error() == "chosen_logprob: at least one token must stay unmasked"
    assert call([1, 1]) == _lib.DM_ERR_REFUSED  # passes the ids, stops at the workspace
    assert "workspace" in _lib.last_error()
    d.hidden_dtype = _lib.DM_F16
    assert call([]) == _lib.DM_ERR_REFUSED
    assert _lib.last_error() == "chosen_logprob: the log-probability takes bf16 or f32"
    d.hidden_dtype, d.row_chunk = _lib.DM_BF16, 0
    assert call([]) == _lib.DM_ERR_REFUSED
    assert _lib.last_error() == "chosen_logprob: row_chunk must be at least 1"


def test_noalloc_decode_refuses_calls_beyond_its_scratch():
    """The no-allocation decode refuses, before touching the device, a call whose partials would
    not fit its 16 MiB scratch (here 1024 x 64 rows of 256 f32 partials, 64 MiB)."""
    d = _lib.AttentionDesc(b=1024, tq=1, tk=100_000, hq=64, hkv=8, d=256, dtype=_lib.DM_BF16,
                           mask_kind=_lib.DM_MASK_NONE)
    lb = _lib.lib()
    assert lb.dm_attention_decode_workspace(ctypes.byref(d)) > (16 << 20)
    rc = lb.dm_attention_decode_noalloc(ctypes.byref(d), None, None, None, None, None, None)
    assert rc == _lib.DM_ERR_REFUSED
    assert _lib.last_error().startswith("attention_decode: the call needs")


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("b,tq,hq,tk", [
    (1, -1000, 8, 4096), (-1, 100000, 1, 4096), (-1, 1000, 1, 4096), (-3, -70000, 1, 4096), (1, 1000, -4, 4096),
    (1, 1000, 8, -4096), (1 << 40, 1 << 20, 1 << 24, 4096), (1 << 62, 64, 4, 4096), (3, (1 << 63) - 1, 1, 4096),
    (1, 1000, 8, 1 << 62)])
def test_forward_workspace_of_refused_sizes(b, tq, hq, tk, d):
    """The forward's size query answers 0 for sizes that no call has: a caller asks before the call that
    refuses it, so the query neither fails nor names a size."""
    x = _lib.AttentionDesc(b=b, tq=tq, tk=tk, hq=hq, hkv=1, d=d, dtype=_lib.DM_BF16, mask_kind=_lib.DM_MASK_NONE)
    for causal in (0, 1):
        x.options.causal = causal
        assert _lib.lib().dm_attention_fwd_workspace(ctypes.byref(x)) == 0
    if min(b, tq, hq, tk) < 0:
        assert _lib.lib().dm_attention_fwd(ctypes.byref(x), None, None, None, None, None, None, 0,
                                           None) == _lib.DM_ERR_REFUSED
        assert _lib.last_error() == "attention: negative dimension"


@pytest.mark.parametrize("dtype", [_lib.DM_BF16, _lib.DM_F16, _lib.DM_F32])
@pytest.mark.parametrize("n,row_chunk,v,d", [(16384, 1, 50000, 64), (40000, 3072, 151936, 4096), (40000, 100, 8192, 4096),
                                             (3000, 3072, 151936, 64), (1000, 7, 300, 8), (0, 3072, 1000, 64)])
def test_loss_workspace_bounds(dtype, n, row_chunk, v, d):
    """What the loss's backward takes besides its inputs' f32 copies: without the weight's gradient the
    logits of a block of rows, as much for their gradient and a few values a row; with it, no more than an f32 weight
    gradient besides (f32: nothing)."""
    lp = _lib.LogprobDesc(n=n, v=v, d=d, hidden_dtype=dtype, weight_dtype=dtype, vocab_chunk=0, row_chunk=row_chunk)
    x = _lib.LceDesc(lp=lp)
    frozen, both = (_lib.lib().dm_linear_cross_entropy_workspace(ctypes.byref(x), m) for m in (2, 1))
    block = -(-n // -(-n // row_chunk)) if n else 1
    chunk = min(v, 8192)
    copies = {_lib.DM_BF16: n * d, _lib.DM_F16: 2 * n * d + v * d, _lib.DM_F32: 0}[dtype] * 4
    assert frozen <= (64 << 20) + copies + 2 * block * chunk * 4 + 64 * max(n, 1) + v // 8 + 16 * 256
    assert both <= frozen + (0 if dtype == _lib.DM_F32 else v * d * 4 + 256)


def test_forward_split_is_bounded():
    """The forward is cut along the keys into 1024 workgroups at most (their partial outputs 128 MB and
    their references), and a packed call of more than two sequences not at all."""
    rng = np.random.default_rng(5)
    split = 0
    for _ in range(3000):
        d, hq = int(rng.choice([64, 128, 256])), int(rng.choice([1, 2, 4, 8, 11, 16, 64]))
        tq, tk = (int(np.exp(rng.uniform(2, 11.5))) for _ in range(2))
        x = _lib.AttentionDesc(b=1, tq=tq, tk=tk if rng.random() < 0.4 else tq, hq=hq, hkv=1, d=d, dtype=_lib.DM_BF16,
                               mask_kind=_lib.DM_MASK_NONE)
        x.options.causal = int(rng.random() < 0.6)
        if rng.random() < 0.3:
            x.mask_kind, x.nseq = _lib.DM_MASK_PACKED, int(rng.integers(1, 4))
        nbytes = _lib.lib().dm_attention_fwd_workspace(ctypes.byref(x))
        split += nbytes > 0
        queries = 128 if d == 256 else 256
        assert nbytes <= 1024 * queries * (4 * d + 8) + 512
        if x.mask_kind == _lib.DM_MASK_PACKED and x.nseq > 2 or x.tk <= 384:
            assert nbytes == 0
    assert split > 300


@pytest.mark.parametrize("dk,dv", [(16, 16), (64, 64), (96, 64), (128, 128), (256, 256), (136, 72)])
def test_f32_chunk_workspace(dk, dv):
    """The f32 chunked rule holds, per chunk of 64 tokens and head, rows padded to multiples of 64 columns:
    the forward 4 rows of Dk and 2 of Dv, P and, past 128 x 128, the state; the backward 5 and 4, P, A, T
    and two states, and the gates' sums."""
    kp, vp = -(-dk // 64) * 64, -(-dv // 64) * 64
    for b, t, h in ((1, 2048, 8), (3, 130, 2)):
        x = _lib.GdrDesc(b=b, t=t, h=h, dk=dk, dv=dv, dtype=_lib.DM_F32, g_dtype=_lib.DM_F32, beta_dtype=_lib.DM_F32)
        chunks = b * -(-t // 64) * h
        rows = lambda k, v: 64 * (k * kp + v * vp)  # noqa: E731
        fwd = rows(4, 2) + 64 * 64 + 64 * 2 + (vp * kp if vp * kp > 64 * (kp + vp) else 0)
        bwd = rows(5, 4) + 3 * 64 * 64 + 2 * vp * kp + 64 * 5 + 64 * (6 * kp // 64 + vp // 64 + 1)
        for size, want in ((_lib.lib().dm_gdr_chunk_fwd_workspace, fwd), (_lib.lib().dm_gdr_chunk_bwd_workspace, bwd)):
            assert size(ctypes.byref(x)) <= chunks * want * 4 + 24 * 256
