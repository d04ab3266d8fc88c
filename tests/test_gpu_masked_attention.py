"""The MFMA kernels of masked and dropped-out attention (bf16, head dims 64 and
128) at their edges, against the oracle in fp32: 64-row tiles and remainders,
the mask layouts with kernels of their own (one bit per key, boolean per score,
additive; four at a time or one by one), skipped tiles, grouped heads, offsets
and dropout over even and odd key counts."""

from __future__ import annotations

import math

import pytest
import torch

import nano_megatron_amd.functional as Fn
from oracle import reference as R
from tests.parity import rel_l2
from tests.test_gpu_attention_f32 import _reference

pytestmark = pytest.mark.gpu

CASES = [
    # (mask, causal, offset, hq, hkv, sq, sk, d, p)
    ("none", True, 0, 2, 2, 1, 1, 64, 0.3),
    ("none", True, 3, 4, 2, 130, 191, 64, 0.1),  # odd key count: dropout pairs straddle rows
    ("none", False, 0, 4, 1, 64, 128, 128, 0.1),
    ("keys", True, 0, 4, 4, 200, 200, 64, 0.0),
    ("keys", False, 0, 4, 2, 65, 321, 128, 0.0),
    ("keys", True, 16400, 1, 1, 5, 16384, 64, 0.0),  # the most keys kept as bits in LDS
    ("keys", True, 16400, 1, 1, 5, 16385, 64, 0.0),  # one more: read per score
    ("keys_heads", True, 0, 4, 2, 129, 129, 64, 0.2),
    ("bool", True, 0, 2, 2, 63, 64, 64, 0.0),  # four mask bytes per load
    ("bool", False, 0, 2, 1, 70, 131, 128, 0.15),  # one by one
    ("add", False, 0, 4, 4, 96, 128, 64, 0.0),
    ("add", False, 0, 2, 2, 33, 50, 128, 0.1),
]


@pytest.mark.parametrize("kind,causal,offset,hq,hkv,sq,sk,d,p", CASES)
def test_masked_mfma_attention_matches_oracle(kind, causal, offset, hq, hkv, sq, sk, d, p) -> None:
    """Probabilities stay at fp32 precision, so O and dV carry one bf16
    rounding: at most 2^-9 of each element, hence of the norm (bf16
    probabilities would add as much again).  dQ and dK also see delta formed
    from the rounded O: twice that bound.  Keys hidden from every query may
    hold NaN; a row of masks of the lowest value averages over all keys, forward
    and backward."""
    g = torch.Generator().manual_seed(11)
    b = 2
    q, do = (torch.randn(b, hq, sq, d, generator=g).bfloat16() for _ in range(2))
    k, v = (torch.randn(b, hkv, sk, d, generator=g).bfloat16() for _ in range(2))
    mask = None
    if kind == "keys":  # leading, trailing and whole-tile gaps
        mask = torch.rand(b, 1, 1, sk, generator=g) > 0.2
        mask[0, ..., sk // 3:] = False
        mask[1, ..., : sk // 2] = False
    elif kind == "keys_heads":
        mask = torch.rand(b, hq, 1, sk, generator=g) > 0.4
    elif kind == "bool":
        mask = torch.rand(b, 1, sq, sk, generator=g) > 0.3
        mask[1, 0, 3] = False
    elif kind == "add":
        mask = torch.randn(sq, sk, generator=g).bfloat16()
        mask[2, 1:9] = float("-inf")
        mask[1, 4:] = torch.finfo(torch.bfloat16).min
        mask[0] = torch.finfo(torch.bfloat16).min
        mask[4] = float("-inf")
    qr, kr, vr = (t.float().clone().requires_grad_(True) for t in (q, k, v))
    mr = mask.float() if kind == "add" else mask
    if kind == "add":
        # (the oracle's fused CPU backward forms P as exp(x - lse), which is 1 for
        # every key of the row of lowest values: the explicit softmax instead, and
        # zeros for the row of -inf)
        mr[4] = 0.0
        o_ref = _reference(qr.double(), kr.double(), vr.double(), causal, offset, mr, p, 77)
        o_ref = o_ref.index_fill(2, torch.tensor([4]), 0.0)
    else:
        o_ref = R.local_attention(qr, kr, vr, causal=causal, sequence_offset=offset, attention_mask=mr, dropout_p=p,
                                  dropout_seed=77)
    o_ref.backward(do.to(o_ref.dtype))
    if kind == "keys":
        hidden = ~mask[:, :, 0, :, None].expand(b, hkv, sk, d)
        k, v = k.masked_fill(hidden, float("nan")), v.masked_fill(hidden, float("nan"))
    qd, kd, vd = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o = Fn.masked_attention(qd, kd, vd, None if mask is None else mask.cuda(), causal=causal,
                            sequence_offset=offset, dropout_p=p, seed=77)
    o.backward(do.cuda())
    ulp = 2.0 ** -9
    for name, got, exp, bound in (("o", o, o_ref, 1.02 * ulp), ("dv", vd.grad, vr.grad, 1.02 * ulp),
                                  ("dq", qd.grad, qr.grad, 2 * ulp), ("dk", kd.grad, kr.grad, 2 * ulp)):
        assert torch.isfinite(got).all(), name
        if float(exp.detach().abs().max()) < 1e-6:
            # one visible key per query: dS = dO . V - delta vanishes but for the
            # rounding of the O that delta is formed from
            ds = ulp * float((do.float() * o_ref.detach()).abs().sum(-1).max())
            x = max(float(q.float().abs().max()), float(k.float().abs().max()))
            assert float(got.detach().abs().max()) <= 1.02 * ds * x / d ** 0.5 / (1 - p), name
        else:
            assert rel_l2(got, exp) <= bound, (name, rel_l2(got, exp))


@pytest.mark.parametrize("kind", ["keys", "bool", "add"])
@pytest.mark.parametrize("d", [64, 128])
def test_probabilities_keep_their_fp32_bits(kind, d) -> None:
    """Pairs of keys whose scores differ by 2^-12 and whose values are opposite,
    and such pairs of queries: every sum is of differences of 2^-12 of its
    terms, so that two bf16 terms per probability (2^-18 of it in error, 2^-19.5
    in the mean) would show as 2^-7.5 of the results.  The dots are exact in
    fp32 (multiples of 2^-12 below 2^8); a probability within 2^-22 gives 2^-10
    of a result beside its rounding, 2^-9; dQ and dK also see delta from the
    rounded O: twice that."""
    g = torch.Generator().manual_seed(3)
    b, h, n = 1, 2, 96

    def grid(*shape):  # multiples of 1/8 up to 1.5
        return (torch.randint(-12, 13, shape, generator=g) / 8).double()

    def pairs(x, col):
        x = x.repeat_interleave(2, 2)
        x[..., col] = 0
        x[:, :, 1::2, col] = 2.0 ** -9
        return x

    q, k = grid(b, h, n, d), grid(b, h, n, d)
    q[..., 0], k[..., 1] = 1.5, 1.5
    k[:, :, ::2, 1] = -1.5
    q, k = pairs(q, 1), pairs(k, 0)
    v, do = (torch.randn(b, h, n, d, generator=g).bfloat16().double().repeat_interleave(2, 2) for _ in range(2))
    v[:, :, 1::2], do[:, :, 1::2] = -v[:, :, 1::2], -do[:, :, 1::2]
    for t in (q, k):
        assert torch.equal(t, t.bfloat16().double())
    ref = [t.clone().requires_grad_() for t in (q, k, v)]
    o_ref = torch.softmax(ref[0] @ ref[1].transpose(2, 3) / 8, -1) @ ref[2]
    grads = torch.autograd.grad(o_ref, ref, do)
    mask = {"keys": torch.ones(b, 1, 1, 2 * n, dtype=torch.bool), "bool": torch.ones(2 * n, 2 * n, dtype=torch.bool),
            "add": torch.zeros(2 * n, 2 * n, dtype=torch.bfloat16)}[kind]
    dev = [t.bfloat16().cuda().requires_grad_() for t in (q, k, v)]
    o = Fn.masked_attention(*dev, mask.cuda(), causal=False, scale=0.125)
    got = (o, *torch.autograd.grad(o, dev, do.bfloat16().cuda()))
    ulp = 2.0 ** -9
    for name, a, e, bound in zip(("o", "dq", "dk", "dv"), got, (o_ref, *grads), (1.5, 3, 3, 1.5)):
        assert rel_l2(a, e) <= bound * ulp, (name, rel_l2(a, e) / ulp)


HIDDEN = [
    # (dtype, mask, causal, offset, sq, sk, d, p, keys and queries that hold NaN or infinity)
    ("bf16", "none", True, 0, 130, 130, 64, 0.1, [70, 129], []),  # seen by the last queries only
    ("bf16", "none", True, 5, 1, 40, 128, 0.1, list(range(6, 40)), []),  # one query before keys never written
    ("bf16", "bool", True, 0, 100, 100, 64, 0.0, [3, 64, 90], [7]),
    ("bf16", "bool", False, 0, 70, 131, 128, 0.2, [130], [0, 69]),
    ("bf16", "add", False, 0, 66, 96, 64, 0.0, [0, 50], [65]),
    ("bf16", "keys", True, 0, 65, 65, 64, 0.0, [20], [64]),
    ("bf16", "bool", True, 0, 40, 50, 80, 0.0, [3, 17], [7]),
    ("fp32", None, True, 0, 40, 40, 64, 0.0, [20, 39], []),
    ("fp32", None, True, 5, 1, 16, 100, 0.0, list(range(6, 16)), []),
    ("fp32", "none", True, 0, 33, 33, 128, 0.3, [17], [2, 32]),
    ("fp32", "bool", False, 0, 30, 50, 20, 0.0, [3, 40], [29]),
    ("fp32", "add", False, 0, 30, 50, 64, 0.2, [3, 40], [0]),
]


@pytest.mark.parametrize("dtype,kind,causal,offset,sq,sk,d,p,bad_keys,bad_queries", HIDDEN)
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_hidden_rows_may_hold_anything(dtype, kind, causal, offset, sq, sk, d, p, bad_keys, bad_queries, value) -> None:
    """Keys hidden from a query, and queries without a finite score, are not read
    for it: every other query's results and every gradient are those of finite
    data (the bounds of the tests above; fp32: 64 roundings), with the keys
    masked from all queries, from some, or by causality alone."""
    dt, (b, hq, hkv) = (torch.bfloat16 if dtype == "bf16" else torch.float32), (2, 4, 2)
    g = torch.Generator().manual_seed(sq + sk + d)
    q, do = (torch.randn(b, hq, sq, d, generator=g).to(dt) for _ in range(2))
    k, v = (torch.randn(b, hkv, sk, d, generator=g).to(dt) for _ in range(2))
    see = torch.ones(b, 1, sq, sk, dtype=torch.bool)
    mask = None
    if kind == "keys":
        mask = torch.rand(b, 1, 1, sk, generator=g) > 0.2
        mask[..., bad_keys] = False
        see = mask.expand_as(see)
    elif kind in ("bool", "add"):
        see = torch.rand(b, 1, sq, sk, generator=g) > 0.3
        see[..., bad_keys[1:]] = False  # the first one is hidden from some queries
        mask = see if kind == "bool" else torch.randn(b, 1, sq, sk, generator=g).masked_fill(~see, -math.inf).to(dt)
    if causal:
        see = see & (torch.arange(sk)[None] <= offset + torch.arange(sq)[:, None])
    lost = see[..., bad_keys].any(-1).expand(b, hq, sq).clone()  # queries whose result is NaN
    lost[..., bad_queries] = True
    ref = [t.double().requires_grad_() for t in (q, k, v)]
    kr, vr = (t.repeat_interleave(hq // hkv, 1) for t in ref[1:])
    s = ref[0] @ kr.transpose(2, 3) / math.sqrt(d)
    s = (s + mask.double() if kind == "add" else s).masked_fill(~see, -math.inf)
    pr = torch.softmax(s, -1).nan_to_num(0.0)
    if p:
        pr = pr * R.dropout_keep(9, tuple(s.shape), p) / (1 - p)
    o_ref = pr @ vr
    grads = torch.autograd.grad(o_ref, ref, do.double().masked_fill(lost[..., None], 0.0))
    k[:, :, bad_keys], v[:, :, bad_keys] = value, -value
    q[:, :, bad_queries], do[:, :, bad_queries] = value, value
    dev = [t.cuda().requires_grad_() for t in (q, k, v)]
    if kind is None:
        o = Fn.attention(*dev, causal=causal, sequence_offset=offset)
    else:
        o = Fn.masked_attention(*dev, None if mask is None else mask.cuda(), causal=causal, sequence_offset=offset,
                                dropout_p=p, seed=9)
    got = torch.autograd.grad(o, dev, do.cuda())
    if math.isnan(value):
        assert torch.isnan(o.cpu()[lost & see.any(-1)]).all()
    ulp = 2.0 ** -9
    bounds = (1.02 * ulp, 2 * ulp, 2 * ulp, 1.02 * ulp) if dtype == "bf16" else (64 * 2.0 ** -24,) * 4
    keep = ~lost
    pairs = [("o", o.cpu()[keep], o_ref[keep])] + list(zip(("dq", "dk", "dv"), got, grads))
    for (name, a, e), bound in zip(pairs, bounds):
        assert torch.isfinite(a).all(), name
        assert rel_l2(a, e) <= bound if float(e.detach().abs().max()) > 1e-6 else float(a.abs().max()) < 1e-2, name
