"""The fp32 matrix-core attention kernels at their edges, against fp64: 16-row
tiles and remainders, head dims below, at and between 64 and 128, 16-byte and
element loads, several K/V blocks, masks, dropout and rows with nothing visible."""

from __future__ import annotations

import math

import pytest
import torch

import nano_megatron_amd.functional as Fn
from oracle import reference as R

pytestmark = pytest.mark.gpu


def _reference(q, k, v, causal, offset, mask, p, seed):
    """fp64 attention with the oracle's masks; rows without a visible key give zeros."""
    group = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(group, 1), v.repeat_interleave(group, 1)
    s = q @ k.transpose(2, 3) / math.sqrt(q.shape[-1])
    if mask is not None:
        s = s.masked_fill(~mask, -math.inf) if mask.dtype == torch.bool else s + mask.double()
    if causal:
        pos = offset + torch.arange(q.shape[2])[:, None]
        s = s.masked_fill(torch.arange(k.shape[2])[None] > pos, -math.inf)
    pr = torch.softmax(s, -1).nan_to_num(0.0)
    if p:
        pr = pr * R.dropout_keep(seed, tuple(s.shape), p) / (1 - p)
    return pr @ v


@pytest.mark.parametrize("causal,offset,kind,hq,hkv,sq,sk,d,p", [
    (True, 0, None, 2, 2, 1, 1, 1, 0.0),
    (True, 0, None, 4, 2, 16, 16, 64, 0.0),
    (True, 5, None, 4, 1, 17, 67, 66, 0.0),  # no 16-byte rows at head dim 66
    (False, 0, None, 2, 2, 130, 33, 128, 0.3),
    (True, -3, None, 2, 2, 40, 200, 20, 0.0),  # the first three queries see no key
    (True, 0, "bool", 2, 2, 65, 64, 100, 0.2),
    (False, 0, "add", 2, 1, 31, 49, 64, 0.0),
])
def test_fp32_attention_matches_fp64(causal, offset, kind, hq, hkv, sq, sk, d, p) -> None:
    """Every element within 2^-24 times 64 of the scale of its tensor (dots of up
    to 128 terms and sums of up to 200 in fp32, an exponential and a division)."""
    g = torch.Generator().manual_seed(5)
    q, do = (torch.randn(2, hq, sq, d, generator=g) for _ in range(2))
    k, v = (torch.randn(2, hkv, sk, d, generator=g) for _ in range(2))
    mask = None
    if kind == "bool":
        mask = torch.rand(2, 1, sq, sk, generator=g) > 0.3
        mask[0, 0, 7] = False
        mask[1, 0, :, 20:36] = False
    elif kind == "add":
        mask = torch.randn(sq, sk, generator=g)
        mask[3, :40] = -math.inf
        mask[5] = torch.finfo(torch.float32).min
    ref = [t.double().requires_grad_() for t in (q, k, v)]
    o_ref = _reference(*ref, causal, offset, mask, p, 9)
    grads = torch.autograd.grad(o_ref, ref, do.double())
    dev = [t.cuda().requires_grad_() for t in (q, k, v)]
    if kind is None and not p:
        o = Fn.attention(*dev, causal=causal, sequence_offset=offset)
    else:
        o = Fn.masked_attention(*dev, None if mask is None else mask.cuda(), causal=causal,
                                sequence_offset=offset, dropout_p=p, seed=9)
    got = (o, *torch.autograd.grad(o, dev, do.cuda()))
    for name, a, b in zip(("o", "dq", "dk", "dv"), got, (o_ref, *grads)):
        scale = max(float(b.detach().abs().max()), float(do.abs().max()) / 16)
        assert float((a.detach().cpu().double() - b.detach()).abs().max()) <= 64 * 2.0 ** -24 * scale, name


def test_fp32_ring_attention_blocks_match_fp64() -> None:
    """Four K/V blocks of 37 keys (three 16-key tiles, so the waves' turns shift
    from block to block) against attention over their concatenation."""
    g = torch.Generator().manual_seed(6)
    q, do = (torch.randn(1, 4, 37, 64, generator=g) for _ in range(2))
    blocks = [tuple(torch.randn(1, 2, 37, 64, generator=g) for _ in range(2)) for _ in range(4)]
    ref = [q.double().requires_grad_()] + [torch.cat([b[i] for b in blocks], 2).double().requires_grad_()
                                           for i in (0, 1)]
    o_ref = _reference(*ref, True, 111, None, 0.0, 0)
    dq, dk, dv = torch.autograd.grad(o_ref, ref, do.double())
    qd = q.cuda().requires_grad_()
    kv = [tuple(t.cuda().requires_grad_() for t in b) for b in blocks]
    o = Fn.ring_attention(qd, kv, [37 * i for i in range(4)], query_offset=111)
    flat = [t for b in kv for t in b]
    gq, *gkv = torch.autograd.grad(o, [qd, *flat], do.cuda())
    pairs = [(o, o_ref), (gq, dq), (torch.cat(gkv[0::2], 2), dk), (torch.cat(gkv[1::2], 2), dv)]
    for a, b in pairs:
        b = b.detach()
        assert float((a.detach().cpu().double() - b).abs().max()) <= 64 * 2.0 ** -24 * float(b.abs().max())


def test_keys_hidden_from_every_query_may_hold_nan() -> None:
    """bf16 at head dim 80 takes these kernels too; NaN in padded keys does not
    reach the visible ones' results."""
    g = torch.Generator().manual_seed(7)
    q, k, v, do = (torch.randn(2, 2, 50, 80, generator=g).bfloat16() for _ in range(4))
    mask = torch.ones(2, 1, 1, 50, dtype=torch.bool)
    mask[0, ..., 23:] = False
    ref = [t.double().requires_grad_() for t in (q, k, v)]
    o_ref = _reference(*ref, True, 0, mask, 0.0, 0)
    grads = torch.autograd.grad(o_ref, ref, do.double())
    k[0, :, 23:], v[0, :, 23:] = float("nan"), float("nan")
    dev = [t.cuda().requires_grad_() for t in (q, k, v)]
    o = Fn.masked_attention(*dev, mask.cuda(), causal=True)
    got = (o, *torch.autograd.grad(o, dev, do.cuda()))
    for a, b in zip(got, (o_ref, *grads)):
        err = (a.detach().cpu().double() - b.detach()).norm() / b.detach().norm()
        assert float(err) <= 2.0 ** -8  # bf16 results, delta from the rounded o
