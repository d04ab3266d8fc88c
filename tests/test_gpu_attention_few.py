"""bf16 attention forward on workgroups of 64 queries (few queries): edges of the tiles, blocks and masks."""

from __future__ import annotations

import pytest
import torch

import nano_megatron_amd.functional as Fn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("sq", [1, 15, 16, 63, 64, 65, 193])
@pytest.mark.parametrize("causal,blocks,offset", [(True, 1, 0), (False, 1, 0), (True, 2, 0), (True, 2, 193),
                                                  (True, 1, -20), (False, 2, 0)])
def test_few_queries_match_the_large_workgroups(d, sq, causal, blocks, offset) -> None:
    """Queries do not depend on each other and see their keys in the same order
    whatever the workgroup, so a few of them give the bits of the same ones in a
    launch over 256 batches (which runs the large workgroups); and the fp64
    softmax to bf16's rounding: P and O each 2^-8 of the largest value."""
    sk, h, hkv, batches = 193, 4, 2, 256
    g = torch.Generator(device="cuda").manual_seed(sq + d)
    rnd = lambda s, n: torch.randn(1, s, n, d, generator=g, device="cuda").bfloat16()  # noqa: E731
    q, ks, vs = rnd(sq, h), [rnd(sk, hkv) for _ in range(blocks)], [rnd(sk, hkv) for _ in range(blocks)]
    many = lambda t: t.expand(batches, -1, -1, -1).contiguous()  # noqa: E731
    args = dict(causal=causal, q_offset=offset, scale=None)
    offs = tuple(sk * i for i in range(blocks))
    o, lse = Fn.attn_fwd_bshd(q, ks, vs, offs, **args)
    ob, lb = Fn.attn_fwd_bshd(many(q), [many(t) for t in ks], [many(t) for t in vs], offs, **args)
    assert torch.equal(o[0], ob[0]) and torch.equal(lse[0], lb[0])
    k, v = (torch.cat(t, 1)[0].double().repeat_interleave(h // hkv, 1).transpose(0, 1).contiguous() for t in (ks, vs))
    s = q[0].double().transpose(0, 1).contiguous() @ k.transpose(1, 2).contiguous() / d ** 0.5
    if causal:
        hidden = torch.arange(sk * blocks, device="cuda")[None] > offset + torch.arange(sq, device="cuda")[:, None]
        s = s.masked_fill(hidden, float("-inf"))
    exp = torch.softmax(s, -1).nan_to_num(0.0) @ v  # a query that sees no key gives zeros
    bound = 2.0 ** -7 * v.abs().amax()
    assert ((o[0].double().transpose(0, 1) - exp).abs() <= bound).all()
