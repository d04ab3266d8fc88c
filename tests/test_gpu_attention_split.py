"""The dK/dV kernel with its query streams divided over several workgroups."""

from __future__ import annotations

import ctypes

import pytest
import torch

import nano_megatron_amd as nm
import nano_megatron_amd.functional as Fn
from nano_megatron_amd import _lib

pytestmark = pytest.mark.gpu


def _undivided(q, ks, vs, offs, o, do, lse, causal, q_offset):
    """nmb_attn_bwd with the smaller workspace, which has no room for partial sums."""
    b, sq, hq, d = q.shape
    _, sk, hkv, _ = ks[0].shape
    dq, dks, dvs = torch.empty_like(q), [torch.empty_like(k) for k in ks], [torch.empty_like(v) for v in vs]
    nbytes = ctypes.c_size_t(0)
    _lib.call("nmb_attn_bwd_workspace_bytes", b, hq, sq, ctypes.byref(nbytes))
    ws = torch.empty(nbytes.value, dtype=torch.uint8, device=q.device)
    ptrs = lambda ts: _lib.ptr_array(t.data_ptr() for t in ts)  # noqa: E731
    st = lambda t: _lib.i64x3(Fn._eff_strides(t))  # noqa: E731
    _lib.call("nmb_attn_bwd", q.data_ptr(), ptrs(ks), ptrs(vs), _lib.i64_array(offs), len(ks), o.data_ptr(),
              do.data_ptr(), lse.data_ptr(), dq.data_ptr(), ptrs(dks), ptrs(dvs), ws.data_ptr(), ws.numel(), b, hq,
              hkv, sq, sk, d, st(q), st(ks[0]), st(o), int(causal), q_offset, 0.0, _lib.NMB_BF16, _lib.stream_of(q))
    return dq, dks, dvs


@pytest.mark.parametrize("b,hq,hkv,sq,sk,d,nblk,causal,q_off", [
    (1, 16, 2, 100, 100, 64, 1, True, 0),      # two tiles per workgroup
    (1, 4, 1, 64, 320, 64, 1, True, 0),        # key tiles that no query sees
    (2, 4, 2, 1000, 1000, 64, 1, True, 0),     # streams shorter than the splits at the last keys
    (2, 16, 4, 700, 700, 128, 1, True, 0),
    (1, 8, 2, 300, 129, 128, 3, True, 258),    # several K/V blocks
    (1, 8, 2, 1029, 257, 128, 1, False, 0),
    (1, 3, 3, 3000, 60, 64, 1, False, 0),
])
def test_divided_streams_match_undivided(b, hq, hkv, sq, sk, d, nblk, causal, q_off) -> None:
    """The same fp32 terms summed in another order, then one bf16 rounding: at
    most one bf16 step (2^-7 of the value) apart, plus 2^-20 of the largest sum
    for the order.  The RoPE variant equals the plain one rotated afterwards,
    bit for bit."""
    g = torch.Generator(device="cuda").manual_seed(4)
    rnd = lambda s, h: torch.randn(b, s, h, d, generator=g, device="cuda").bfloat16()  # noqa: E731
    size = ctypes.c_size_t(0)
    _lib.call("nmb_attn_bwd_workspace_bytes_split", b, hq, hkv, sq, sk, d, nblk, _lib.NMB_BF16, ctypes.byref(size))
    assert size.value > 8 * b * hq * sq  # these shapes are divided
    q, do = rnd(sq, hq), rnd(sq, hq)
    ks, vs = [rnd(sk, hkv) for _ in range(nblk)], [rnd(sk, hkv) for _ in range(nblk)]
    offs = tuple(sk * i for i in range(nblk))
    o, lse = Fn.attn_fwd_bshd(q, ks, vs, offs, causal=causal, q_offset=q_off, scale=None)
    ref = _undivided(q, ks, vs, offs, o, do, lse, causal, q_off)
    dq, dks, dvs = torch.empty_like(q), [torch.empty_like(k) for k in ks], [torch.empty_like(v) for v in vs]
    Fn.attn_bwd_bshd(q, ks, vs, offs, o, do, lse, dq, dks, dvs, causal=causal, q_offset=q_off, scale=None)
    assert torch.equal(dq, ref[0])
    for a, r in zip(dks + dvs, ref[1] + ref[2]):
        a, r = a.double(), r.double()
        assert ((a - r).abs() <= 2.0 ** -7 * r.abs() + 2.0 ** -20 * r.abs().max()).all()
    if nblk == 1 and sq == sk:
        tab = nm.RotaryEmbedding(d).tables(q.device, sq)
        dq2, dk2, dv2 = torch.empty_like(q), torch.empty_like(ks[0]), torch.empty_like(vs[0])
        Fn.attn_bwd_rope_bshd(q, ks[0], vs[0], o, do, lse, dq2, dk2, dv2, causal=causal, q_offset=q_off, scale=None,
                              cos=tab.cos, sin=tab.sin)
        Fn.rope_apply(dks[0], dks[0], tab.cos, tab.sin, inverse=True)
        assert torch.equal(dk2, dks[0]) and torch.equal(dv2, dvs[0])
