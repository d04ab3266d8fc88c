"""The K loop of the 256-row GEMM tiles: few K tiles, partial ones and the fused pair of products."""

from __future__ import annotations

import pytest
import torch

import nano_megatron_amd.functional as Fn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(4096, 4096), (8192, 1024), (4090, 4104)])
@pytest.mark.parametrize("k", [8, 64, 72, 128, 136, 192, 200, 264, 512])
@pytest.mark.parametrize("at,bt", [(False, True), (False, False), (True, False), (True, True)])
def test_gemm_k_tiles(m, n, k, at, bt) -> None:
    """One to eight 64-deep K tiles, whole and partial, with two and three
    stages in flight and every operand layout.  Bound: the bf16 rounding of the
    result, 2^-8 of it, and k fp32 additions, 2^-23 k sum |a b| / sqrt(k)
    (products of bf16 are exact in fp32)."""
    m = m if not at else m // 8 * 8
    g = torch.Generator(device="cuda").manual_seed(m + n + k)

    def operand(rows, cols, transposed):
        r, c = (cols, rows) if transposed else (rows, cols)
        t = torch.randn(r, c, generator=g, device="cuda").bfloat16()
        return t.t() if transposed else t

    a, b = operand(m, k, at), operand(k, n, bt)
    out = Fn.mm(a, b)
    af, bf = a.float().contiguous(), b.float().contiguous()
    exp = af @ bf
    bound = 2.0 ** -8 * exp.abs() + 2.0 ** -23 * (k ** 0.5 + 4) * (af.abs() @ bf.abs())
    assert ((out.float() - exp).abs() <= bound).all()
    assert torch.equal(Fn.mm(a, b), out)


@pytest.mark.parametrize("k1", [64, 128, 192, 256, 320])
@pytest.mark.parametrize("k2", [64, 128, 200])
def test_gate_up_swiglu_backward_k_tiles(k1, k2) -> None:
    """The fused gate/up backward (its second product's first loads go out in the
    first one's last K tile) gives the bits of the two products one by one."""
    m, f = 300, 264
    g = torch.Generator(device="cuda").manual_seed(k1 + k2)
    x, wgu, dy, wd = (torch.randn(*s, generator=g, device="cuda").bfloat16()
                      for s in ((m, k1), (2 * f, k1), (m, k2), (k2, f)))
    _, gu = Fn.mm_gate_up(x, wgu, act=False, gu=True)
    exp = Fn.mm_swiglu_bwd(dy, wd, gu)
    for _ in range(3):
        out = Fn.mm_gate_up_swiglu_bwd(x, wgu, dy, wd)
        assert torch.equal(out[0], exp[0]) and torch.equal(out[1], exp[1])
