"""The K loop of the 256-row GEMM tiles: few K tiles, partial ones and the fused pair of products."""

from __future__ import annotations

import pytest
import torch

import nano_megatron_amd.functional as Fn
from nano_megatron_amd import _lib

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


@pytest.mark.parametrize("m,n", [(40, 72), (296, 3000), (4096, 4096)])
@pytest.mark.parametrize("la,lb", [(0, 0), (0, 1), (1, 1)])
def test_no_k_gives_beta_c(m, n, la, lb) -> None:
    """K = 0: the product is zero, D = beta C, on every tile shape (the C entry
    points take it; a product of NaN runs first, whose values LDS may still hold)."""
    stream = torch.cuda.current_stream().cuda_stream
    nan = torch.full((512, 512), float("nan"), device="cuda", dtype=torch.bfloat16)
    c = torch.randn(m, n, device="cuda").bfloat16()
    a, b = torch.ones(m, 8, device="cuda").bfloat16(), torch.ones(n, 8, device="cuda").bfloat16()
    lda, ldb = (8 if la == 0 else m), (8 if lb == 0 else n)
    for beta in (0.0, 1.0):
        Fn.mm(nan, nan.t())
        d = torch.full_like(c, 5.0)
        _lib.call("nmb_gemm_bf16", la, lb, m, n, 0, 1.0, a.data_ptr(), lda, b.data_ptr(), ldb, beta,
                  c.data_ptr() if beta else None, n, d.data_ptr(), n, None, 0, stream)
        assert torch.equal(d, c * beta)
        d32 = torch.full((m, n), 3.0, device="cuda")
        _lib.call("nmb_gemm_bf16_f32out", la, lb, m, n, 0, 1.0, a.data_ptr(), lda, b.data_ptr(), ldb, beta,
                  d32.data_ptr(), n, None, 0, stream)
        assert (d32 == 3.0 * beta).all()


@pytest.mark.parametrize("m,f", [(40, 72), (512, 4096)])
def test_no_k_in_the_fused_products(m, f) -> None:
    """K = 0 with the RoPE, SwiGLU and SwiGLU backward epilogues: zero products."""
    stream = torch.cuda.current_stream().cuda_stream
    bf = dict(device="cuda", dtype=torch.bfloat16)
    nan = torch.full((512, 512), float("nan"), **bf)
    x, w = torch.ones(m, 8, **bf), torch.ones(2 * f, 8, **bf)
    ang = torch.rand(m, 32, device="cuda")
    cos, sin = ang.cos(), ang.sin()
    Fn.mm(nan, nan.t())
    d = torch.full((m, 128), 5.0, **bf)
    _lib.call("nmb_gemm_bf16_rope", 0, m, 128, 0, x.data_ptr(), 8, w.data_ptr(), 8, d.data_ptr(), 128,
              cos.data_ptr(), sin.data_ptr(), m, None, 0, 0, m, 64, 64, stream)
    assert (d == 0).all()
    act, gu = torch.full((m, f), 5.0, **bf), torch.full((m, 2 * f), 5.0, **bf)
    Fn.mm(nan, nan.t())
    _lib.call("nmb_gemm_bf16_swiglu", m, f, 0, x.data_ptr(), 8, w.data_ptr(), 8, act.data_ptr(), f, gu.data_ptr(),
              2 * f, stream)
    assert (act == 0).all() and (gu == 0).all()
    gu = torch.randn(m, 2 * f, device="cuda").bfloat16()
    for lb, ldb in ((0, 8), (1, f)):
        dgu = torch.full_like(gu, 5.0)
        Fn.mm(nan, nan.t())
        _lib.call("nmb_gemm_bf16_swiglu_bwd", lb, m, f, 0, x.data_ptr(), 8, w.data_ptr(), ldb, gu.data_ptr(), 2 * f,
                  dgu.data_ptr(), 2 * f, act.data_ptr(), f, stream)
        assert (dgu == 0).all() and torch.equal(act, Fn.swiglu_fwd(gu[:, :f], gu[:, f:]))
        # the fused pair: no gate / up product (K1 = 0) before a ds of 8 x 1
        dy, wd = torch.ones(m, 8, **bf), torch.ones(f * 8, **bf)
        Fn.mm(nan, nan.t())
        _lib.call("nmb_gemm_bf16_gate_up_swiglu_bwd", m, f, 0, x.data_ptr(), 8, w.data_ptr(), 8, 8, dy.data_ptr(), 8,
                  lb, wd.data_ptr(), ldb, dgu.data_ptr(), 2 * f, act.data_ptr(), f, stream)
        assert (dgu == 0).all() and (act == 0).all()
