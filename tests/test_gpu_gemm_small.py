"""bf16 products of few rows (64 x 64 tiles of csrc/gemm.hip) with each of their epilogues."""

from __future__ import annotations

import pytest
import torch

import nano_megatron_amd.functional as Fn
from nano_megatron_amd import _lib

pytestmark = pytest.mark.gpu


def _bf(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda").bfloat16()


@pytest.mark.parametrize("m", [1, 63, 64, 65, 193])
@pytest.mark.parametrize("n", [8, 64, 72, 1032])
@pytest.mark.parametrize("k", [8, 64, 72, 200, 1032, 2744])
def test_few_rows_match_fp64(m, n, k) -> None:
    """fp32 sums of exact bf16 products and one bf16 rounding: 2^-8 of the value
    plus 2^-24 (2 sqrt(k) + 8) sum |a b| for the sums' order."""
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w, c = _bf(g, m, k), _bf(g, n, k), _bf(g, m, n)
    wt = w.double().t().contiguous()
    exp = a.double() @ wt
    slack = 2.0 ** -24 * (2 * k ** 0.5 + 8) * (a.double().abs() @ wt.abs())
    assert ((Fn.mm(a, w.t()).double() - exp).abs() <= 2.0 ** -8 * exp.abs() + slack).all()
    exp = exp + c.double()
    got = Fn.mm(a, w.t(), c=c, beta=1.0)
    assert ((got.double() - exp).abs() <= 2.0 ** -8 * exp.abs() + 2 * slack + 2.0 ** -22 * c.double().abs()).all()
    out = torch.full((m, n), 3.0, device="cuda")
    Fn.mm_f32out(a, w.t(), out, alpha=0.5, beta=2.0)
    exp = 0.5 * (exp - c.double()) + 6.0
    assert ((out.double() - exp).abs() <= slack + 2.0 ** -22 * (exp.abs() + 6.0)).all()


@pytest.mark.parametrize("m", [1, 65, 193])
@pytest.mark.parametrize("k", [64, 200, 1024])
def test_few_rows_epilogues_match_the_large_tiles(m, k) -> None:
    """Rows of a product do not depend on each other and every tile sums K in the
    same order, so the first rows of a product of 8,192 give the bits."""
    g = torch.Generator(device="cuda").manual_seed(m + k)
    a = _bf(g, 8192, k)
    few = a[:m].contiguous()
    ang = torch.rand(8192, 32, generator=g, device="cuda")
    wq = _bf(g, 6 * 64, k)
    big, small = (Fn.mm_rope(x, wq.t(), seq=x.shape[0], head_dim=64, rope_cols=4 * 64, cos=ang.cos(), sin=ang.sin())
                  for x in (a, few))
    assert torch.equal(big[:m], small)
    wgu = _bf(g, 2 * 264, k)
    big, small = (Fn.mm_gate_up(x, wgu, act=True, gu=True) for x in (a, few))
    assert torch.equal(big[0][:m], small[0]) and torch.equal(big[1][:m], small[1])
    gu, wd = small[1], _bf(g, k, 264)
    dy, wdt = _bf(g, m, k), wd.t().contiguous()  # Wd^T: K-contiguous rows of 264 columns
    exp = Fn.mm_swiglu_bwd(dy, wd, gu)
    dgu, act = torch.empty_like(exp[0]), torch.empty_like(exp[1])
    _lib.call("nmb_gemm_bf16_swiglu_bwd", 0, m, 264, k, dy.data_ptr(), k, wdt.data_ptr(), k, gu.data_ptr(), 528,
              dgu.data_ptr(), 528, act.data_ptr(), 264, _lib.stream_of(dy))
    assert torch.equal(dgu, exp[0]) and torch.equal(act, exp[1])
