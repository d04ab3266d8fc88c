"""bf16 products over the plans of csrc/gemm.hip: every tile configuration, with
and without a K split, at sizes with remainders in all three dimensions."""

from __future__ import annotations

import ctypes

import pytest
import torch

import nano_megatron_amd.functional as Fn
from nano_megatron_amd import _lib

pytestmark = pytest.mark.gpu

SHAPES = [  # (m, n, k, split?): M and N off the tiles, K off the K tile and the split
    (1003, 2056, 5640, True),   # 256 x 128, split
    (2001, 2056, 11272, True),  # 256 x 256, split
    (193, 1032, 1000, False),   # NT: 64 x 64; the others: 128 x 128, split
    (50, 1024, 2744, True),     # NT: 64 x 64, split
    (2127, 1032, 1032, False),  # 128 x 128, one workgroup per CU
    (5501, 1024, 2744, False),  # 256 x 128
    (2056, 4104, 2056, False),  # 256 x 256
    (8, 8, 8, False),
]


@pytest.mark.parametrize("m,n,k,split", SHAPES)
@pytest.mark.parametrize("layout", ["NT", "NN", "TN"])
def test_planned_products_match_fp64(m, n, k, split, layout) -> None:
    """fp32 sums of exact bf16 products and one bf16 rounding: 2^-8 of the value
    plus 2^-24 (2 sqrt(k) + 8) sum |a b| for the sums' order; twice the same
    call gives the same bits; beta adds C before the rounding."""
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    bf = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()  # noqa: E731
    if layout[0] == "T":
        m = (m + 7) // 8 * 8  # the contiguous extent of a transposed A
    a = bf(m, k) if layout[0] == "N" else bf(k, m).t()
    b = bf(n, k).t() if layout[1] == "T" else bf(k, n)
    c = bf(m, n)
    if layout == "NT":
        size = ctypes.c_int64()
        _lib.call("nmb_gemm_bf16_workspace_bytes", 0, 0, m, n, k, ctypes.byref(size))
        assert (size.value > 0) == split
    exp = a.double() @ b.double()
    slack = 2.0 ** -24 * (2 * k ** 0.5 + 8) * (a.double().abs() @ b.double().abs())
    got = Fn.mm(a, b)
    assert ((got.double() - exp).abs() <= 2.0 ** -8 * exp.abs() + slack).all()
    assert torch.equal(got, Fn.mm(a, b))
    exp = exp + c.double()
    got = Fn.mm(a, b, c=c, beta=1.0)
    assert ((got.double() - exp).abs() <= 2.0 ** -8 * exp.abs() + 2 * slack + 2.0 ** -22 * c.double().abs()).all()
