"""The fp32 GEMM's tile edges, split K range and unaligned operands, against fp64."""

from __future__ import annotations

import pytest
import torch

import nano_megatron_amd.functional as Fn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(64, 64, 32), (64, 64, 127), (64, 64, 128), (65, 63, 161), (128, 64, 2049),
                                   (1, 1, 4096), (512, 4096, 96), (7, 4098, 640)])
@pytest.mark.parametrize("at,bt", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("shift", [0, 1])
def test_gemm_f32_tiles_and_splits(m, n, k, at, bt, shift) -> None:
    """Around one K tile (32), the first split (128), remainders of both and the
    most splits, with every operand layout; shift 1 puts operands and output at
    bases and strides that are no multiples of 16 bytes.  Bound: the recursive
    sum of k products, 2^-24 (k + 2) sum |a b|, which for these k is far above
    what the MFMA's order gives; 2^-24 (2 sqrt(k) + 8) of the same is used."""
    g = torch.Generator(device="cuda").manual_seed(m + 3 * n + 5 * k)

    def operand(rows, cols, transposed):
        r, c = (cols, rows) if transposed else (rows, cols)
        t = torch.randn(r, c + shift, generator=g, device="cuda")[:, shift:]
        return t.t() if transposed else t

    a, b = operand(m, k, at), operand(k, n, bt)
    c = torch.randn(m, n + shift, generator=g, device="cuda")[:, shift:]
    out = torch.full((m, n + 2 * shift), 7.0, device="cuda")[:, shift:shift + n]
    Fn.mm(a, b, out=out, c=c, alpha=0.5, beta=2.0)
    exp = 0.5 * (a.double() @ b.double()) + 2.0 * c.double()
    bound = 2.0 ** -24 * ((2 * k ** 0.5 + 8) * (a.double().abs() @ b.double().abs()) + 4 * c.double().abs())
    assert ((out.double() - exp).abs() <= bound).all()
    first = out.clone()
    Fn.mm(a, b, out=out, c=c, alpha=0.5, beta=2.0)
    assert torch.equal(out, first)
