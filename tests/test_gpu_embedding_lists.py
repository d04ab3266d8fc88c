"""The embedding backward through its token lists, at the edges of lists, row
groups and column chunks."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import nano_megatron_amd.functional as Fn
from nano_megatron_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tokens,vocab,hidden", [(1, 1, 8), (64, 512, 128), (65, 17, 136), (8192, 513, 256),
                                                 (8193, 1025, 120), (20000, 3000, 64), (600, 50257, 264)])
@pytest.mark.parametrize("tied", [False, True])
def test_listed_tokens_are_added_in_order(dtype, tokens, vocab, hidden, tied) -> None:
    """A hot id over half the tokens (runs of more than a 64-entry step), ids
    outside the table, rows without tokens: every row equals the sequential fp32
    sum in token order, rounded, plus the tied gradient, bit for bit; so does
    the entry without lists."""
    g = torch.Generator(device="cuda").manual_seed(tokens + vocab)
    ids = torch.randint(0, vocab, (tokens,), generator=g, device="cuda")
    ids[torch.rand(tokens, generator=g, device="cuda") < 0.5] = vocab // 2
    if tokens > 8:
        ids[3], ids[5] = -1, vocab
    dout = torch.randn(tokens, hidden, generator=g, device="cuda").to(dtype)
    lm = torch.randn(vocab, hidden, generator=g, device="cuda").to(dtype) if tied else None
    tie = Fn.TiedGrad()
    tie.grad = lm
    table = torch.zeros(vocab, hidden, dtype=dtype, device="cuda", requires_grad=True)
    (got,) = torch.autograd.grad(Fn.embedding(table, ids, tie), table, dout)
    plain = torch.empty_like(got)
    _lib.call("nmb_embedding_bwd", dout.data_ptr(), ids.data_ptr(), _lib.ptr(lm), plain.data_ptr(), tokens, vocab,
              hidden, _lib.dtype_code(dtype), _lib.stream_of(dout))
    assert torch.equal(got, plain)
    host, rows = ids.cpu().numpy(), dout.float().cpu().numpy()
    exp = np.zeros((vocab, hidden), np.float32)
    for v in np.unique(host[(host >= 0) & (host < vocab)]):
        exp[v] = np.add.accumulate(rows[host == v], axis=0, dtype=np.float32)[-1]
    exp = torch.from_numpy(exp).to(dtype)
    if tied:
        exp = (exp.float() + lm.cpu().float()).to(dtype)
    assert torch.equal(got.cpu(), exp)


@pytest.mark.parametrize("entry,tokens", [("nmb_embedding_bwd_ws", 64), ("nmb_embedding_bwd_ws", 300),
                                          ("nmb_embedding_bwd", 30), ("nmb_embedding_bwd", 192), ("nmb_embedding_bwd", 300)])
@pytest.mark.parametrize("vocab", [17, 8190, 50257])
def test_repeated_ids_past_the_table_write_nothing(entry, tokens, vocab) -> None:
    """More than 24 tokens of one id (the rows a whole workgroup adds up) at and
    past a table that ends inside a workgroup's 16 rows: the rows behind the
    table gradient stay as they were, and the table's are the other tokens'."""
    hidden, band = 64, 32
    g = torch.Generator(device="cuda").manual_seed(vocab + tokens)
    ids = torch.full((tokens,), vocab, device="cuda")
    ids[::10] = vocab + 1
    ids[0], ids[-1] = vocab - 1, vocab - 1
    assert int((ids == vocab).sum()) > 24
    dout = torch.randn(tokens, hidden, generator=g, device="cuda")
    out = torch.full((vocab + band, hidden), 7.0, device="cuda")
    nbytes = _lib.ctypes.c_int64()
    _lib.call("nmb_embedding_bwd_workspace_bytes", tokens, vocab, _lib.ctypes.byref(nbytes))
    ws = torch.empty(max(nbytes.value, 16), dtype=torch.uint8, device="cuda")
    extra = (ws.data_ptr(), nbytes.value) if entry.endswith("_ws") else ()
    _lib.call(entry, dout.data_ptr(), ids.data_ptr(), None, out.data_ptr(), tokens, vocab, hidden, *extra,
              _lib.dtype_code(torch.float32), _lib.stream_of(dout))
    assert (out[vocab:] == 7.0).all()
    assert (out[: vocab - 1] == 0).all()
    assert torch.equal(out[vocab - 1], dout[0] + dout[-1])


@pytest.mark.parametrize("first", [961, 970, 1024])
def test_frequent_rows_whose_last_gather_is_empty(first) -> None:
    """A row's tokens are gathered up to 1,024 at a time and a gather stops past
    960: with 961 to 1,024 tokens, all in the first 8,192, the second gather of
    the row finds nothing.  Seven more frequent rows of the same 16 follow."""
    tokens, vocab, hidden = 2 * 8192, 64, 264
    g = torch.Generator(device="cuda").manual_seed(first)
    ids = torch.full((tokens,), vocab - 1, device="cuda")
    ids[:first] = 16
    for i, n in enumerate((40, 100, 970, 1000, 1500, 65, 30)):
        at = 1100 + 1600 * i
        ids[at: at + n] = 18 + 2 * i
    dout = torch.randn(tokens, hidden, generator=g, device="cuda")
    table = torch.zeros(vocab, hidden, device="cuda", requires_grad=True)
    (got,) = torch.autograd.grad(Fn.embedding(table, ids, None), table, dout)
    host, rows = ids.cpu().numpy(), dout.cpu().numpy()
    exp = np.zeros((vocab, hidden), np.float32)
    for v in np.unique(host):
        exp[v] = np.add.accumulate(rows[host == v], axis=0, dtype=np.float32)[-1]
    assert np.array_equal(got.cpu().numpy(), exp)
