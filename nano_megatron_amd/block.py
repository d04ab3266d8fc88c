"""The GPT transformer block as two autograd Functions: checkpointed and eager.

Both run the same device sequence (reference GPTLayer.forward,
models/gpt/layer.py:91-137):

    n1 = RMSNorm(x)                          nmb_rmsnorm_fwd
    [q|k|v] = n1 [Wq;Wk;Wv]^T, RoPE(q, k)    nmb_gemm_bf16_rope (RoPE in the epilogue)
    o, lse = attention(q, k, v)              nmb_attn_fwd (MFMA, online softmax)
    h = x + o Wo^T                           nmb_gemm_bf16 with the residual as C input
    n2 = RMSNorm(h)                          nmb_rmsnorm_fwd
    s = silu(n2 Wg^T) * (n2 Wu^T)            nmb_gemm_bf16_swiglu (activation in the epilogue)
    y = h + s Wd^T                           nmb_gemm_bf16 with the residual as C input

enqueued by one call into csrc/block.hip (two for the backward).

``CheckpointedBlockFunction`` is the full-recompute policy of
``activation_checkpoint`` (nn/activation_checkpoint.py:73-100, selected by
models/gpt/model.py:162-170, 215-233): it saves only the block input x.  Its
backward re-runs the sequence above with the same kernels and shapes (so the
recomputed tensors, the attention output and its lse included, are
bit-identical to the forward's) up to n2, and never re-runs the down
projection, whose output the backward does not need.  The gate/up product is
recomputed inside the MLP backward's GEMM (``nmb_gemm_bf16_gate_up_swiglu_bwd``:
per output tile [g|u] = n2 [Wg;Wu]^T, ds = dY Wd and the SwiGLU backward with
all three in registers, the same bits as the forward's gate/up product
followed by the SwiGLU backward; neither [g|u] nor ds reaches memory), which
re-emits s for the Wd gradient.  A block that keeps [g|u] (no checkpoint)
runs the down projection's backward GEMM with the SwiGLU backward as its
epilogue instead (``nmb_gemm_bf16_swiglu_bwd``).  With ``offload`` the saved input goes to
pinned host memory (the reference's saved-tensor offload,
nn/activation_checkpoint.py:24-41); the weights are parameters, never copied.
``EagerBlockFunction`` (activation_checkpoint.mode = "none") keeps the
intermediates instead and shares the backward; ``SelectiveBlockFunction``
("selective") keeps the sub-block inputs and recomputes only the checkpointed
sub-blocks' products.
"""

from __future__ import annotations

import weakref
from dataclasses import dataclass
from typing import Any, Callable

import torch
from torch import Tensor

from nano_megatron_amd import _lib
from nano_megatron_amd import functional as Fn


@dataclass(frozen=True)
class BlockMeta:
    heads: int
    kv_heads: int
    head_dim: int
    eps: float
    sequence_offset: int  # query offset of the causal mask (models/gpt/attention.py:199-206)
    cos: Tensor          # fp32 [n_pos, head_dim/2]
    sin: Tensor
    positions: Tensor | None  # int32 [S] or [B,S], or None for rope_offset + arange
    rope_offset: int | None = None  # RoPE position of token 0 without positions (default: sequence_offset)
    keep: bool = True    # False: no backward will follow (gradients are off), so nothing is kept for one

    @property
    def pos_offset(self) -> int:
        return self.sequence_offset if self.rope_offset is None else self.rope_offset


def _adjacent(ws: tuple[Tensor, ...]) -> bool:
    """True if the row blocks ws[0], ws[1], ... lie back to back in memory."""
    w0 = ws[0]
    ptr = w0.data_ptr()
    for w in ws:
        if (w.data_ptr() != ptr or not w.is_contiguous() or w.dtype != w0.dtype or w.device != w0.device
                or w.shape[1:] != w0.shape[1:]):
            return False
        ptr += w.numel() * w.element_size()
    return True


def pack_adjacent(params) -> None:
    """Re-home parameters as adjacent row blocks of one buffer (values and
    Parameter objects unchanged), so the fused projections read them in place."""
    ws = tuple(p.data for p in params)
    if _adjacent(ws):
        return
    buf = torch.empty(sum(w.shape[0] for w in ws), *ws[0].shape[1:], dtype=ws[0].dtype,
                      device=ws[0].device)
    off = 0
    with torch.no_grad():
        for p in params:
            n = p.shape[0]
            buf[off:off + n].copy_(p.data)
            p.data = buf[off:off + n]
            off += n


def _align(n: int) -> int:
    return (n + 255) // 256 * 256


class _Block:
    """One call's ``nmb_block``: the weights checked against the block's shape
    (the C side sees addresses only) and the tensors that must outlive the
    launches on this stream."""

    __slots__ = ("desc", "ref", "keep", "dtype", "device", "stream", "tokens", "hidden", "qd", "kd", "ffn")

    def __init__(self, like: Tensor, shape, w: tuple[Tensor, ...], m: BlockMeta) -> None:
        Fn._require_gpu(like, m.cos, m.sin)
        b, s, h = shape
        qd, kd, f = m.heads * m.head_dim, m.kv_heads * m.head_dim, w[6].shape[0]
        dtype, device = like.dtype, like.device
        for t, want in zip(w, ((h,), (qd, h), (kd, h), (kd, h), (h, qd), (h,), (f, h), (f, h), (h, f))):
            if t.shape != want:
                raise ValueError(f"block: a weight of shape {tuple(t.shape)} where {want} is needed")
            if t.dtype != dtype or t.device != device:
                raise ValueError(f"block: a {t.dtype} weight on {t.device} with {dtype} activations on {device}")
        if not all([t.is_contiguous() for t in w]):
            w = tuple(t.contiguous() for t in w)
        w_in, wq, wk, wv, wo, w_post, wg, wu, wd = w
        # [Wq; Wk; Wv] and [Wg; Wu] as the model packs them, else copies
        w_qkv = wq if _adjacent((wq, wk, wv)) else torch.cat((wq, wk, wv))
        w_gu = wg if _adjacent((wg, wu)) else torch.cat((wg, wu))
        pos, pos_ptr, pos_bstride = m.positions, None, 0
        if pos is not None:
            if pos.dtype != torch.int32:
                raise ValueError("block: positions must be int32")
            pos_ptr, pos_bstride = pos.data_ptr(), pos.stride(0) if pos.ndim == 2 else 0
        self.desc = _lib.Block(
            b, s, h, m.heads, m.kv_heads, m.head_dim, f, m.sequence_offset, w_in.data_ptr(), w_qkv.data_ptr(),
            wo.data_ptr(), w_post.data_ptr(), w_gu.data_ptr(), wd.data_ptr(), m.cos.data_ptr(), m.sin.data_ptr(),
            m.cos.shape[0], pos_ptr, pos_bstride, m.pos_offset, m.eps, _lib.dtype_code(dtype))
        self.ref = _lib.ctypes.byref(self.desc)
        self.keep = (w, w_qkv, w_gu)
        self.dtype, self.device, self.stream = dtype, device, _lib.stream_of(like)
        self.tokens, self.hidden, self.qd, self.kd, self.ffn = b * s, h, qd, kd, f

    def checked(self, acts: dict, shape, m: BlockMeta) -> dict:
        """The activations a backward reads, contiguous: saved-tensor hooks may
        have given back others (the C side sees addresses only)."""
        h, n = self.hidden, self.tokens
        wants = dict(x2=(n, h), n1=(n, h), qkv=(n, self.qd + 2 * self.kd), o2=(n, self.qd),
                     lse=(shape[0], m.heads, shape[1]), h=(n, h), n2=(n, h), gu=(n, 2 * self.ffn))
        out = {}
        for name, want in wants.items():
            t = acts.get(name)
            if t is None and name == "gu":
                continue
            dtype = torch.float32 if name == "lse" else self.dtype
            if t.shape != want or t.dtype != dtype or t.device != self.device:
                raise ValueError(f"block: {name} saved as a {t.dtype} tensor of shape {tuple(t.shape)} on {t.device} "
                                 f"where {dtype} of shape {want} on {self.device} is needed")
            out[name] = t if t.is_contiguous() else t.contiguous()
        return out

    def forward_ws(self) -> int:
        size = _lib.ctypes.c_int64()
        _lib.call("nmb_block_sizes", self.ref, _lib.ctypes.byref(size), None)
        return size.value

    def backward_bytes(self) -> int:
        size = _lib.ctypes.c_int64()
        _lib.call("nmb_block_sizes", self.ref, None, _lib.ctypes.byref(size))
        return size.value

    def new(self, cols: int) -> Tensor:
        return torch.empty(self.tokens, cols, dtype=self.dtype, device=self.device)

    def bytes(self, n: int) -> Tensor:
        return torch.empty(max(n, 16), dtype=torch.uint8, device=self.device)


def _attention_part(n1: Tensor, w: tuple[Tensor, ...], m: BlockMeta, shape) -> tuple:
    """[q|k|v] (RoPE applied), the attention output o [B*S, Hq*D] and its lse
    from the normalised block input n1."""
    blk = _Block(n1, shape, w, m)
    if n1.shape != (blk.tokens, blk.hidden):
        raise ValueError(f"block: n1 saved with shape {tuple(n1.shape)}")
    n1 = n1.contiguous()
    qkv, o = blk.new(blk.qd + 2 * blk.kd), blk.new(blk.qd)
    lse = torch.empty(shape[0], m.heads, shape[1], dtype=torch.float32, device=blk.device)
    ws_bytes = blk.forward_ws()
    ws = blk.bytes(ws_bytes)
    _lib.call("nmb_block_attention", blk.ref, n1.data_ptr(), qkv.data_ptr(), o.data_ptr(), lse.data_ptr(),
              ws.data_ptr(), ws_bytes, blk.stream)
    return qkv, o, lse


def block_forward(x: Tensor, w: tuple[Tensor, ...], m: BlockMeta, *, recompute: bool,
                  keep_gu: bool = True, gate_up: bool = True) -> dict:
    """Run the block on x [B,S,H].  With recompute=True stop after [g|u] (no s, no y),
    or after n2 with gate_up=False (the backward then recomputes [g|u] inside its
    fused gate/up + SwiGLU-backward GEMM).  With keep_gu=False the gate/up GEMM
    applies the activation in its epilogue and (bf16) [g|u] is never written."""
    x = x.contiguous()
    b, s, hdim = x.shape
    blk = _Block(x, x.shape, w, m)
    x2 = x.view(b * s, hdim)
    acts = dict(x2=x2, n1=blk.new(hdim), qkv=blk.new(blk.qd + 2 * blk.kd), o2=blk.new(blk.qd),
                lse=torch.empty(b, m.heads, s, dtype=torch.float32, device=x.device), h=blk.new(hdim),
                n2=blk.new(hdim))
    gu = None
    if gate_up or not recompute:
        if recompute or keep_gu or x.dtype == torch.float32:
            gu = blk.new(2 * blk.ffn)
        if recompute or keep_gu:
            acts["gu"] = gu
        if not recompute:
            acts["s"] = blk.new(blk.ffn)
            acts["y"] = torch.empty_like(x)
    ws_bytes = blk.forward_ws()
    ws = blk.bytes(ws_bytes)
    n1, qkv, o2, lse, h, n2 = [acts[k].data_ptr() for k in ("n1", "qkv", "o2", "lse", "h", "n2")]
    _lib.call("nmb_block_forward", blk.ref, x2.data_ptr(), n1, qkv, o2, lse, h, n2, _lib.ptr(gu),
              _lib.ptr(acts.get("s")), _lib.ptr(acts.get("y")), ws.data_ptr(), ws_bytes, blk.stream)
    return acts


def block_output(x: Tensor, w: tuple[Tensor, ...], m: BlockMeta) -> Tensor:
    """The block's output alone: its intermediates share one scratch buffer,
    freed on return.  Same kernels as ``block_forward``, same bits."""
    x = x.contiguous()
    b, s, hdim = x.shape
    blk = _Block(x, x.shape, w, m)
    t, es, ws_bytes = blk.tokens, x.element_size(), blk.forward_ws()
    sizes = (t * hdim * es, t * (blk.qd + 2 * blk.kd) * es, t * blk.qd * es, 4 * t * m.heads, t * hdim * es,
             0 if x.dtype == torch.bfloat16 else 2 * t * blk.ffn * es, t * blk.ffn * es, ws_bytes)
    at = [0]
    for n in sizes:
        at.append(at[-1] + _align(n))
    scratch = blk.bytes(at[-1])
    base = scratch.data_ptr()
    n1, qkv, o, lse, h, gu, act, ws = [base + off for off in at[:-1]]
    if x.dtype == torch.bfloat16:
        gu = None
    y = torch.empty_like(x)
    _lib.call("nmb_block_forward", blk.ref, x.data_ptr(), n1, qkv, o, lse, h, n1, gu, act, y.data_ptr(), ws,
              ws_bytes, blk.stream)
    return y


_SIDE_STREAMS: dict[int, torch.cuda.Stream] = {}
# Multiply-adds of the larger MLP weight gradient from which a host-launched
# backward uses the second stream: its events and waits cost ~60-100 us of host
# and queue time, which short products do not give back.  One layer, forward and
# backward, with / without it: 2^32.4 (1,024 tokens of hidden 1024) 517 / 442 us,
# 2^33.4 542 / 558 us with full recompute and 494 / 458 us without, 2^34.4 781 /
# 806 us and (hidden 768) 681 / 696 us, 2^35.4 1,139 / 1,171 us, 2^37.5 3,561 /
# 3,625 us.
_SIDE_MIN_MACS = 1 << 34


def _side_stream(blk: _Block, captured: bool) -> int:
    """The stream of the MLP's weight gradients: a second one of the device (at
    default priority, like every stream here) where the products are long enough
    for the overlap to pay, else the block's own."""
    if not captured and 2 * blk.tokens * blk.ffn * blk.hidden < _SIDE_MIN_MACS:
        return blk.stream
    side = _SIDE_STREAMS.get(blk.device.index)
    if side is None:
        side = _SIDE_STREAMS[blk.device.index] = torch.cuda.Stream(blk.device)
    return side.cuda_stream


def block_backward(acts: dict, dy: Tensor, w: tuple[Tensor, ...], m: BlockMeta, shape,
                   prefetch: Callable[[], None] | None = None) -> tuple:
    """Gradients (dx, dw_in, dWq, dWk, dWv, dWo, dw_post, dWg, dWu, dWd) of the
    block (csrc/block.hip holds the sequence and which products run on a second
    stream).  ``prefetch`` (the recompute prefetch of a captured step) is called
    once the out-projection's products are queued, before the attention
    backward.  The temporaries and gradients are allocated and freed in this
    stream's order: the second stream joins it before this function returns or
    raises."""
    dy = dy.contiguous()
    if dy.dtype != acts["x2"].dtype or tuple(dy.shape) != tuple(shape):
        raise ValueError(f"block: a {dy.dtype} gradient of shape {tuple(dy.shape)} for a "
                         f"{acts['x2'].dtype} output of shape {tuple(shape)}")
    blk = _Block(dy, shape, w, m)
    h, f, qd, kd = blk.hidden, blk.ffn, blk.qd, blk.kd
    acts = blk.checked(acts, shape, m)
    captured = torch.cuda.is_current_stream_capturing()
    side = _side_stream(blk, captured)
    new = lambda *sz: torch.empty(sz, dtype=blk.dtype, device=blk.device)  # noqa: E731
    dx, dw_in, dwqkv, dwo = torch.empty_like(dy), new(h), new(qd + 2 * kd, h), new(h, qd)
    dw_post, dwgu, dwd = new(h), new(2 * f, h), new(h, f)
    nbytes = blk.backward_bytes()
    scratch = blk.bytes(nbytes)
    gu = acts.get("gu")
    x2, n1, qkv, o2, lse, hh, n2 = (acts[k].data_ptr() for k in ("x2", "n1", "qkv", "o2", "lse", "h", "n2"))
    try:
        _lib.call("nmb_block_backward_mlp", blk.ref, dy.data_ptr(), o2, hh, n2, _lib.ptr(gu), dwo.data_ptr(),
                  dw_post.data_ptr(), dwgu.data_ptr(), dwd.data_ptr(), scratch.data_ptr(), nbytes,
                  1 if captured else 0, blk.stream, side)
        if prefetch is not None:
            prefetch()
        _lib.call("nmb_block_backward_attention", blk.ref, x2, n1, qkv, o2, lse, dx.data_ptr(), dw_in.data_ptr(),
                  dwqkv.data_ptr(), scratch.data_ptr(), nbytes, blk.stream)
    finally:
        if side != blk.stream:
            _lib.call("nmb_stream_join", blk.stream, side)
    dwq, dwk, dwv = dwqkv.split((qd, kd, kd))
    dwg, dwu = dwgu.split((f, f))
    return dx, dw_in, dwq, dwk, dwv, dwo, dw_post, dwg, dwu, dwd


_PREFETCH_STREAMS: dict[int, torch.cuda.Stream] = {}
# device index -> weak reference to the latest CheckpointedBlockFunction
# context of the forward pass being captured
_LAST_CHECKPOINTED: dict[int, Any] = {}


def begin_forward_pass(device: torch.device) -> None:
    """Called by the model at the start of each forward: the recompute prefetch
    links the checkpointed blocks of one forward pass only."""
    if device.type == "cuda":
        _LAST_CHECKPOINTED.pop(device.index, None)


def _prefetch_recompute(ctx: Any, device: torch.device) -> None:
    """Queues the recompute of the checkpointed block ``ctx`` on a third
    stream; its backward waits for the recorded event, then uses the result.

    In a captured step, a block's backward starts the recompute of the
    checkpointed block before it (in forward order) once its own
    out-projection products are queued, so that the recompute's launches
    overlap the attention backward, the QKV products and the norm backward of
    the block being differentiated instead of following them (replayed config-3
    step -2.1%, same process, bit-identical: the same kernels on the same
    inputs; started before the block's MLP backward instead, -0.7%; launched
    from the host, 2.1% slower, so host-launched steps recompute in place).
    Costs one block's recompute outputs held at the peak."""
    main = torch.cuda.current_stream(device)
    stream = _PREFETCH_STREAMS.get(device.index)
    if stream is None:
        stream = _PREFETCH_STREAMS[device.index] = torch.cuda.Stream(device)
    saved = ctx.saved_tensors
    x, weights = saved[0], tuple(saved[1:])
    stream.wait_stream(main)
    with torch.cuda.stream(stream):
        acts = block_forward(x, weights, ctx.meta, recompute=True, gate_up=False)
        done = torch.cuda.Event()
        done.record(stream)
    ctx.prefetched = (acts, weights, done)


class CheckpointedBlockFunction(torch.autograd.Function):
    """Full per-layer recompute: saves x (the block input) only; with
    ``offload`` x waits for the backward in pinned host memory.  In a captured
    step the recompute of the block before runs early, on a third stream
    (``_prefetch_recompute``)."""

    @staticmethod
    def forward(ctx: Any, x: Tensor, meta: BlockMeta, offload: bool, *weights: Tensor) -> Tensor:
        x = x.contiguous()
        y = block_output(x, weights, meta)
        ctx.meta = meta
        ctx.shape = tuple(x.shape)
        ctx.offloaded = None
        if offload:
            # enqueued after the block's kernels on the same stream, which read x first
            host = torch.empty(x.shape, dtype=x.dtype, pin_memory=True)
            host.copy_(x, non_blocking=True)
            ctx.offloaded = (host, x.device)
            ctx.save_for_backward(*weights)
        else:
            ctx.save_for_backward(x, *weights)
        ctx.prefetched = None
        ctx.prefetch_prev = None
        if not offload and x.is_cuda and torch.cuda.is_current_stream_capturing():
            ctx.prefetch_prev = _LAST_CHECKPOINTED.get(x.device.index)
            _LAST_CHECKPOINTED[x.device.index] = weakref.ref(ctx)
        return y

    @staticmethod
    def backward(ctx: Any, dy: Tensor):
        prev = ctx.prefetch_prev() if ctx.prefetch_prev is not None else None
        ctx.prefetch_prev = None
        with torch.no_grad():
            if ctx.prefetched is not None:
                acts, weights, done = ctx.prefetched
                ctx.prefetched = None
                main = torch.cuda.current_stream(dy.device)
                main.wait_event(done)
                for t in acts.values():
                    t.record_stream(main)
            else:
                saved = ctx.saved_tensors
                if ctx.offloaded is not None:
                    host, device = ctx.offloaded
                    x, weights = host.to(device, non_blocking=True), saved
                    ctx.offloaded = None
                else:
                    x, weights = saved[0], saved[1:]
                weights = tuple(weights)
                # the recompute re-runs the forward's attention kernel: o and lse come
                # out bit-identical to the forward's, so the lse needs no saving; the
                # gate/up product is recomputed inside the MLP backward's GEMM
                acts = block_forward(x, weights, ctx.meta, recompute=True, gate_up=False)
            prefetch = None
            if (prev is not None and prev.prefetched is None and prev.offloaded is None
                    and any(prev.needs_input_grad) and torch.cuda.is_current_stream_capturing()):
                prefetch = lambda: _prefetch_recompute(prev, dy.device)  # noqa: E731
            grads = block_backward(acts, dy, weights, ctx.meta, ctx.shape, prefetch=prefetch)
        return (grads[0], None, None, *grads[1:])


class SelectiveBlockFunction(torch.autograd.Function):
    """Selective recompute (activation_checkpoint.mode = "selective",
    models/gpt/layer.py:68-89): the sub-blocks named in ``ops`` ("attention":
    the Q/K/V projection, RoPE, attention and out projection; "mlp": gate/up,
    SwiGLU and down projection) are checkpointed on their inputs, as the
    reference's per-sub-block ``activation_checkpoint`` does.  Saved: the block
    input x and the residual midpoint h (the norms' inputs, outside the
    checkpoints), n1 and n2 (the checkpointed sub-blocks' inputs), and the
    intermediates of a sub-block that is not checkpointed.  The backward
    recomputes a checkpointed attention's [q|k|v], o and lse from n1 and a
    checkpointed MLP's [g|u] from n2 (inside the fused gate/up + SwiGLU
    backward GEMM) with the forward's arithmetic (same bits),
    never the norms, the out projection or the down projection, whose outputs
    it does not read, then runs the shared block backward.  With ``offload``
    the checkpointed sub-blocks' inputs wait in pinned host memory."""

    @staticmethod
    def forward(ctx: Any, x: Tensor, meta: BlockMeta, ops: tuple[str, ...], offload: bool,
                *weights: Tensor) -> Tensor:
        x = x.contiguous()
        attn_ck, mlp_ck = "attention" in ops, "mlp" in ops
        acts = block_forward(x, weights, meta, recompute=False, keep_gu=not mlp_ck)
        ctx.meta = meta
        ctx.shape = tuple(x.shape)
        ctx.ops = (attn_ck, mlp_ck)
        keep = ["h"] + ([] if attn_ck else ["n1", "qkv", "o2", "lse"]) + ([] if mlp_ck else ["n2", "gu"])
        ck = ([acts["n1"]] if attn_ck else []) + ([acts["n2"]] if mlp_ck else [])
        ctx.keys = keep
        ctx.offloaded = None
        if offload and ck:
            # enqueued after the block's kernels on the same stream, which read them first
            host = [torch.empty(t.shape, dtype=t.dtype, pin_memory=True) for t in ck]
            for hst, t in zip(host, ck):
                hst.copy_(t, non_blocking=True)
            ctx.offloaded = (host, x.device)
            ck = []
        ctx.n_ck = len(ck)
        ctx.save_for_backward(x, *(acts[k] for k in keep), *ck, *weights)
        return acts["y"]

    @staticmethod
    def backward(ctx: Any, dy: Tensor):
        saved = ctx.saved_tensors
        x, weights = saved[0], tuple(saved[1 + len(ctx.keys) + ctx.n_ck:])
        acts = dict(zip(ctx.keys, saved[1:1 + len(ctx.keys)]))
        ck = list(saved[1 + len(ctx.keys):1 + len(ctx.keys) + ctx.n_ck])
        if ctx.offloaded is not None:
            host, device = ctx.offloaded
            ck = [t.to(device, non_blocking=True) for t in host]
            ctx.offloaded = None
        attn_ck, mlp_ck = ctx.ops
        b, s, hdim = ctx.shape
        m = ctx.meta
        acts["x2"] = x.reshape(b * s, hdim)
        with torch.no_grad():
            if attn_ck:
                acts["n1"] = ck.pop(0)
                acts["qkv"], acts["o2"], acts["lse"] = _attention_part(acts["n1"], weights, m, ctx.shape)
            if mlp_ck:
                # [g|u] is recomputed inside the MLP backward's GEMM
                acts["n2"] = ck.pop(0)
            grads = block_backward(acts, dy, weights, m, ctx.shape)
        return (grads[0], None, None, None, *grads[1:])


class EagerBlockFunction(torch.autograd.Function):
    """No checkpoint: keeps every intermediate the backward reads."""

    @staticmethod
    def forward(ctx: Any, x: Tensor, meta: BlockMeta, *weights: Tensor) -> Tensor:
        if not meta.keep:
            return block_output(x, weights, meta)
        acts = block_forward(x, weights, meta, recompute=False)
        ctx.meta = meta
        ctx.shape = tuple(x.shape)
        keys = ("x2", "n1", "qkv", "o2", "lse", "h", "n2", "gu")
        ctx.keys = keys
        ctx.save_for_backward(*(acts[k] for k in keys), *weights)
        return acts["y"]

    @staticmethod
    def backward(ctx: Any, dy: Tensor):
        saved = ctx.saved_tensors
        n = len(ctx.keys)
        acts = dict(zip(ctx.keys, saved[:n]))
        weights = tuple(saved[n:])
        with torch.no_grad():
            grads = block_backward(acts, dy, weights, ctx.meta, ctx.shape)
        return (grads[0], None, *grads[1:])
