"""The workloads whose speed is measured, one pass each through the public entry points.

What this library is used for: training GPT blocks (bf16, full recompute or
none, MHA and GQA, the configurations' widths and the defaults of
``GPTConfig``), the fp32 smoke configuration, full-prefix logits for text
generation (no KV cache: every new token is one forward over the whole
prefix), attention through the kernel backend with ragged lengths, grouped
heads, padding masks and dropout, one ring-attention rank's share, the LM head
with its loss at the default vocabulary, the embedding with its gradient, and
the fp32-master AdamW step.  ``listed`` names twelve of these calls; ``draw``
gives others of the same ranges.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from nano_megatron_amd import ActivationCheckpointConfig, GPTConfig, GPTModel
from nano_megatron_amd import functional as Fn
from nano_megatron_amd.kernels import HipKernelBackend
from nano_megatron_amd.optim import MasterAdamW

DEV = "cuda"


# ------------------------------------------------------------------ the cases
def listed() -> list[dict]:
    return [
        # the smoke configuration: 4 fp32 layers, forward and backward with every layer
        # checkpointed; small products, many launches
        dict(name="fp32_model_step", kind="model_step", layers=4, hidden=256, heads=4, kv=4, ffn=688,
             vocab=8192, batch=4, seq=128),
        # one token of text generation: logits of a 193-token prefix through the 24-layer
        # 311M model in bf16
        dict(name="prefix_logits", kind="logits", layers=24, hidden=1024, heads=16, kv=16, ffn=2736,
             vocab=8192, batch=1, seq=193),
        # one layer of the 311M training step: micro-batch 16 x 512, full recompute
        dict(name="layer_full", kind="layer", mode="full", hidden=1024, heads=16, kv=16, ffn=2736,
             batch=16, seq=512),
        # one layer of the grouped-query configuration: 4 x 2048, full recompute
        dict(name="layer_gqa_long", kind="layer", mode="full", hidden=2048, heads=32, kv=8, ffn=5632,
             batch=4, seq=2048),
        # one layer at the default widths on a ragged micro-batch, nothing recomputed
        dict(name="layer_ragged", kind="layer", mode="none", hidden=768, heads=12, kv=12, ffn=2048,
             batch=3, seq=709),
        # the backend's attention with grouped heads of 128 at an odd length, both directions
        dict(name="attn_gqa", kind="attn", batch=2, heads=16, kv=4, seq=1537, dim=128, causal=True),
        # causal attention over a batch of unequal sequences (boolean padding mask)
        dict(name="attn_padding", kind="masked", batch=8, heads=16, kv=16, seq=512, dim=64, mask="padding",
             p=0.0),
        # attention of a model trained with dropout 0.1
        dict(name="attn_dropout", kind="masked", batch=8, heads=12, kv=12, seq=512, dim=64, mask="none",
             p=0.1),
        # the last of four ring ranks: 8192 queries against four K/V blocks of 8192
        dict(name="ring_share", kind="ring", heads=16, kv=16, seq=8192, blocks=4, dim=128),
        # LM head and loss at the default width and vocabulary, both directions
        dict(name="lm_head_loss", kind="lm_head", rows=8192, hidden=768, vocab=50304),
        # token embedding and its table gradient, token frequencies as in text (Zipf)
        dict(name="embedding", kind="embedding", batch=4, seq=2048, hidden=768, vocab=50304),
        # the optimizer step (global clip, fp32 master) over six layers of the grouped-query
        # configuration and its embedding, 294M parameters
        dict(name="adamw_294m", kind="adamw", layers=6, hidden=2048, kv_hidden=512, ffn=5632, vocab=8192),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["model_step", "logits", "layer", "layer", "attn", "attn", "masked", "masked", "ring",
                       "lm_head", "embedding", "adamw"])
    if kind == "model_step":
        heads = rng.choice([2, 4, 8])
        return dict(kind=kind, layers=rng.randint(1, 4), hidden=64 * heads, heads=heads,
                    kv=heads // rng.choice([1, 2]), ffn=8 * _log_int(rng, 12, 172), vocab=_log_int(rng, 500, 8192),
                    batch=rng.randint(1, 4), seq=_log_int(rng, 9, 300))
    if kind == "logits":
        return dict(kind=kind, layers=rng.randint(4, 24), hidden=1024, heads=16, kv=rng.choice([16, 4]),
                    ffn=2736, vocab=8192, batch=rng.choice([1, 1, 2, 4]), seq=_log_int(rng, 5, 500))
    if kind == "layer":
        hidden, heads, kv, ffn = rng.choice([(768, 12, 12, 2048), (1024, 16, 16, 2736), (2048, 32, 8, 5632),
                                             (1024, 8, 4, 2736)])
        seq = _log_int(rng, 40, 2048)
        return dict(kind=kind, mode=rng.choice(["full", "none", "selective"]), hidden=hidden, heads=heads, kv=kv,
                    ffn=ffn, batch=max(1, min(16, _log_int(rng, 100, 8192) // seq)), seq=seq)
    if kind == "attn":
        kv = rng.choice([2, 4, 8])
        return dict(kind=kind, batch=rng.randint(1, 4), heads=kv * rng.choice([1, 2, 4]), kv=kv,
                    seq=_log_int(rng, 33, 3000), dim=rng.choice([64, 64, 128, 128, 80]),
                    causal=rng.random() < 0.8)
    if kind == "masked":
        kv = rng.choice([2, 4, 8])
        return dict(kind=kind, batch=rng.randint(1, 8), heads=kv * rng.choice([1, 2]), kv=kv,
                    seq=_log_int(rng, 33, 600), dim=rng.choice([64, 128]),
                    **rng.choice([dict(mask="padding", p=0.0), dict(mask="none", p=0.1),
                                  dict(mask="bias", p=0.0), dict(mask="padding", p=0.2)]))
    if kind == "ring":
        return dict(kind=kind, heads=8, kv=rng.choice([8, 2]), seq=_log_int(rng, 500, 4096),
                    blocks=rng.randint(2, 4), dim=rng.choice([64, 128]))
    if kind == "lm_head":
        return dict(kind=kind, rows=_log_int(rng, 60, 8192), hidden=rng.choice([768, 1024]),
                    vocab=rng.choice([8192, 32000, 50257, 50304]))
    if kind == "embedding":
        return dict(kind=kind, batch=rng.randint(1, 8), seq=_log_int(rng, 30, 2048),
                    hidden=rng.choice([256, 768, 1024, 2048]), vocab=rng.choice([8192, 32000, 50257, 50304]))
    hidden, ffn = rng.choice([(256, 688), (768, 2048), (1024, 2736), (2048, 5632)])
    return dict(kind="adamw", layers=rng.randint(1, 6), hidden=hidden, kv_hidden=hidden // rng.choice([1, 4]),
                ffn=ffn, vocab=8192)


# --------------------------------------------------------------------- inputs
def _gen(seed: int, stream: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(1_000_003 * seed + stream)


def _normal(shape, gen, dtype=torch.bfloat16, std: float = 1.0):
    return (torch.randn(shape, generator=gen, device=DEV) * std).to(dtype)


def _weight(shape, gen, dtype):
    """A Linear weight as it is initialised: uniform within 1 / sqrt(in features)."""
    return ((torch.rand(shape, generator=gen, device=DEV) * 2 - 1) / math.sqrt(shape[1])).to(dtype)


def _layer_weights(case, gen, dtype) -> dict:
    h, d = case["hidden"], case["hidden"] // case["heads"]
    f, kvd = case["ffn"], case["kv"] * d
    lin = lambda n, k: _weight((n, k), gen, dtype)  # noqa: E731
    norm = lambda: (1 + 0.1 * torch.randn(h, generator=gen, device=DEV)).to(dtype)  # noqa: E731
    return {
        "input_norm.weight": norm(),
        "attention.q_proj.linear.weight": lin(h, h),
        "attention.k_proj.linear.weight": lin(kvd, h),
        "attention.v_proj.linear.weight": lin(kvd, h),
        "attention.out_proj.linear.weight": lin(h, h),
        "post_attention_norm.weight": norm(),
        "mlp.gate_proj.linear.weight": lin(f, h),
        "mlp.up_proj.linear.weight": lin(f, h),
        "mlp.down_proj.linear.weight": lin(h, f),
    }


def _model_weights(case, gen, dtype) -> dict:
    w = {"embedding.weight": _normal((case["vocab"], case["hidden"]), gen, dtype, 0.02)}
    for i in range(case["layers"]):
        w.update({f"layers.{i}.{n}": t for n, t in _layer_weights(case, gen, dtype).items()})
    w["final_norm.weight"] = (1 + 0.1 * torch.randn(case["hidden"], generator=gen, device=DEV)).to(dtype)
    return w


def _config(case) -> GPTConfig:
    return GPTConfig(layers=case.get("layers", 1), hidden_size=case["hidden"], ffn_hidden_size=case["ffn"],
                     heads=case["heads"], kv_heads=case["kv"], seq_length=case["seq"],
                     vocab_size=case.get("vocab", 8192))


def _load(model, weights: dict):
    with torch.no_grad():
        for name, p in model.named_parameters():
            p.copy_(weights[name])
    return model


def _heads(case, seq: int, n: int, gen):
    """[B, n, S, D] as the projections leave it: a view of [B, S, n, D] memory."""
    return _normal((case.get("batch", 1), seq, n, case["dim"]), gen).transpose(1, 2)


def _tokens(shape, vocab: int, gen):
    """Token ids with Zipf-like frequencies (log-uniform ranks, shuffled over the table)."""
    ranks = torch.exp(torch.rand(shape, generator=gen, device=DEV, dtype=torch.float64) * math.log(vocab)).long() - 1
    return torch.randperm(vocab, generator=gen, device=DEV)[ranks.clamp_(0, vocab - 1)]


def _adamw_shapes(case) -> list[tuple]:
    h, f = case["hidden"], case["ffn"]
    layer = [(h,), (h, h), (case["kv_hidden"], h), (case["kv_hidden"], h), (h, h), (h,), (f, h), (f, h), (h, f)]
    return [(case["vocab"], h)] + layer * case["layers"] + [(h,)]


def _inputs(case, seed: int) -> dict:
    """Every tensor of a case, from the seed alone."""
    kind, gen = case["kind"], _gen(seed, 1)
    if kind == "model_step":
        ids = torch.randint(0, case["vocab"], (case["batch"], case["seq"] + 1), generator=gen, device=DEV)
        return dict(weights=_model_weights(case, _gen(seed, 2), torch.float32), ids=ids)
    if kind == "logits":
        ids = torch.randint(0, case["vocab"], (case["batch"], case["seq"]), generator=gen, device=DEV)
        return dict(weights=_model_weights(case, _gen(seed, 2), torch.bfloat16), ids=ids)
    if kind == "layer":
        shape = (case["batch"], case["seq"], case["hidden"])
        return dict(weights=_layer_weights(case, _gen(seed, 2), torch.bfloat16), x=_normal(shape, gen),
                    dy=_normal(shape, gen))
    if kind in ("attn", "masked"):
        q, k, v, do = (_heads(case, case["seq"], case[n], gen) for n in ("heads", "kv", "kv", "heads"))
        out = dict(q=q, k=k, v=v, do=do)
        if kind == "masked":
            b, s = case["batch"], case["seq"]
            out["mask"] = None
            if case["mask"] == "padding":  # every sequence keeps its first half at least
                lengths = torch.randint(max(1, s // 2), s + 1, (b,), generator=gen, device=DEV)
                out["mask"] = (torch.arange(s, device=DEV)[None] < lengths[:, None])[:, None, None, :]
            elif case["mask"] == "bias":  # a position bias per head (with it, not causal)
                out["mask"] = _normal((1, case["heads"], s, s), gen)
        return out
    if kind == "ring":
        q, do = (_heads(case, case["seq"], case["heads"], gen) for _ in range(2))
        kv = [tuple(_heads(case, case["seq"], case["kv"], gen) for _ in range(2)) for _ in range(case["blocks"])]
        return dict(q=q, do=do, kv=kv)
    if kind == "lm_head":
        x = _normal((case["rows"], case["hidden"]), gen)
        w = _normal((case["vocab"], case["hidden"]), gen, std=0.02)
        t = _tokens((case["rows"],), case["vocab"], gen)
        t[torch.rand(case["rows"], generator=gen, device=DEV) < 0.05] = Fn.IGNORE_INDEX  # padding tokens
        t[0] = 0
        return dict(x=x, w=w, t=t)
    if kind == "embedding":
        return dict(w=_normal((case["vocab"], case["hidden"]), gen, std=0.02),
                    ids=_tokens((case["batch"], case["seq"]), case["vocab"], gen),
                    dy=_normal((case["batch"], case["seq"], case["hidden"]), gen))
    shapes = _adamw_shapes(case)
    return dict(params=[_normal(s, gen, std=0.02) for s in shapes], grads=[_normal(s, gen, std=1e-3) for s in shapes])


def prepare(case, seed: int) -> dict:
    st = _inputs(case, seed)
    st["case"] = case
    kind = case["kind"]
    if kind == "model_step":
        ck = ActivationCheckpointConfig(mode="full")
        with torch.device(DEV):
            model = GPTModel(_config(case), activation_checkpoint_config=ck)
        st["model"] = _load(model, st.pop("weights")).train()
    elif kind == "logits":
        with torch.device(DEV):
            model = GPTModel(_config(case)).to(torch.bfloat16)
        st["model"] = _load(model, st.pop("weights")).eval()
    elif kind == "layer":
        # one layer as a pipeline stage owns it: hidden states in, hidden states out
        ck = ActivationCheckpointConfig(mode=case["mode"])
        with torch.device(DEV):
            model = GPTModel(_config(case), activation_checkpoint_config=ck, owns_embedding=False,
                             owns_final_norm=False, owns_lm_head=False).to(torch.bfloat16)
        weights = {f"layers.0.{n}": t for n, t in st.pop("weights").items()}
        st["model"] = _load(model, weights).train()
        st["x"].requires_grad_()
    elif kind in ("attn", "masked"):
        st["backend"] = HipKernelBackend()
        for n in "qkv":
            st[n].requires_grad_()
    elif kind == "ring":
        st["q"].requires_grad_()
        for k, v in st["kv"]:
            k.requires_grad_(), v.requires_grad_()
    elif kind == "lm_head":
        st["x"].requires_grad_(), st["w"].requires_grad_()
    elif kind == "embedding":
        st["w"].requires_grad_()
    else:
        st["params"] = [torch.nn.Parameter(p) for p in st["params"]]
        for p, g in zip(st["params"], st.pop("grads")):
            p.grad = g
        st["opt"] = MasterAdamW(st["params"])
    return st


# ----------------------------------------------------------------- one pass
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "model_step":
        model, ids = st["model"], st["ids"]
        names, params = zip(*model.named_parameters())
        loss = model(ids[:, :-1], labels=ids[:, 1:]).loss
        return {"loss": loss.detach(), "grads": dict(zip(names, torch.autograd.grad(loss, params)))}
    if kind == "logits":
        with torch.no_grad():
            return st["model"](st["ids"]).logits
    if kind == "layer":
        names, params = zip(*st["model"].named_parameters())
        y = st["model"](hidden_states=st["x"]).hidden_states
        dx, *dw = torch.autograd.grad(y, (st["x"], *params), st["dy"])
        return {"y": y.detach(), "dx": dx, **dict(zip(names, dw))}
    if kind == "attn":
        q, k, v = st["q"], st["k"], st["v"]
        o = st["backend"].local_attention(q, k, v, causal=case["causal"])
        return (o.detach(), *torch.autograd.grad(o, (q, k, v), st["do"]))
    if kind == "masked":
        q, k, v = st["q"], st["k"], st["v"]
        o = Fn.masked_attention(q, k, v, st["mask"], causal=case["mask"] != "bias", dropout_p=case["p"],
                                seed=_drop_seed(case))
        return (o.detach(), *torch.autograd.grad(o, (q, k, v), st["do"]))
    if kind == "ring":
        s, n = case["seq"], case["blocks"]
        o = Fn.ring_attention(st["q"], st["kv"], [s * i for i in range(n)], query_offset=s * (n - 1))
        flat = [t for kv in st["kv"] for t in kv]
        return (o.detach(), *torch.autograd.grad(o, (st["q"], *flat), st["do"]))
    if kind == "lm_head":
        loss = Fn.lm_head_cross_entropy(st["x"], st["w"], st["t"])
        return (loss.detach(), *torch.autograd.grad(loss, (st["x"], st["w"])))
    if kind == "embedding":
        y = Fn.embedding(st["w"], st["ids"])
        return (y.detach(), *torch.autograd.grad(y, (st["w"],), st["dy"]))
    st["opt"].step()
    opt = st["opt"]
    return {"params": [p.detach() for p in st["params"]], "norm": opt.last_grad_norm, "master": opt.master,
            "exp_avg": opt.exp_avg, "exp_avg_sq": opt.exp_avg_sq}


def _drop_seed(case) -> int:
    return 977 + 31 * case["seq"] + case["heads"]


# ------------------------------------------------------- what a pass cannot do without
def _pairs(sq: int, sk: int, causal: bool, offset: int = 0) -> int:
    """Visible (query, key) pairs of one head."""
    if not causal:
        return sq * sk
    return sum(min(sk, max(0, offset + i + 1)) for i in range(sq))


def _attn_work(b, hq, hkv, d, sq, sk, pairs) -> tuple[int, int]:
    """(bytes, flops) of attention forward (2 products) and backward (5)."""
    flops = 14 * b * hq * pairs * d
    return 2 * b * d * (4 * sq * hq + 4 * sk * hkv), flops


def work(case) -> dict:
    kind = case["kind"]
    if kind in ("attn", "masked"):
        s = case["seq"]
        causal = case.get("causal", case.get("mask") != "bias")
        by, fl = _attn_work(case["batch"], case["heads"], case["kv"], case["dim"], s, s, _pairs(s, s, causal))
        if case.get("mask") == "bias":
            by += 2 * case["heads"] * s * s
        return {"bytes": by, "flops": fl}
    if kind == "ring":
        s, n = case["seq"], case["blocks"]
        by, fl = _attn_work(1, case["heads"], case["kv"], case["dim"], s, s * n, _pairs(s, s * n, True, s * (n - 1)))
        return {"bytes": by, "flops": fl}
    if kind == "lm_head":
        r, h, v = case["rows"], case["hidden"], case["vocab"]
        return {"bytes": 2 * (2 * r * h + 2 * v * h) + 8 * r, "flops": 6 * r * h * v}
    if kind == "embedding":
        t = case["batch"] * case["seq"]
        # rows gathered and written, the incoming gradient read, the table gradient written
        return {"bytes": 2 * (3 * t * case["hidden"] + case["vocab"] * case["hidden"]) + 8 * t,
                "flops": t * case["hidden"]}
    if kind == "adamw":
        n = sum(math.prod(s) for s in _adamw_shapes(case))
        return {"bytes": 28 * n, "flops": 14 * n}
    h, f, d = case["hidden"], case["ffn"], case["hidden"] // case["heads"]
    b, s = case["batch"], case["seq"]
    t = b * s
    w_layer = h * h * 2 + 2 * case["kv"] * d * h + 3 * h * f + 2 * h
    gemm = 2 * t * (w_layer - 2 * h)
    att = 4 * b * case["heads"] * _pairs(s, s, True) * d
    if kind == "layer":
        # forward and backward of the products (3x) and of attention (3.5x), weights and
        # hidden states read, outputs and gradients written; recomputing is the policy's choice
        return {"bytes": 2 * (4 * t * h + 2 * w_layer), "flops": int(3 * gemm + 3.5 * att)}
    v, n = case["vocab"], case["layers"]
    w_all = n * w_layer + v * h + h
    if kind == "logits":
        return {"bytes": 2 * (w_all + t * v) + 8 * t, "flops": n * (gemm + att) + 2 * t * h * v}
    return {"bytes": 4 * 2 * w_all + 16 * t, "flops": int(n * (3 * gemm + 3.5 * att) + 6 * t * h * v)}


# ----------------------------------------------------------------- tolerances
def tolerance(case) -> dict:
    """About four times the error of one pass against ``exact``."""
    kind = case["kind"]
    if kind == "model_step":  # fp32 sums throughout
        return {"rel": 1.5e-5}
    if kind == "logits":  # bf16 roundings carried through every layer
        return {"rel": 4e-2}
    if kind == "layer":  # bf16 intermediates between the products
        return {"rel": 2.5e-2}
    if kind in ("attn", "ring"):  # bf16 probabilities and results
        return {"rel": 1e-2}
    if kind == "masked":  # bf16 results
        return {"rel": 8e-3}
    if kind == "lm_head":  # bf16 logits
        return {"rel": 7e-3}
    return {"rel": 6e-3}  # embedding, AdamW: one bf16 rounding of an fp32 result


# ------------------------------------------------- the same in 64 bits, plain torch
def _norm64(x, w, eps=1e-5):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w


def _rope64(x):
    """x [B, S, H, D] rotated by its positions 0 .. S - 1 (theta 10000)."""
    d, s = x.shape[-1], x.shape[1]
    inv = 1.0 / (10000.0 ** (torch.arange(0, d, 2, dtype=torch.float32) / d))
    ang = torch.arange(s, dtype=torch.float64, device=x.device)[:, None] * inv.to(x.device, torch.float64)
    c, sn = ang.cos()[None, :, None], ang.sin()[None, :, None]
    x1, x2 = x.chunk(2, -1)
    return torch.cat((x1 * c - x2 * sn, x2 * c + x1 * sn), -1)


class _Attention64(torch.autograd.Function):
    """softmax(q k^T / sqrt(d) + mask) (x keep) v for [B, H, S, D], head by head."""

    @staticmethod
    def forward(ctx, q, k, v, causal, offset, mask, keep):
        ctx.save_for_backward(q, k, v)
        ctx.args = (causal, offset, mask, keep)
        out = torch.empty_like(q)
        for b in range(q.shape[0]):
            for h in range(q.shape[1]):
                pr, z = _Attention64.probs(q, k, b, h, causal, offset, mask, keep)
                out[b, h] = (pr if z is None else pr * z) @ v[b, h // (q.shape[1] // k.shape[1])]
        return out

    @staticmethod
    def probs(q, k, b, h, causal, offset, mask, keep):
        sq, sk = q.shape[2], k.shape[2]
        s = (q[b, h] @ k[b, h // (q.shape[1] // k.shape[1])].t().contiguous()).mul_(1.0 / math.sqrt(q.shape[3]))
        if mask is not None:
            m = mask.expand(q.shape[0], q.shape[1], sq, sk)[b, h]
            s = s.masked_fill_(~m, -math.inf) if m.dtype == torch.bool else s.add_(m.double())
        if causal:
            pos = torch.arange(sk, device=q.device)[None] > offset + torch.arange(sq, device=q.device)[:, None]
            s.masked_fill_(pos, -math.inf)
        return torch.softmax(s, -1), (None if keep is None else keep(b, h))

    @staticmethod
    def backward(ctx, do):
        q, k, v = ctx.saved_tensors
        causal, offset, mask, keep = ctx.args
        dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
        scale, group = 1.0 / math.sqrt(q.shape[3]), q.shape[1] // k.shape[1]
        for b in range(q.shape[0]):
            for h in range(q.shape[1]):
                pr, z = _Attention64.probs(q, k, b, h, causal, offset, mask, keep)
                g = do[b, h].contiguous()
                dp = g @ v[b, h // group].t().contiguous()
                if z is not None:
                    dp.mul_(z)
                dv[b, h // group] += (pr if z is None else pr * z).t().contiguous() @ g
                ds = pr.mul_(dp.sub_((dp * pr).sum(-1, keepdim=True))).mul_(scale)
                dq[b, h] = ds @ k[b, h // group]
                dk[b, h // group] += ds.t().contiguous() @ q[b, h]
        return dq, dk, dv, None, None, None, None


def _layer64(x, w, pre, heads, kv):
    b, s, h = x.shape
    d = h // heads
    n = _norm64(x, w[pre + "input_norm.weight"])
    q, k, v = (F.linear(n, w[pre + f"attention.{t}_proj.linear.weight"]) for t in "qkv")
    q, k = _rope64(q.view(b, s, heads, d)), _rope64(k.view(b, s, kv, d))
    o = _Attention64.apply(q.transpose(1, 2).contiguous(), k.transpose(1, 2).contiguous(),
                           v.view(b, s, kv, d).transpose(1, 2).contiguous(), True, 0, None, None)
    x = x + F.linear(o.transpose(1, 2).reshape(b, s, h), w[pre + "attention.out_proj.linear.weight"])
    n = _norm64(x, w[pre + "post_attention_norm.weight"])
    a = F.silu(F.linear(n, w[pre + "mlp.gate_proj.linear.weight"])) * F.linear(n, w[pre + "mlp.up_proj.linear.weight"])
    return x + F.linear(a, w[pre + "mlp.down_proj.linear.weight"])


def _model64(case, w, ids):
    x = F.embedding(ids, w["embedding.weight"])
    for i in range(case["layers"]):
        x = _layer64(x, w, f"layers.{i}.", case["heads"], case["kv"])
    return F.linear(_norm64(x, w["final_norm.weight"]), w["embedding.weight"])


def _keep64(case, seed: int):
    """The factor (0 or 1 / (1 - p)) of every probability of head (b, h): element
    idx = ((b H + h) S + i) S + j is kept iff half idx & 1 of SplitMix64's output
    for counter idx >> 1 is at least floor(p 2^32)."""
    hq, s, p = case["heads"], case["seq"], case["p"]

    def shr(z, n):  # logical shift of 64-bit words held in int64
        return (z >> n) & ((1 << (64 - n)) - 1)

    def signed(v):
        v &= (1 << 64) - 1
        return v - (1 << 64) if v >> 63 else v

    def keep(b, h):
        idx = (b * hq + h) * s * s + torch.arange(s * s, device=DEV)
        z = ((idx >> 1) + 1) * signed(0x9E3779B97F4A7C15) + signed(seed)
        z = (z ^ shr(z, 30)) * signed(0xBF58476D1CE4E5B9)
        z = (z ^ shr(z, 27)) * signed(0x94D049BB133111EB)
        z = z ^ shr(z, 31)
        bits = torch.where((idx & 1).bool(), shr(z, 32), z & 0xFFFFFFFF)
        return ((bits >= int(p * 4294967296.0)).double() / (1.0 - p)).view(s, s)

    return keep if p else None


def exact(case, seed: int):
    st, kind = _inputs(case, seed), case["kind"]
    dbl = lambda t: t.detach().double()  # noqa: E731
    leaf = lambda t: t.detach().double().contiguous().requires_grad_()  # noqa: E731
    if kind in ("model_step", "logits"):
        w = {n: leaf(t) for n, t in st["weights"].items()}
        if kind == "logits":
            with torch.no_grad():
                return _model64(case, w, st["ids"])
        logits = _model64(case, w, st["ids"][:, :-1])
        loss = F.cross_entropy(logits.flatten(0, 1), st["ids"][:, 1:].flatten())
        return {"loss": loss.detach(), "grads": dict(zip(w, torch.autograd.grad(loss, list(w.values()))))}
    if kind == "layer":
        w, x = {n: leaf(t) for n, t in st["weights"].items()}, leaf(st["x"])
        y = _layer64(x, w, "", case["heads"], case["kv"])
        dx, *dw = torch.autograd.grad(y, (x, *w.values()), dbl(st["dy"]))
        return {"y": y.detach(), "dx": dx, **{f"layers.0.{n}": g for n, g in zip(w, dw)}}
    if kind in ("attn", "masked"):
        q, k, v = (leaf(st[n]) for n in "qkv")
        keep = _keep64(case, _drop_seed(case)) if kind == "masked" else None
        causal = case.get("causal", case.get("mask") != "bias")
        o = _Attention64.apply(q, k, v, causal, 0, st.get("mask"), keep)
        return (o.detach(), *torch.autograd.grad(o, (q, k, v), dbl(st["do"])))
    if kind == "ring":
        s, n = case["seq"], case["blocks"]
        q = leaf(st["q"])
        k, v = (leaf(torch.cat([kv[i] for kv in st["kv"]], 2)) for i in (0, 1))
        o = _Attention64.apply(q, k, v, True, s * (n - 1), None, None)
        dq, dk, dv = torch.autograd.grad(o, (q, k, v), dbl(st["do"]))
        grads = [g[:, :, s * i:s * (i + 1)] for i in range(n) for g in (dk, dv)]
        return (o.detach(), dq, *grads)
    if kind == "lm_head":
        x, w, t = dbl(st["x"]), dbl(st["w"]), st["t"]
        valid = t != Fn.IGNORE_INDEX
        count = valid.sum().clamp_min(1)
        loss, dx, dw = 0.0, torch.empty_like(x), torch.zeros_like(w)
        for i in range(0, x.shape[0], 2048):
            xc, vc = x[i:i + 2048], valid[i:i + 2048]
            tc = t[i:i + 2048].masked_fill(~vc, 0)[:, None]
            lp = torch.log_softmax(xc @ w.t(), -1)
            loss = loss - (lp.gather(1, tc)[:, 0] * vc).sum() / count
            g = lp.exp_().scatter_add_(1, tc, -torch.ones_like(tc, dtype=torch.float64))
            g *= (vc / count)[:, None]
            dx[i:i + 2048] = g @ w
            dw += g.t() @ xc
        return (loss, dx, dw)
    if kind == "embedding":
        w, dy = dbl(st["w"]), dbl(st["dy"])
        dw = torch.zeros_like(w).index_add_(0, st["ids"].flatten(), dy.flatten(0, 1))
        return (F.embedding(st["ids"], w), dw)
    # AdamW: lr 3e-4, betas (0.9, 0.95), eps 1e-8, decay 0.1, clip 1.0, first step
    p = torch.cat([dbl(t).flatten() for t in st["params"]])
    g = torch.cat([dbl(t).flatten() for t in st["grads"]])
    norm = g.norm()
    g *= min(1.0, 1.0 / (float(norm) + 1e-6))
    m, v = 0.1 * g, 0.05 * g * g
    p -= 3e-4 * 0.1 * p
    p -= 3e-4 * (m / 0.1) / ((v / 0.05).sqrt() + 1e-8)
    sizes = [t.numel() for t in st["params"]]
    params = [c.view(t.shape) for c, t in zip(p.split(sizes), st["params"])]
    return {"params": params, "norm": norm, "master": p, "exp_avg": m, "exp_avg_sq": v}
