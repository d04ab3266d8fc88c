"""Saved-tensor hooks around the fused block: what its backward reads is checked before a launch."""

from __future__ import annotations

import pytest
import torch

import nano_megatron_amd as nm

pytestmark = pytest.mark.gpu


def _layer_grads(mode: str, unpack, *, raises: bool = False):
    cfg = nm.GPTConfig(layers=1, hidden_size=128, ffn_hidden_size=264, heads=2, kv_heads=1, seq_length=24,
                       vocab_size=64)
    torch.manual_seed(0)
    ck = nm.ActivationCheckpointConfig(mode=mode)
    model = nm.GPTModel(cfg, activation_checkpoint_config=ck, owns_embedding=False, owns_final_norm=False,
                        owns_lm_head=False).to(device="cuda", dtype=torch.bfloat16).train()
    x = torch.randn(2, 24, 128, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        y = model(hidden_states=x).hidden_states
    if raises:
        with pytest.raises(ValueError, match="block"):
            y.float().square().sum().backward()
        return None
    return torch.autograd.grad(y, (x, *model.parameters()), torch.ones_like(y))


def _restrided(t):
    """The same values with the last dimension strided (no dense rows)."""
    out = torch.empty(*t.shape, 2, dtype=t.dtype, device=t.device)[..., 0]
    return out.copy_(t.detach())


@pytest.mark.parametrize("mode", ["none", "selective", "full"])
def test_strided_saved_tensors_give_the_same_bits(mode) -> None:
    exp = _layer_grads(mode, lambda t: t)
    got = _layer_grads(mode, lambda t: _restrided(t) if t.ndim >= 2 else t)
    assert all(torch.equal(a, b) for a, b in zip(exp, got))


@pytest.mark.parametrize("change", [
    lambda t: t.cpu() if t.dtype == torch.float32 and t.ndim == 3 else t,      # lse elsewhere
    lambda t: t.half() if t.dtype == torch.float32 and t.ndim == 3 else t,     # lse in another type
    lambda t: t[:-1] if t.shape == (48, 264 * 2) else t,                       # [g|u] a row short
], ids=["device", "dtype", "shape"])
def test_wrong_saved_tensors_are_refused(change) -> None:
    _layer_grads("none", change, raises=True)
