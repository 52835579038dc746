"""The gated MLP's projection is a module like any other: hooks on it, a forward put
in its place and another module in its place are run."""

import torch
from torch import nn

from parallax_amd.models.config import ModelConfig
from parallax_amd.models.llama import LlamaMLP
from parallax_amd.ops import reference as ref


def _mlp():
    torch.manual_seed(0)
    m = LlamaMLP(ModelConfig(
        architecture="LlamaForCausalLM", vocab_size=64, hidden_size=32, num_layers=1,
        num_heads=2, num_kv_heads=1, head_dim=16, intermediate_size=48,
        max_position_embeddings=64, eos_token_ids=[]))
    for p in m.parameters():
        p.data.normal_(std=0.2)
    return m, torch.randn(3, 32)


def _check(m, x, y):
    """48 products below 20 each, summed in fp32 in any order."""
    want = ref.silu_and_mul(y) @ m.down_proj.weight.t()
    torch.testing.assert_close(m(x), want, rtol=0, atol=48 * 20 * 2 ** -20)


def test_hooks_see_and_replace_the_projection():
    m, x = _mlp()
    y = x @ m.gate_up_proj.weight.t()
    seen = []
    h = m.gate_up_proj.register_forward_hook(
        lambda mod, args, out: (seen.append(out), out * 2)[1])
    _check(m, x, y * 2)
    torch.testing.assert_close(seen[0], y)
    h.remove()
    h = m.gate_up_proj.register_forward_pre_hook(lambda mod, args: (args[0] * 3,))
    _check(m, x, y * 3)
    h.remove()
    h = nn.modules.module.register_module_forward_hook(
        lambda mod, args, out: seen.append(out) if mod is m.gate_up_proj else None)
    _check(m, x, y)
    h.remove()
    assert len(seen) == 2


def test_another_forward_or_module_is_called():
    m, x = _mlp()
    y = x @ m.gate_up_proj.weight.t()
    m.gate_up_proj.forward = lambda t: t @ m.gate_up_proj.weight.t() - 1
    _check(m, x, y - 1)
    lin = nn.Linear(32, 96, bias=False)
    m.gate_up_proj = lin
    _check(m, x, lin(x))
