"""Which calls keep torch's expressions instead of the decoder layer's kernels, as far as that shows without a GPU."""

import pytest
import torch

from minillm.model import kernels, llama
from minillm.model.config import LlamaConfig

CFG = LlamaConfig(vocab_size=64, hidden_size=64, intermediate_size=96, num_hidden_layers=1, num_attention_heads=4,
                  num_key_value_heads=2, head_dim=16, rms_norm_eps=1e-5, rope_theta=1e4)


@pytest.mark.parametrize("module", [llama.RMSNorm(64, 1e-5), llama.LlamaMLP(CFG)], ids=["norm", "mlp"])
def test_modules_can_be_scripted(module):
    x = torch.randn(3, 64, generator=torch.Generator().manual_seed(0))
    with torch.no_grad():
        assert torch.equal(torch.jit.script(module)(x), module(x))


def test_wrapped_operands_are_refused():
    # tensors of a functorch transform, while it runs and after it: no storage to hand to a kernel
    x, seen = torch.zeros(3, 64, dtype=torch.bfloat16), []

    def look(t):
        seen.append(t)
        assert not kernels.sum_ok(x, t) and not kernels.norm_ok(x, t) and not kernels.small_rows(t)
        return t.sum()

    torch.func.vmap(look)(torch.zeros(2, 64, dtype=torch.bfloat16))
    torch.func.grad(look)(torch.zeros(64, dtype=torch.bfloat16))
    for t in seen:
        assert not kernels.norm_ok(x, t)
    assert kernels.norm_ok(x, torch.zeros(64, dtype=torch.bfloat16))


def test_weights_held_as_plain_attributes():
    x = torch.zeros(3, 256, dtype=torch.bfloat16)
    lin = torch.nn.Linear(256, 32, bias=False, dtype=torch.bfloat16)
    assert kernels.weights_ok(x, 256, lin)
    replica = lin._replicate_for_data_parallel()
    replica.weight, replica.bias = lin.weight.detach(), None
    assert not kernels.weights_ok(x, 256, replica)
    for name in ("weight", "bias"):
        other = torch.nn.Linear(256, 32, bias=name == "bias", dtype=torch.bfloat16)
        value = getattr(other, name).detach()
        delattr(other, name)
        setattr(other, name, value)
        assert not kernels.weights_ok(x, 256, other)
