"""Which calls keep torch's expressions instead of the decoder layer's kernels, and the rules that size the kernels' launches,
as far as they show without a GPU."""

from concurrent.futures import ThreadPoolExecutor

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


def test_more_rows_than_a_launch_takes(monkeypatch):
    # a launch has fewer than 2^32 threads: larger calls keep torch's expressions, and the entry points refuse them
    # before they launch anything
    from minillm import _native

    empty = lambda *s: torch.empty(s, dtype=torch.bfloat16, device="meta")  # noqa: E731
    assert kernels.norm_ok(empty((1 << 24) - 1, 8), empty(8)) and not kernels.norm_ok(empty(1 << 24, 8), empty(8))
    monkeypatch.setattr(kernels, "usable", lambda x, dtype=None: True)
    assert kernels.silu_mul_ok(empty((1 << 35) - 2048), empty((1 << 35) - 2048))
    assert not kernels.silu_mul_ok(empty(1 << 35), empty(1 << 35))
    pos = torch.empty(1 << 26, dtype=torch.int64, device="meta")
    assert not kernels.rope_ok(pos, torch.bfloat16, 64) and kernels.rope_ok(pos[:-4], torch.bfloat16, 64)
    call, p = _native.lib().call, 1 << 20  # 16-byte aligned, never read
    for name, args in (("mllm_rms_norm", (p, None, p, 1 << 24, 8, 1e-5, 2, None, p, None)),
                       ("mllm_silu_mul", (p, p, 1 << 35, 2, p, None)),
                       ("mllm_sum_partials", (p, 1, 1 << 24, 2048, None, 2, p, None)),
                       ("mllm_sum_partials_norm", (p, 1, p, p, 1 << 24, 8, 1e-5, 2, p, p, None)),
                       ("mllm_rope_table", (p, 1 << 26, p, 64, 2, p, p, None))):
        with ThreadPoolExecutor(1) as own, pytest.raises(ValueError, match="fewer than|too many"):
            own.submit(call, name, *args).result()  # the last error is kept per thread: other tests' stays empty


def test_dense_workgroup_rows():
    # (batch, heads, KV heads, queries): 128 rows only where a head's queries need more than one workgroup of 32
    from minillm import _native

    rows = _native.lib().fn("mllm_dense_rows")
    for shape, expected in [((1, 32, 8, 512), 32), ((2, 32, 8, 777), 128), ((4, 32, 8, 777), 128), ((64, 32, 8, 1), 32),
                            ((64, 32, 8, 8), 32), ((64, 32, 8, 9), 128), ((128, 32, 8, 8), 32), ((16, 32, 32, 32), 32),
                            ((16, 32, 32, 33), 128), ((12, 32, 32, 33), 128), ((11, 32, 32, 33), 32), ((1, 32, 8, 0), 0)]:
        assert rows(*shape, 256) == expected, shape


def test_launch_rules_follow_the_cu_count():
    from minillm import _native

    rows, parts = _native.lib().fn("mllm_dense_rows"), _native.lib().fn("mllm_linear_ksplit")
    # one sequence of 512 tokens: 128 workgroups of 128 rows, 1.5 per CU up to 85 CUs
    assert [rows(1, 32, 8, 512, cus) for cus in (256, 86, 85, 32)] == [32, 32, 128, 128]
    # q, k and v of Llama-3.1-8B: 48 tiles; o: 32; never below 1 part, nor parts of less than two chunks of 256
    assert [parts(4096, 4096, 1024, 1024, cus) for cus in (256, 128, 64, 32)] == [5, 2, 1, 1]
    assert [parts(4096, 4096, 0, 0, cus) for cus in (256, 128, 64, 32)] == [8, 4, 2, 1]
    assert parts(512, 16, 0, 0, 256) == 1 and parts(1024, 16, 0, 0, 256) == 2
