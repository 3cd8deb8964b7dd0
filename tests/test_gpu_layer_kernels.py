"""The decoder layer's own kernels against the torch expressions they stand in for, in float64 where those round:
RMSNorm with and without the residual sum (rows shorter and longer than a workgroup keeps in registers), SwiGLU, and
the calls that keep torch's path."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}  # one rounding to 8 / 11 significant bits: at most this, relative


def _randn(shape, dtype, seed, std=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * std).to(dtype).to(DEV)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,dim", [(1, 8), (3, 2040), (5, 4096), (2, 8192), (3, 8200), (2, 20480), (777, 256)])
def test_rms_norm(hip, dtype, rows, dim):
    from minillm.model.llama import RMSNorm
    from minillm.model import kernels

    norm = RMSNorm(dim, 1e-5).to(DEV, dtype)
    x, y = _randn((1, rows, dim), dtype, 1, 3.0), _randn((1, rows, dim), dtype, 2)
    with torch.no_grad():
        norm.weight.copy_(_randn((dim,), dtype, 3) * 0.1 + 1)
        assert kernels.usable(x) and kernels.norm_ok(x, norm.weight)
        out = norm(x)
        total, out2 = kernels.add_rms_norm(x, y, norm.weight, norm.eps)
    assert torch.equal(total, x + y)
    for got, src in ((out, x), (out2, total)):
        d = src.double()
        ref = norm.weight.double() * (d * torch.rsqrt(d.square().mean(-1, keepdim=True) + 1e-5))
        # two roundings: the cast, the product with the weight
        torch.testing.assert_close(got.double(), ref, rtol=2.02 * EPS[dtype], atol=1e-6)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [8, 2040, 14336 * 3])
def test_silu_mul(hip, dtype, n):
    from minillm.model import kernels

    gate, up = _randn((n,), dtype, 4, 4.0), _randn((n,), dtype, 5)
    gate[:4] = torch.tensor([-100.0, 100.0, 0.0, -20.0], dtype=dtype)
    with torch.no_grad():
        out = kernels.silu_mul(gate, up)
    g = gate.double()
    torch.testing.assert_close(out.double(), g / (1 + torch.exp(-g)) * up.double(), rtol=1.01 * EPS[dtype], atol=1e-7)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 1), (2, 37), (1, 1000)])
def test_rope_table(hip, dtype, shape):
    from minillm.model.config import LLAMA_3_1_8B, LlamaConfig
    from minillm.model.llama import RotaryEmbedding

    rot = RotaryEmbedding(LlamaConfig(**LLAMA_3_1_8B))
    pos = torch.randint(0, 131072, shape, generator=torch.Generator().manual_seed(22)).to(DEV)
    pos[0, 0] = 0
    with torch.no_grad():
        got = rot(pos, dtype)
    exp = rot(pos, dtype)  # gradients on: torch's expressions
    # the same fp32 angles; cos and sin within some 2^-24 before one rounding, which may then fall to the other side
    for g, e in zip(got, exp):
        assert g.shape == (*shape, 128) and g.dtype == dtype
        torch.testing.assert_close(g.float(), e.float(), rtol=2 * EPS[dtype], atol=1e-6)


def test_torch_path_kept(hip):
    # gradients, hooks, float32, odd widths and transforms see torch's own operations
    from minillm.model import kernels
    from minillm.model.llama import RMSNorm

    x = _randn((4, 64), torch.bfloat16, 6)
    norm = RMSNorm(64, 1e-5).to(DEV, torch.bfloat16)
    xg = x.clone().requires_grad_()
    norm(xg).sum().backward()
    assert xg.grad is not None and norm.weight.grad is not None
    with torch.no_grad():
        assert not kernels.usable(x.float()) and not kernels.usable(x.cpu())
        assert not kernels.norm_ok(_randn((4, 63), torch.bfloat16, 7), norm.weight)
        assert not kernels.norm_ok(x.t().contiguous().t(), norm.weight)
        torch.testing.assert_close(torch.func.vmap(norm)(x), norm(x), rtol=2 * EPS[torch.bfloat16], atol=1e-6)
        with torch.autograd.forward_ad.dual_level():
            assert not kernels.usable(x)
    assert kernels.bare(norm, RMSNorm)
    norm.register_forward_hook(lambda *a: None)
    assert not kernels.bare(norm, RMSNorm)


@pytest.mark.parametrize("part", ["norm", "mlp"])
def test_vmap_over_weights(hip, part):
    # an ensemble: one x, a batch of parameters
    from minillm.model import llama
    from minillm.model.config import LlamaConfig

    cfg = LlamaConfig(vocab_size=64, hidden_size=512, intermediate_size=768, num_hidden_layers=1, num_attention_heads=4,
                      num_key_value_heads=2, head_dim=128, rms_norm_eps=1e-5, rope_theta=1e4)
    x = _randn((3, 512), torch.bfloat16, 27)
    modules = [(llama.RMSNorm(512, 1e-5) if part == "norm" else llama.LlamaMLP(cfg)).to(DEV, torch.bfloat16)
               for _ in range(2)]
    with torch.no_grad():
        for i, m in enumerate(modules):
            for p in m.parameters():
                p.add_(0.01 * i)
        params, _ = torch.func.stack_module_state(modules)
        got = torch.func.vmap(lambda p: torch.func.functional_call(modules[0], p, (x,)))(params)
        exp = torch.stack([m(x) for m in modules])
    # torch's expressions against the kernels: a few bf16 roundings of values below 4
    torch.testing.assert_close(got.float(), exp.float(), rtol=4 * EPS[torch.bfloat16], atol=0.03)


@pytest.mark.parametrize("part", ["norm", "mlp", "rotary"])
def test_modules_compile_as_one_graph(hip, part):
    from minillm.model import llama
    from minillm.model.config import LlamaConfig

    cfg = LlamaConfig(vocab_size=64, hidden_size=512, intermediate_size=768, num_hidden_layers=1, num_attention_heads=4,
                      num_key_value_heads=2, head_dim=128, rms_norm_eps=1e-5, rope_theta=1e4)
    x = _randn((1, 3, 512), torch.bfloat16, 26)
    module, args = {"norm": (llama.RMSNorm(512, 1e-5), (x,)), "mlp": (llama.LlamaMLP(cfg), (x,)),
                    "rotary": (llama.RotaryEmbedding(cfg), (torch.arange(3, device=DEV)[None], torch.bfloat16))}[part]
    module = module.to(DEV, torch.bfloat16)
    with torch.no_grad():
        compiled = torch.compile(module, fullgraph=True, backend="eager")
        got_exp = compiled(*args), module(*args)
    # the kernels keep silu and the norm in fp32 where torch's expressions round: a few bf16 roundings of values below 4
    for got, exp in zip(*(y if part == "rotary" else (y,) for y in got_exp)):
        torch.testing.assert_close(got.float(), exp.float(), rtol=4 * EPS[torch.bfloat16], atol=0.03)


def _ref(x, w):
    return x.double() @ w.double().t()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k,rows", [(1, 256, (16,)), (15, 512, (144, 16)), (16, 4096, (4096, 1024, 1024)),
                                      (17, 1024, (272,)), (33, 2048, (128, 112, 240)), (48, 768, (4096,)),
                                      (49, 14336, (256,)), (64, 4096, (1008,))])
def test_linear_of_few_rows(hip, dtype, m, k, rows):
    from minillm.model import kernels

    x, res = _randn((1, m, k), dtype, 8), _randn((1, m, sum(rows)), dtype, 9)
    ws = [_randn((n, k), dtype, 10 + i, 0.05) for i, n in enumerate(rows)]
    out, plus = kernels.linear(x, *ws), kernels.linear(x, *ws, residual=res)
    ref = torch.cat([_ref(x, w) for w in ws], dim=-1)
    # one rounding, and the fp32 sums' error: k terms of some 0.05, each addition off by at most 2^-24 of a partial sum
    # of at most some 10, in random directions: sqrt(14,336) x 6e-7 < 1e-4
    torch.testing.assert_close(out.double(), ref, rtol=1.01 * EPS[dtype], atol=1e-4)
    torch.testing.assert_close(plus.double(), ref + res.double(), rtol=1.01 * EPS[dtype], atol=1e-4)
    # a row's result is the same alone, and whatever rows are beside it
    assert torch.equal(kernels.linear(x[:, -1:].contiguous(), *ws), out[:, -1:])


@pytest.mark.parametrize("m,k,n", [(1, 256, 16), (16, 512, 80), (37, 4096, 14336), (64, 1024, 144)])
def test_linear_swiglu_and_norm_behind_a_product(hip, m, k, n):
    from minillm.model import kernels

    dtype = torch.bfloat16
    x = _randn((1, m, k), dtype, 11)
    gate, up = _randn((n, k), dtype, 12, 0.05), _randn((n, k), dtype, 13, 0.05)
    g = _ref(x, gate)
    # the sums' fp32 error (1e-5 and less) moves silu by less than 1.1 times itself, times |up| of some units
    torch.testing.assert_close(kernels.linear_swiglu(x, gate, up).double(), g / (1 + torch.exp(-g)) * _ref(x, up),
                               rtol=1.01 * EPS[dtype], atol=1e-3)
    res, w = _randn((1, m, n), dtype, 14), _randn((n,), dtype, 15) * 0.1 + 1
    total, out = kernels.linear_add_norm(x, gate, res, w, 1e-5)
    torch.testing.assert_close(total.double(), res.double() + g, rtol=1.01 * EPS[dtype], atol=1e-4)
    d = total.double()
    torch.testing.assert_close(out.double(), w.double() * (d * torch.rsqrt(d.square().mean(-1, keepdim=True) + 1e-5)),
                               rtol=2.02 * EPS[dtype], atol=1e-6)


def test_few_row_layers_keep_hooks_biases_and_wide_rows(hip):
    from minillm.model import kernels

    lin = torch.nn.Linear(256, 32, bias=False, device=DEV, dtype=torch.bfloat16)
    x = _randn((1, 64, 256), torch.bfloat16, 16)
    with torch.no_grad():
        assert kernels.small_rows(x) and kernels.weights_ok(x, 256, lin)
        assert not kernels.small_rows(_randn((1, 65, 256), torch.bfloat16, 17)) and not kernels.weights_ok(x, 128, lin)
        assert not kernels.weights_ok(x.half(), 256, lin)
        assert not kernels.weights_ok(x, 256, torch.nn.Linear(256, 32, device=DEV, dtype=torch.bfloat16))
        assert not kernels.weights_ok(x, 256, torch.nn.Linear(256, 24, bias=False, device=DEV, dtype=torch.bfloat16))
    handle = lin.register_forward_pre_hook(lambda *a: None)
    assert not kernels.weights_ok(x, 256, lin)
    handle.remove()
    assert kernels.weights_ok(x, 256, lin)


@pytest.mark.parametrize("part", ["o_proj", "mlp", "post_attention_layernorm"])
def test_decoder_layer_with_a_hook_calls_it(hip, part):
    from minillm.attention import get_backend
    from minillm.model.config import LlamaConfig
    from minillm.model.llama import LlamaDecoderLayer, LlamaModel, random_init_  # noqa: F401

    cfg = LlamaConfig(vocab_size=64, hidden_size=512, intermediate_size=768, num_hidden_layers=1, num_attention_heads=4,
                      num_key_value_heads=2, head_dim=128, rms_norm_eps=1e-5, rope_theta=1e4, rope_scaling=None,
                      max_position_embeddings=512)
    layer = LlamaDecoderLayer(cfg, get_backend("hip"), 0).to(DEV, torch.bfloat16)
    x = _randn((2, 9, 512), torch.bfloat16, 18)
    ang = torch.randn(2, 9, 128, device=DEV)
    with torch.inference_mode():
        cos, sin = ang.cos().bfloat16(), ang.sin().bfloat16()
        plain = layer(x, cos, sin)
        seen = []
        target = layer.self_attn.o_proj if part == "o_proj" else getattr(layer, part)
        target.register_forward_hook(lambda *a: seen.append(1))
        hooked = layer(x, cos, sin)
    assert seen == [1]
    # the two paths round at different places: a few bf16 roundings of values of some units
    torch.testing.assert_close(plain.float(), hooked.float(), rtol=4 * EPS[torch.bfloat16], atol=0.03)


@pytest.mark.parametrize("where", ["self_attn.q_proj", "self_attn.o_proj", "mlp.up_proj", "mlp.down_proj", "mlp",
                                   "input_layernorm", "post_attention_layernorm"])
def test_decoder_layer_with_a_wrapped_submodule(hip, where):
    # a submodule that is not the plain class and has no weight of its own (an adapter, a quantized layer) is called
    from minillm.attention import get_backend
    from minillm.model.config import LlamaConfig
    from minillm.model.llama import LlamaDecoderLayer

    class Wrap(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, x):
            return self.inner(x)

    cfg = LlamaConfig(vocab_size=64, hidden_size=512, intermediate_size=768, num_hidden_layers=1, num_attention_heads=4,
                      num_key_value_heads=2, head_dim=128, rms_norm_eps=1e-5, rope_theta=1e4)
    torch.manual_seed(24)
    layer = LlamaDecoderLayer(cfg, get_backend("hip"), 0).to(DEV, torch.bfloat16)
    x, ang = _randn((1, 9, 512), torch.bfloat16, 25), torch.randn(1, 9, 128, device=DEV)
    with torch.inference_mode():
        cos, sin = ang.cos().bfloat16(), ang.sin().bfloat16()
        plain = layer(x, cos, sin)
        parent = layer.get_submodule(where.rpartition(".")[0])
        name = where.rpartition(".")[2]
        setattr(parent, name, Wrap(getattr(parent, name)))
        wrapped = layer(x, cos, sin)
    # the two paths round at different places: a few bf16 roundings of values of some units
    torch.testing.assert_close(plain.float(), wrapped.float(), rtol=4 * EPS[torch.bfloat16], atol=0.03)


@pytest.mark.parametrize("dtype,kv", [(torch.bfloat16, None), (torch.float16, None), (torch.bfloat16, torch.float8_e4m3fn)])
@pytest.mark.parametrize("rows", [[(0, 1)], [(5, 1), (300, 1), (47, 1)], [(9, 1), (33, 20), (0, 40), (100, 2)], [(7, 1)] * 64,
                                  [(3, 65)]])
def test_decoder_layer_in_one_call(hip, dtype, kv, rows):
    # the same launches as the submodules one after the other (which a backend with overlap_mixed set gets), bit for
    # bit, on the output and both pools; more than 64 rows never take the call
    from minillm.attention import get_backend
    from minillm.attention.metadata import AttentionMetadata, SeqStep
    from minillm.cache.paged import PagedKVCache
    from minillm.model import kernels
    from minillm.model.config import LlamaConfig
    from minillm.model.llama import LlamaDecoderLayer

    cfg = LlamaConfig(vocab_size=64, hidden_size=1024, intermediate_size=1536, num_hidden_layers=1, num_attention_heads=8,
                      num_key_value_heads=2, head_dim=128, rms_norm_eps=1e-5, rope_theta=1e4, rope_scaling=None,
                      max_position_embeddings=512)
    backend = get_backend("hip")
    torch.manual_seed(19)
    layer = LlamaDecoderLayer(cfg, backend, 0).to(DEV, dtype)
    n = sum(new for _, new in rows)
    x, ang = _randn((1, n, 1024), dtype, 20), torch.randn(1, n, 128, device=DEV)
    at, seqs = 0, []
    for cached, new in rows:
        need = -(-(cached + new) // 16)
        seqs.append(SeqStep(cached, new, list(range(at, at + need))))
        at += need
    scales = {"k_scale": 0.02, "v_scale": 0.03} if kv else {}
    results = []
    with torch.inference_mode():
        cos, sin = ang.cos().to(dtype), ang.sin().to(dtype)
        for overlap in (False, True):
            backend.overlap_mixed = overlap
            g = torch.Generator(device=DEV).manual_seed(21)
            cache = PagedKVCache(cfg, at, DEV, kv or dtype, **scales)
            for pool in (cache.k[0], cache.v[0]):
                pool.copy_(torch.randn(pool.shape, device=DEV, generator=g).to(pool.dtype))
            step = cache.step(AttentionMetadata.build(seqs, 16, DEV))
            assert kernels.small_rows(x) == (n <= 64)
            if n <= 64:
                assert (kernels.decoder_layer(layer, x, cos, sin, step) is None) == overlap
            results.append((layer(x, cos, sin, step), cache.k[0], cache.v[0]))
    for a, b in zip(*results):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
