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
