"""The matrix-core kernels behind `prefill` (Dh 64 and 128) at the sizes where they can go wrong:
edges of the 16-, 32- and 64-key tiles and of the 16-, 32- and 128-row workgroups, one query on a long context, every
group size, padding masks (whole padded tiles, windows past 4,096 keys, rows without a real key), unaligned
views, and values that are not finite behind masked keys.  Against the oracle in float64."""

import math

import pytest
import torch

from oracle import torch_ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(b, h, hkv, tq, tk, dh, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(b, t, n, dh, generator=g).to(dtype).transpose(1, 2)
            for t, n in ((tq, h), (tk, hkv), (tk, hkv))]


def _run(q, k, v, key_valid=None):
    from minillm.attention import get_backend

    to = lambda x: x.transpose(1, 2).to(DEV).transpose(1, 2)  # noqa: E731  (keeps the [B, T, H, Dh] storage)
    return get_backend("hip").prefill(to(q), to(k), to(v), key_valid=None if key_valid is None else key_valid.to(DEV)).cpu()


def _compare(out, ref, dtype):
    if dtype == torch.float32:  # sums of up to 1,000 terms: a few times 2^-24 of the terms' size
        torch.testing.assert_close(out.double(), ref, rtol=1e-5, atol=1e-5)
        return
    # the output's own rounding (2^-8 bf16, 2^-11 fp16 of the value), plus the weights' 16 bits or more:
    # 2^-16 of |v| <= 6, and fp32 sums: 2e-4 covers both
    torch.testing.assert_close(out.double(), ref, rtol=2 ** (-8 if dtype == torch.bfloat16 else -11), atol=2e-4)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("b,h,hkv,tq,tk,dh", [
    (1, 4, 4, 1, 1, 128), (2, 8, 2, 31, 31, 64), (1, 8, 2, 33, 65, 128), (1, 32, 8, 1, 1000, 128), (3, 4, 4, 5, 129, 64),
    (1, 8, 1, 63, 64, 128), (1, 32, 1, 3, 97, 128), (2, 12, 4, 40, 71, 64), (2, 64, 64, 520, 520, 128),
    (3, 96, 32, 257, 384, 64), (1, 128, 8, 511, 701, 128)])
def test_edges(hip, dtype, b, h, hkv, tq, tk, dh):
    q, k, v = _inputs(b, h, hkv, tq, tk, dh, dtype)
    _compare(_run(q, k, v), torch_ref.prefill(q.double(), k.double(), v.double()), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("b,h,hkv,tq,tk", [(3, 8, 2, 70, 200), (4, 64, 64, 300, 333), (2, 2, 1, 3, 4700)])
def test_key_valid(hip, dtype, dh, b, h, hkv, tq, tk):
    q, k, v = _inputs(b, h, hkv, tq, tk, dh, dtype, seed=1)
    valid = torch.rand(b, tk, generator=torch.Generator().manual_seed(2)) < 0.7
    valid[0, :tk - tq // 2] = False  # the first queries of row 0 have no real key
    valid[1] = torch.arange(tk) >= tk // 2  # left padding of whole tiles
    if b > 2:
        valid[2] = False  # no real key at all
    _compare(_run(q, k, v, valid), torch_ref.prefill(q.double(), k.double(), v.double(), key_valid=valid), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_mask_windows_of_128_row_workgroups(hip, dtype):
    # 384 workgroups of 128 query rows on 4,700 keys, whose mask takes two windows of 4,096: a row whose first real key
    # lies in the second, one without a real key, one whose keys run through both
    from minillm import _native

    b, h, tq, tk = 3, 64, 256, 4700
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert _native.lib().fn("mllm_dense_rows")(b, h, 1, tq, 0) == 128
    q, k, v = _inputs(b, h, 1, tq, tk, 64, dtype, seed=8)
    valid = torch.rand(b, tk, generator=torch.Generator().manual_seed(9)) < 0.7
    valid[0, :4500] = False
    valid[1] = False
    _compare(_run(q, k, v, valid), torch_ref.prefill(q.double(), k.double(), v.double(), key_valid=valid), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("h", [2, 128])
def test_values_behind_masked_keys_do_not_leak(hip, dtype, h):
    # key 40 is not finite: queries before it and (masked) all queries of batch row 1 never see it
    b, t = 2, 300
    q, k, v = _inputs(b, h, h, t, t, 128, dtype, seed=3)
    valid = torch.ones(b, t, dtype=torch.bool)
    valid[1, 40] = False
    ref = torch_ref.prefill(q.double(), k.double(), v.double(), key_valid=valid)
    for bad in (float("nan"), float("inf")):
        v2 = v.clone()
        v2[:, :, 40, 7] = bad
        out = _run(q, k, v2, valid)
        _compare(out[0, :, :40], ref[0, :, :40], dtype)
        _compare(out[1], ref[1], dtype)
        seen = out[0, :, 40:, 7].float()
        assert (torch.isnan(seen) if bad != bad else seen == bad).all()
        _compare(out[0, :, 40:, 8:], ref[0, :, 40:, 8:], dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("b,h", [(1, 4), (3, 128)])  # workgroups of 32 and of 128 query rows
def test_weights_keep_fp32_precision(hip, dtype, b, h):
    # values of +-1 whose signs make the last query's weighted sum cancel, so that the error of the weights shows where
    # the output's rounding is far smaller; queries and keys of few bits and a scale of 1 / 8, so that the scores are exact
    t, dh = 128, 64
    q, k, _ = ((4 * x.float()).round().div(4).to(dtype) for x in _inputs(b, h, h, t, t, dh, dtype, seed=6))
    q = 2 * q
    p = torch.softmax((q[:, :, -1:].double() @ k.double().transpose(2, 3))[:, :, 0] * dh ** -0.5, -1)
    order = p.argsort(-1, descending=True)
    sign = (torch.rand(b, h, t, dh, generator=torch.Generator().manual_seed(7)) < 0.5).double() * 2 - 1
    total = torch.zeros(b, h, dh, dtype=torch.float64)
    for j in range(t):  # the eight largest weights at random, then each against the sum so far
        if j >= 8:
            sign[:, :, j] = torch.where(total > 0, -1.0, 1.0)
        total += p.gather(-1, order[..., j:j + 1]) * sign[:, :, j]
    v = torch.empty(b, h, t, dh).scatter_(2, order[..., None].expand(b, h, t, dh), sign.float()).to(dtype)
    got = _run(q, k, v)[:, :, -1].double()
    small = total.abs() < 2.0 ** -16
    assert int(small.sum()) > 100
    rms = (got - total)[small].square().mean().sqrt().item()
    # fp32 weights: off by two units of 2^-23 of themselves in random directions, and the squares of the weights sum to
    # about 0.3^2: 7e-8.  The sums: some ten additions rounded at 2^-25 of values below 1: 9e-8.  The output: 2^-9 of 2^-16.
    assert rms < 1.5e-7, rms


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("b,h", [(1, 4), (3, 128)])
def test_small_weights_keep_their_precision(hip, dtype, b, h):
    # key 0 takes nearly all the weight and has the value 0: what is left is the weight of key 1, 2^-4 to 2^-24, times a
    # large value
    t, dh = 128, 128
    q, k, v = (torch.zeros(b, h, t, dh) for _ in range(3))
    q[..., 0] = 16.0
    k[..., 0] = -48.0
    k[:, :, 0, 0] = 0.0
    drop = torch.linspace(4, 24, b * h).view(b, h)  # log2 of the weights' ratio
    k[:, :, 1, 0] = -drop * math.log(2) * dh ** 0.5 / 16
    v[:, :, 1] = 60000.0
    q, k, v = (x.to(dtype) for x in (q, k, v))
    ref = torch_ref.prefill(q.double(), k.double(), v.double())[:, :, -1]
    got = _run(q, k, v)[:, :, -1].double()
    # one rounding of the output; the exponent's 2^-24 of up to 17, and for fp16 weights the grid of their low part,
    # 2^-39 of the largest weight: 2^-15 covers both
    eps = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}[dtype]
    torch.testing.assert_close(got, ref, rtol=1.01 * eps + 2.0 ** -15, atol=0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("b,h", [(1, 4), (2, 128)])
def test_values_near_the_largest_stay_finite(hip, dtype, b, h):
    # key 200's score lies 2^7.5 above the rest, which holds the running max back, and its value is 2^-3 of the largest
    # there is: the output, a little less than that value, is finite however the sums are scaled on the way
    t, dh = 300, 64
    q, k, v = (torch.zeros(b, h, t, dh) for _ in range(3))
    q[..., 0] = 8.0
    k[:, :, 200, 0] = 7.5 * math.log(2)
    v[:, :, 200] = 4.2e37
    v[:, :, 200, 1::2] = -4.2e37
    q, k, v = (x.to(dtype) for x in (q, k, v))
    _compare(_run(q, k, v) * 2.0 ** -120, torch_ref.prefill(q.double(), k.double(), v.double()) * 2.0 ** -120, dtype)


def test_unaligned_rows_and_large_scores(hip):
    q, k, v = _inputs(1, 4, 2, 50, 80, 64, torch.float16, seed=4)
    wide = torch.zeros(1, 4, 50, 65, dtype=torch.float16)
    wide[..., 1:] = q
    _compare(_run(wide[..., 1:], k, v), torch_ref.prefill(q.double(), k.double(), v.double()), torch.float16)
    q, k = q * 30, k * 30  # scores of some thousands: one key takes all the weight, the max moves far
    _compare(_run(q, k, v), torch_ref.prefill(q.double(), k.double(), v.double()), torch.float16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_more_workgroups_than_a_launch_takes(hip, dtype):
    # 2^24 and more workgroups of 256 threads are past HIP's 2^32 work-items along x: those calls run on dense_kernel.
    # One query and one key each, so that a row's result is its value.
    from minillm.attention import get_backend

    b, h = 4096, 4096
    v = torch.randn(b, 1, 1, 64, generator=torch.Generator().manual_seed(5)).to(DEV, dtype).expand(b, h, 1, 64)
    q = k = torch.ones(1, 1, 1, 64, device=DEV, dtype=dtype).expand(b, h, 1, 64)
    assert torch.equal(get_backend("hip").prefill(q, k, v), v)
