"""
moehip_dense_gemm_int8 (QLinear for a few tokens) against the dequantised weights' product in
float64: token counts around the 32-token tiles and the 64-token passes, ragged row counts at each
of the kernel's rows-per-workgroup choices, K of one group up to several rounds of the four waves,
with and without bias. Bar: one rounding of the output (the sums are fp32 over exact products).
"""

import numpy as np
import pytest
import torch

from moelab_hip import denseq as D

pytestmark = pytest.mark.gpu

ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _check(dev, T, O, K, dtype, bias, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randint(-127, 128, (O, K), generator=g, dtype=torch.int8)
    s = (torch.rand(O, K // 64, generator=g) * 2e-3 + 1e-4).half()
    b = torch.randn(O, generator=g).to(dtype) if bias else None
    x = torch.randn(T, K, generator=g).to(dtype)
    ql = D.QLinear(q.to(dev), s.to(dev), 64, None if b is None else b.to(dev), dtype)
    assert ql._few(x.to(dev))
    y = ql(x.to(dev))
    assert y.shape == (T, O) and y.dtype == dtype
    w = (q.to(dev).double().view(O, K // 64, 64) * s.to(dev).double().unsqueeze(-1)).view(O, K)
    xd = x.to(dev).double()
    ref = xd @ w.t()
    mag = xd.abs() @ w.abs().t()
    if bias:
        ref, mag = ref + b.to(dev).double(), mag + b.to(dev).double().abs()
    # half an ulp of the result, and fp32 sums of K products (K * 2^-24 of the summed magnitudes)
    bar = ULP[dtype] * ref.abs() + K * 2.0 ** -24 * mag + 1e-7
    assert bool(((y.double() - ref).abs() <= bar).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T", [2, 31, 32, 33, 64, 65, 130, 256])
@pytest.mark.parametrize("O,K", [(33, 64), (130, 192), (100, 640), (2048, 2048)])
def test_dense_gemm_int8(dev, T, O, K, dtype):
    _check(dev, T, O, K, dtype, bias=(T + O) % 2 == 1, seed=T * 7 + O)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T,O", [(3, 32801), (17, 32801), (32, 32700), (64, 32801), (70, 16400)])
def test_dense_gemm_int8_many_rows(dev, T, O, dtype):
    _check(dev, T, O, 192, dtype, bias=False, seed=T + O)


def test_dense_gemm_int8_routes(dev):
    """What the kernel does not take goes the dequantised way: fp32 activations, other groups, an
    input at an odd address, many tokens; an input that wants a gradient is refused as before."""
    g = torch.Generator().manual_seed(1)
    q = torch.randint(-127, 128, (96, 128), generator=g, dtype=torch.int8).to(dev)
    ql = D.QLinear(q, torch.full((96, 2), 1e-3, dtype=torch.float16, device=dev), 64, None, torch.float16)
    x = torch.randn(4, 128, generator=g).to(dev)
    odd = torch.zeros(4 * 128 + 1, dtype=torch.float16, device=dev)[1:].view(4, 128).copy_(x)
    many = torch.zeros(D.FEW_TOKENS + 1, 128, dtype=torch.float16, device=dev)
    q32 = D.QLinear(q, torch.full((96, 4), 1e-3, dtype=torch.float16, device=dev), 32, None, torch.float16)
    for m, v in ((ql, x), (ql, odd), (ql, many), (q32, x.half())):
        assert not m._few(v)
        ref = v.double() @ (q.double() * float(torch.tensor(1e-3, dtype=torch.float16))).t()
        assert np.allclose(m(v).double().cpu(), ref.cpu(), rtol=2e-3, atol=2e-3)
    assert ql._few(x.half())
    with pytest.raises(RuntimeError):
        ql(x.half().requires_grad_())


def test_dense_gemm_int8_other_calls(dev):
    """No tokens, a strided bias, a trainable bias and a forward-mode tangent: as the dequantised way
    takes or refuses them."""
    g = torch.Generator().manual_seed(2)
    q = torch.randint(-127, 128, (96, 128), generator=g, dtype=torch.int8).to(dev)
    s = torch.full((96, 2), 1e-3, dtype=torch.float16, device=dev)
    x = torch.randn(4, 128, generator=g).half().to(dev)
    bias = torch.randn(192, generator=g).half().to(dev)[::2]
    ql = D.QLinear(q, s, 64, bias, torch.float16)
    assert ql(x[:0]).shape == (0, 96) and ql(x.new_zeros(2, 0, 128)).shape == (2, 0, 96)
    ref = x.double() @ (q.double() * s[0, 0].double()).t() + bias.double()
    assert ql._few(x) and np.allclose(ql(x).double().cpu(), ref.cpu(), rtol=2e-3, atol=2e-3)
    with torch.autograd.forward_ad.dual_level():
        assert not ql._few(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))
    ql.bias.requires_grad_(True)
    assert not ql._few(x)
    with pytest.raises(RuntimeError):
        ql(x)
