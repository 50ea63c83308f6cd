"""``gemv`` on the register kernel: the edges of its rows per wave (2 and 8), of the chunks per lane and
of the batch, against FP64, and row for row against the general kernel (an input that is not 16-byte
aligned), which adds the same products in the same order."""

import pytest
import torch

from iris_mi355x import kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n,k", [(1, 256), (7, 512), (8191, 264), (8192, 256), (8201, 512), (2561, 2560), (8195, 2056)])
@pytest.mark.parametrize("batch", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("extra", [0, 1, 9])
def test_gemv_rows(n, k, batch, extra):
    g = torch.Generator(device=DEV).manual_seed(50)
    w = (0.05 * torch.randn(n, k, generator=g, device=DEV)).to(torch.bfloat16)
    w[n // 2, k - 1] = float("inf")  # reaches its own row only
    flat = torch.randn(batch * k + 1, generator=g, device=DEV).abs()
    x, x_odd = flat[:-1].view(batch, k), flat.clone()[1:].view(batch, k)
    x_odd.copy_(x)
    bias = torch.randn(n, generator=g, device=DEV)
    add = torch.randn(extra, n, generator=g, device=DEV) if extra else None
    shape = (extra, batch, n) if extra else (batch, n)
    for acts in ({}, {"in_silu": True, "out_silu": True}):
        out, odd = (torch.full(shape, 7.0, device=DEV) for _ in range(2))
        K.gemv(w, x.contiguous(), bias, out, extra_bias=add, **acts)
        K.gemv(w, x_odd, bias, odd, extra_bias=add, **acts)
        assert torch.equal(out, odd)
        xd = x.double()
        want = (torch.nn.functional.silu(xd) if acts else xd) @ w.double().T + bias.double()
        want = torch.nn.functional.silu(want) if acts else want
        want = want + add.double()[:, None] if extra else want
        assert torch.equal(torch.isinf(out), torch.isinf(want))
        # k <= 2560 products of N(0, 0.05) in FP32 (and silu's ~1 ulp reciprocal): 2^-24 sqrt(k) of their sum
        ok = torch.isfinite(want)
        torch.testing.assert_close(out.double()[ok], want[ok], rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("ns,k", [((8200, 37), 256), ((7, 1), 512), ((9000, 8192), 2560), ((40, 24), 520)])
@pytest.mark.parametrize("batch", [1, 2, 4, 7])
def test_gemv_pair_is_two_gemvs(ns, k, batch):
    """Two products in one launch, exactly as two calls (520: the general kernel)."""
    g = torch.Generator(device=DEV).manual_seed(51)
    ws = [(0.05 * torch.randn(n, k, generator=g, device=DEV)).to(torch.bfloat16) for n in ns]
    x = torch.randn(batch, k, generator=g, device=DEV)
    biases = [torch.randn(n, generator=g, device=DEV) for n in ns]
    extras = [torch.randn(j, n, generator=g, device=DEV) for j, n in zip((24, 8), ns)]
    outs = [[torch.full((e.shape[0], batch, n), 7.0, device=DEV) for e, n in zip(extras, ns)] for _ in range(2)]
    K.gemv_pair(ws, x, biases, outs[0], extras, in_silu=True)
    for w, b, o, e in zip(ws, biases, outs[1], extras):
        K.gemv(w, x, b, o, extra_bias=e, in_silu=True)
    for got, want in zip(*outs):
        assert torch.equal(got, want)


@pytest.mark.parametrize("n,half", [(2560, 128), (1, 4), (259, 256), (8195, 100)])
@pytest.mark.parametrize("batch", [1, 3, 6])
def test_timestep_gemv_is_features_then_gemv(n, half, batch):
    g = torch.Generator(device=DEV).manual_seed(52)
    w = (0.05 * torch.randn(n, 2 * half, generator=g, device=DEV)).to(torch.bfloat16)
    bias = torch.randn(n, generator=g, device=DEV)
    t, freqs = 1000 * torch.rand(batch, generator=g, device=DEV), torch.rand(half, generator=g, device=DEV)
    features, out, want = (torch.empty(batch, m, device=DEV) for m in (2 * half, n, n))
    K.timestep_gemv(t, freqs, w, bias, out, out_silu=True)
    K.gemv(w, K.timestep_features(t, freqs, features), bias, want, out_silu=True)
    assert torch.equal(out, want)
