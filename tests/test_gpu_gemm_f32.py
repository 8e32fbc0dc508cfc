"""fp32 products on the matrix cores (``lng_linear`` fp32) and bf16 rows against split fp32 weights
(``lng_linear_split``) at the edges of their tiles.

An output is an fp32 sum of K products: K * 2^-24 * sum|x w| off at most.  The split form's products
are exact; its weight (norm_w * w) is rounded once to fp32, its pieces hold 24 bits of it, and the row
scale costs a few roundings: 2^-21 relative besides the sum's error."""

from __future__ import annotations

import pytest
import torch

from lngram_hip import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1, 1, 32), (33, 35, 64), (512, 32, 128), (512, 256, 64), (1024, 1024, 96),
                                   (1025, 1024, 32), (4100, 260, 160), (70, 30, 40)])
def test_linear_fp32(dev, m, n, k):
    gen = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn(m, k, generator=gen), torch.randn(n, k, generator=gen)
    got = ops.linear(x.to(dev), w.to(dev)).cpu().double()
    ref = x.double() @ w.double().t()
    err = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert bool(((got - ref).abs() <= err).all())
    # a row's result does not depend on the rows beside it
    assert torch.equal(ops.linear(x[m - 1:].to(dev), w.to(dev)).cpu().double()[0], got[m - 1])


@pytest.mark.parametrize("m,n,k", [(1, 256, 1024), (31, 4, 64), (97, 36, 128), (3072, 256, 192), (3073, 256, 128),
                                   (8192, 256, 64), (8193, 256, 64)])
def test_norm_linear_split(dev, m, n, k):
    gen = torch.Generator().manual_seed(m + n + k)
    x = (torch.randn(m, k, generator=gen) * 0.02).to(torch.bfloat16)
    w, nw = torch.randn(n, k, generator=gen) * 0.02, torch.rand(k, generator=gen) + 0.5
    assert ops.lib().lng_linear_split_workspace_bytes(n, k) > 0
    got = ops.norm_linear_fp32(x.to(dev), nw.to(dev), w.to(dev), 1e-5).cpu().double()
    y = x.double() * torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + 1e-5) * nw.double()
    ref, mass = y @ w.double().t(), y.abs() @ w.double().abs().t()
    # 3 k terms are summed (each weight's pieces)
    assert bool(((got - ref).abs() <= (3 * k * 2.0 ** -24 + 2.0 ** -21) * mass).all())
    two = ops.norm_linear_fp32(x[m - 1:].to(dev), nw.to(dev), w.to(dev), 1e-5).cpu().double()
    assert torch.equal(two[0], got[m - 1])


def test_norm_linear_other_shapes(dev):
    gen = torch.Generator().manual_seed(2)
    x, w, nw = torch.randn(9, 72, generator=gen), torch.randn(8, 72, generator=gen), torch.ones(72)
    for xt in (x.to(torch.bfloat16), x):                      # K % 64 != 0; fp32 rows
        got = ops.norm_linear_fp32(xt.to(dev), nw.to(dev), w.to(dev), 1e-5)
        assert torch.equal(got, ops.linear(ops.rmsnorm(xt.to(dev).float(), nw.to(dev), 1e-5), w.to(dev)))
