"""The kernel-4, dilation-3 short conv (fp32, and bf16 widths past the fused kernel's) at the edges of its
position tiles: fp64 within the sums' rounding (1e-6 fp32; 2^-7 bf16, three roundings), and a window of
cached rows bit for bit."""

from __future__ import annotations

import pytest
import torch

from lngram_hip import ops
from oracle import memory as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,t,d,dt", [(1, 1, 8, torch.float32), (2, 7, 128, torch.float32), (1, 8, 520, torch.float32),
                                      (3, 17, 1024, torch.float32), (32, 257, 64, torch.float32),
                                      (2, 33, 2056, torch.bfloat16), (40, 200, 2056, torch.bfloat16)])
def test_short_conv_tiles(dev, b, t, d, dt):
    gen = torch.Generator().manual_seed(t + d)
    x = torch.randn(b, t, d, generator=gen).to(dt)
    nw, cw = torch.rand(d, generator=gen).to(dt) + 0.5, (torch.randn(d, 1, 4, generator=gen) * 0.3).to(dt)
    got = ops.causal_conv(x.to(dev), nw.to(dev), cw.to(dev), 3, 1e-5)
    xn = x.double() * torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + 1e-5) * nw.double()
    y = torch.zeros_like(xn)
    for k in range(4):
        back = 9 - 3 * k
        if back < t:
            y[:, back:] += xn[:, :t - back] * cw.double()[:, 0, k]
    ref = x.double() + y * torch.sigmoid(y)
    assert om.rel_err(got.cpu(), ref) < (1e-6 if dt == torch.float32 else 2.0 ** -7)
    # a window of cached rows gives the same outputs
    if t > 4:
        tail = ops.causal_conv_at(x.to(dev), nw.to(dev), cw.to(dev), 3, 1e-5, pos0=t - 3, n=3)
        assert torch.equal(tail, got[:, t - 3:])
