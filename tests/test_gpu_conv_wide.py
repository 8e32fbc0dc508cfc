"""The kernel-4, dilation-3 short conv of wide rows (several outputs a thread) at the edges of its tiles
and rounds: fp64 within the sums' rounding (1e-6 fp32; 2^-7 bf16, three roundings), and the last
positions alone, a small launch, bit for bit."""

from __future__ import annotations

import pytest
import torch

from lngram_hip import ops
from oracle import memory as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,t,d,dt", [
    (1, 1, 384, torch.float32), (2, 7, 392, torch.float32), (1, 9, 1024, torch.float32),
    (1, 64, 768, torch.float32),       # 8 tiles: mapped to the XCDs
    (2, 66, 2048, torch.float32),      # 9 tiles: not
    (8, 1024, 400, torch.float32),     # 512 tiles of 16
    (8, 1029, 512, torch.float32), (3, 70, 4096, torch.bfloat16), (40, 208, 2560, torch.bfloat16)])
def test_wide_rows(dev, b, t, d, dt):
    gen = torch.Generator().manual_seed(t + d)
    x = torch.randn(b, t, d, generator=gen).to(dt)
    nw, cw = torch.rand(d, generator=gen).to(dt) + 0.5, (torch.randn(d, 1, 4, generator=gen) * 0.3).to(dt)
    xd, nd, cd = x.to(dev), nw.to(dev), cw.to(dev)
    got = ops.causal_conv(xd, nd, cd, 3, 1e-5)
    xn = x.double() * torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + 1e-5) * nw.double()
    y = torch.zeros_like(xn)
    for k in range(4):
        back = 9 - 3 * k
        if back < t:
            y[:, back:] += xn[:, :t - back] * cw.double()[:, 0, k]
    assert om.rel_err(got.cpu(), x.double() + y * torch.sigmoid(y)) < (1e-6 if dt == torch.float32 else 2.0 ** -7)
    for n in (1, 3, 17):
        if n < t:
            tail = ops.causal_conv_at(xd, nd, cd, 3, 1e-5, pos0=t - n, n=n)
            assert torch.equal(tail, got[:, t - n:])
    x2 = xd.clone()                                            # not finite: its row and the nine after it, no others
    x2[0, t // 2, d - 1] = float("nan")
    bad, keep = ops.causal_conv(x2, nd, cd, 3, 1e-5), torch.ones(b, t, dtype=torch.bool, device=dev)
    keep[0, t // 2:t // 2 + 10:3] = False
    assert torch.equal(bad[keep], got[keep]) and not torch.isfinite(bad[0, t // 2].float()).all()
