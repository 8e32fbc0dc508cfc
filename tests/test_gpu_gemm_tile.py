"""The tiled bf16 GEMMs between the skinny kernel and the 256-row tiles: every tile of the choice at
its edges (rows and columns past the last tile, the blocks that end each tile's range).

bf16 products are exact in fp32, so an output is an fp32 sum of K terms: K * 2^-24 * sum|x w| off at
most, plus the output's rounding.  Codes are compared where the logit is past that bound."""

from __future__ import annotations

import pytest
import torch

from lngram_hip import ops

pytestmark = pytest.mark.gpu

# (M, K, N): the tile each takes is noted as columns x rows (plain / with row statistics)
SHAPES = [
    (65, 64, 32),        # 32x32, one K stage
    (97, 128, 36),       # 32x32, N past a tile by 4
    (640, 1024, 1024),   # 32x32: 640 blocks, its last
    (641, 1024, 1024),   # 64x32
    (1280, 192, 1024),   # 64x32: 640 blocks, its last; three K stages
    (1281, 256, 1024),   # 64x64
    (3072, 64, 1020),    # 64x64: 768 blocks, its last
    (3073, 1024, 1024),  # 128x64
    (1536, 320, 1000),   # row statistics on 128x32: 384 blocks, its last
    (1537, 320, 1000),   # row statistics on 128x64
    (6144, 128, 1024),   # 128x64: 768 blocks, its last
    (6145, 128, 1024),   # past the tiles
    (4096, 2304, 724),   # router of 128x64
]


def _inputs(m, k, n, dev):
    gen = torch.Generator().manual_seed(m + k + n)
    x, w = torch.randn(m, k, generator=gen).to(torch.bfloat16), torch.randn(n, k, generator=gen).to(torch.bfloat16)
    ref = (x.double().to(dev) @ w.double().to(dev).t()).cpu()
    err = k * 2.0 ** -24 * (x.double().abs().to(dev) @ w.double().abs().to(dev).t()).cpu()
    return x.to(dev), w.to(dev), ref, err


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_linear_and_row_statistics(dev, m, k, n):
    x, w, ref, err = _inputs(m, k, n, dev)
    bound = err + 2.0 ** -8 * ref.abs()
    assert bool(((ops.linear(x, w).cpu().double() - ref).abs() <= bound).all())
    y, rowsq = ops.linear_rowsq(x, w)
    assert bool(((y.cpu().double() - ref).abs() <= bound).all())
    got, want = rowsq.cpu().double().sum(0), y.cpu().double().pow(2).sum(-1)
    assert bool(((got - want).abs() <= n * 2.0 ** -23 * want).all())
    if ops.linear_rowscale_ok(x, w):
        s = torch.rsqrt(x.cpu().double().pow(2).mean(-1, keepdim=True) + 1e-5)
        # the scale is a hardware reciprocal square root of an fp32 sum (under 2^-20 relative)
        got = ops.linear_rowscale(x, w, 1e-5).cpu().double()
        assert bool(((got - ref * s).abs() <= (bound + 2.0 ** -20 * ref.abs()) * s).all())


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("codes_dtype", [torch.uint8, torch.int32])
def test_router_codes(dev, m, k, n, codes_dtype):
    x, w, ref, err = _inputs(m, k, n, dev)
    logits, codes = ops.router_codes(x, w, 4, want_logits=True, codes_dtype=codes_dtype)
    assert bool(((logits.cpu().double() - ref).abs() <= err + 2.0 ** -24 * ref.abs()).all())
    bit = 1 << torch.arange(4)
    want = ((ref > 0).view(m, n // 4, 4).long() * bit).sum(-1)
    clear = (ref.abs() > err).view(m, n // 4, 4).all(-1)
    assert codes.dtype == codes_dtype and bool((codes.cpu().long() == want)[clear].all())
    assert torch.equal(ops.router_codes(x, w, 4, want_logits=False, codes_dtype=codes_dtype)[1], codes)
