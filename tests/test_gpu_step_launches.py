"""Launches that hold two steps: the router and query projection of a decode step, and the fp32 router
with its codes."""

from __future__ import annotations

import pytest
import torch

from lngram_hip import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,n,k,routes,kq,nq", [(1, 1, 32, 4, 64, 16), (8, 1, 1024, 184, 1024, 1024),
                                                (4, 16, 2304, 181, 1024, 1024), (3, 5, 64, 8, 96, 48)])
@pytest.mark.parametrize("on_device", [False, True])
def test_router_and_query_equal_the_two_calls(dev, b, n, k, routes, kq, nq, on_device):
    gen = torch.Generator().manual_seed(b * n + k)

    def rnd(*s):
        return torch.randn(*s, generator=gen).to(torch.bfloat16).to(dev)

    x, w, h, wq = rnd(b, n, k), rnd(4 * routes, k), rnd(b, n, kq), rnd(nq, kq)
    one, two = (torch.full((b, n + 7, routes), 77, dtype=torch.uint8, device=dev) for _ in range(2))
    pos = dict(pos0_dev=torch.tensor([3], dtype=torch.int32, device=dev)) if on_device else dict(pos0=3)
    if 4 * routes % 16:
        with pytest.raises(RuntimeError, match="N % 16"):
            ops.router_query_at(x, w, one, h, wq, **pos)
        return
    q = ops.router_query_at(x, w, one, h, wq, **pos)
    ops.router_codes_at(x, w, two, **pos)
    assert torch.equal(one, two) and torch.equal(q, ops.linear(h, wq))


@pytest.mark.parametrize("m,k,n", [(1, 32, 4), (33, 64, 36), (512, 128, 32), (1100, 32, 1024)])
@pytest.mark.parametrize("codes_dtype", [torch.uint8, torch.int32])
def test_fp32_router_codes_are_the_logits_signs(dev, m, k, n, codes_dtype):
    gen = torch.Generator().manual_seed(m + n)
    x, w = torch.randn(m, k, generator=gen).to(dev), torch.randn(n, k, generator=gen).to(dev)
    x[0] = 0.0                                                       # logits of exactly 0 are not positive
    logits, codes = ops.router_codes(x, w, 4, codes_dtype=codes_dtype)
    assert torch.equal(logits, ops.linear(x, w))
    assert codes.dtype == codes_dtype and torch.equal(codes, ops.pack_route_codes(logits, 4, codes_dtype))
