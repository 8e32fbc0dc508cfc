"""The listed table gradient (``lng_table_grad_rows``) against an fp64 scatter of the same rows.

Error bound per element: a row of n windows is an fp32 sum of n terms, so at most n * 2^-24 * sum|g|,
plus one rounding to the output dtype (2^-8 relative for bf16, half of it to nearest, doubled for
the sum's own error at a rounding boundary)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from lngram_hip import ops
from oracle import memory as om

pytestmark = pytest.mark.gpu

# (B, T, R, route_start, D, order, bits, gradient dtype, table dtype, codes, gradient layout)
CASES = [
    (1, 1, 1, 0, 32, 2, 4, torch.float32, torch.float32, "random", "own"),       # no window at all
    (1, 3, 3, 0, 128, 3, 4, torch.bfloat16, torch.bfloat16, "random", "slice"),  # one window a route
    (1, 63, 65, 0, 128, 2, 4, torch.bfloat16, torch.bfloat16, "random", "slice"),
    (3, 64, 64, 2, 64, 3, 2, torch.bfloat16, torch.float32, "random", "own"),
    (2, 65, 5, 1, 256, 1, 4, torch.float32, torch.bfloat16, "random", "own"),
    (5, 391, 9, 0, 128, 3, 4, torch.bfloat16, torch.bfloat16, "random", "slice"),
    (2, 1500, 3, 0, 128, 2, 4, torch.bfloat16, torch.bfloat16, "constant", "slice"),  # one row of 2998 windows
    (1, 1026, 2, 0, 256, 2, 4, torch.float32, torch.float32, "constant", "slice"),    # 1025: just past a group's share
    (1, 1025, 2, 0, 32, 2, 4, torch.float32, torch.float32, "constant", "own"),       # 1024: the last it takes
    (2, 300, 4, 0, 32, 4, 3, torch.float32, torch.float32, "random", "slice"),
    (1, 700, 2, 0, 64, 1, 1, torch.bfloat16, torch.float32, "random", "own"),
]


@pytest.mark.parametrize("case", CASES, ids=[f"{i}" for i in range(len(CASES))])
@pytest.mark.parametrize("codes_dtype", [torch.uint8, torch.int32])
def test_rows_match_scatter(dev, case, codes_dtype):
    B, T, R, rs, D, order, bits, gdt, odt, how, layout = case
    gen = torch.Generator().manual_seed(B * 1000 + T)
    hi = 1 << bits
    codes = torch.full((B, T, R), hi - 1) if how == "constant" else torch.randint(0, hi, (B, T, R), generator=gen)
    grad = torch.randn(B, T, R, D, generator=gen).to(gdt)
    vt = torch.ones(B, T, dtype=torch.bool)
    if how == "random" and T > 8:
        vt[0, 5] = vt[B - 1, T - 3] = False
    valid = torch.from_numpy(om.valid_mask(order, B, T, valid_tokens=vt.numpy()))
    n_rows = (rs + R) << (bits * order)
    if layout == "slice":
        wide = torch.full((B, T, R, 2 * D), float("nan"), dtype=gdt, device=dev)
        wide[..., D:] = grad.to(dev)
        g = wide[..., D:]
    else:
        g = grad.to(dev)
    assert ops.lib().lng_table_grad_workspace_bytes(B, T, R, order, bits) > 0
    got = ops.table_grad_rows(g, codes.to(codes_dtype).to(dev), valid.to(dev), order, bits, rs, n_rows, odt)
    assert got.dtype == odt and tuple(got.shape) == (n_rows, D)
    rows = om.route_rows(codes.numpy(), [order], bits, 0, R)[..., 0]
    keep = (rows >= 0) & valid.numpy()[..., None]
    at = torch.from_numpy((rows + rs * (1 << (bits * order)))[keep])
    src = grad.double()[torch.from_numpy(keep)]
    want, mass = torch.zeros(n_rows, D, dtype=torch.float64), torch.zeros(n_rows, D, dtype=torch.float64)
    want.index_add_(0, at, src)
    mass.index_add_(0, at, src.abs())
    n = torch.from_numpy(np.bincount(at.numpy(), minlength=n_rows))[:, None]
    bound = n * 2.0 ** -24 * mass + (2.0 ** -8 if odt == torch.bfloat16 else 2.0 ** -24) * want.abs()
    assert bool(((got.cpu().double() - want).abs() <= bound).all())
    assert bool((got.cpu()[n[:, 0] == 0] == 0).all())


def test_shapes_past_the_counters_take_the_atomic_form(dev):
    B, T, R, D, order, bits = 1, 20, 1, 32, 4, 4                    # 65,536 rows a route
    assert ops.lib().lng_table_grad_workspace_bytes(B, T, R, order, bits) == 0
    gen = torch.Generator().manual_seed(3)
    grad = torch.randn(B, T, R, D, generator=gen).to(dev)
    codes = torch.randint(0, 16, (B, T, R), generator=gen, dtype=torch.uint8).to(dev)
    valid = torch.ones(B, T, dtype=torch.bool, device=dev)
    a = ops.table_grad_rows(grad, codes, valid, order, bits, 0, R << 16, torch.float32)
    assert om.rel_err(a.cpu(), ops.table_grad(grad, codes, valid, order, bits, 0, R << 16).cpu()) < 1e-6
