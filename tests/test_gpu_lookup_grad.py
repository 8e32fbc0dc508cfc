"""The one-pass backward of the training lookup (``lng_lookup_grad``) against the order-by-order
kernels and the fp64 oracle, at the edges of its 64-window chunks and 16-window batches.

Tolerances: the route-logit gradient agrees with the direct kernels to fp32 rounding (norm-relative
1e-6: sums of 128 exact products in another order) and with fp64 to 1e-5; a table row of n windows
is an fp32 sum, n * 2^-24 * sum|g| off at most, then rounded once to bf16 (2^-8 relative)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from lngram_hip import ops
from oracle import memory as om

pytestmark = pytest.mark.gpu

# (B, T, R, route_start, codes, q dtype, codes dtype, strided gradient)
CASES = [
    (1, 1, 3, 0, "random", torch.float32, torch.uint8, False),      # no window of either order
    (1, 2, 3, 0, "random", torch.float32, torch.uint8, False),      # one order-2 window, none of order 3
    (2, 3, 9, 1, "random", torch.bfloat16, torch.int32, False),
    (1, 18, 5, 0, "constant", torch.float32, torch.uint8, False),   # 17 and 16 windows of one row
    (1, 66, 8, 0, "random", torch.float32, torch.uint8, True),      # 65 and 64 windows: chunk edge
    (1, 130, 8, 0, "random", torch.float32, torch.int64, True),     # 129 and 128 windows: chunk edge
    (3, 131, 17, 2, "few", torch.float32, torch.uint8, False),      # rows cut by chunks
    (2, 700, 3, 0, "constant", torch.float32, torch.uint8, False),  # one row over 22 chunks
    (5, 391, 11, 0, "random", torch.bfloat16, torch.uint8, True),
    (1, 64, 256, 0, "few", torch.float32, torch.uint8, False),
]


def _inputs(case, dev):
    B, T, R, rs, how, qdt, cdt, strided = case
    gen = torch.Generator().manual_seed(B * 997 + T)
    codes = torch.randint(0, 16, (B, T, R), generator=gen)
    if how == "constant":
        codes.fill_(9)
    elif how == "few":
        codes = codes % 3 + 6
    tables = [(torch.randn((rs + R) << (4 * o), 128, generator=gen) * 0.5).to(torch.bfloat16) for o in (2, 3)]
    q = torch.randn(B, T, R, 4, generator=gen).to(qdt)
    grad = torch.randn(B, T, R, 256, generator=gen).to(torch.bfloat16)
    vt = torch.ones(B, T, dtype=torch.bool)
    if T > 8 and how != "constant":
        vt[0, 5] = vt[B - 1, T - 2] = False
    masks = [torch.from_numpy(om.valid_mask(o, B, T, valid_tokens=vt.numpy())) for o in (2, 3)]
    g = grad.to(dev)
    if strided:
        wide = torch.full((B, T, R, 320), float("nan"), dtype=torch.bfloat16, device=dev)
        wide[..., 32:288] = g
        g = wide[..., 32:288]
    return codes, tables, q, grad, masks, (g, q.to(dev), codes.to(cdt).to(dev), [t.to(dev) for t in tables],
                                           [m.to(dev) for m in masks], (2, 3), 4, rs, 0.8, 1.2, False)


@pytest.mark.parametrize("case", CASES, ids=[f"{i}" for i in range(len(CASES))])
def test_equals_the_orders_kernels_and_fp64(dev, case):
    codes, tables, q, grad, masks, args = _inputs(case, dev)
    B, T, R, rs = case[:4]
    g, qd, cd, td, md = args[:5]
    assert ops.lib().lng_lookup_grad_workspace_bytes(B, T, R, 128, 4, ops.dtype_code(torch.bfloat16), 0) > 0
    gq, gt = ops.lookup_grad(*args, (True, True, True))
    per = [ops.surrogate_grad(g[..., i * 128:(i + 1) * 128].contiguous(), None, qd, cd, td[i], md[i], o, 4, rs, 0.8,
                              1.2, False, workspace=False) for i, o in enumerate((2, 3))]
    want = per[0] + per[1]
    assert gq.dtype == qd.dtype and gq.shape == want.shape
    if float(want.float().abs().max()) == 0:
        assert float(gq.float().abs().max()) == 0
    else:
        # bf16 logits: an fp32 difference may move a rounding of either part or of their sum
        assert om.rel_err(gq.float().cpu(), want.float().cpu()) < (1e-6 if qd.dtype == torch.float32 else 2.0 ** -8)
        hard = [torch.zeros_like(grad[..., :128]) for _ in range(2)]
        for i, o in enumerate((2, 3)):
            rows = om.route_rows(codes.numpy(), [o], 4, 0, R)[..., 0]
            at = torch.from_numpy(np.where(rows >= 0, rows + (rs << (4 * o)), 0))
            hard[i] = tables[i][at] * torch.from_numpy(rows >= 0)[..., None]
        ref = sum(om.surrogate_grad(grad[..., i * 128:(i + 1) * 128], hard[i], q, codes.numpy(), tables[i], masks[i], o,
                                    4, rs, 0.8, 1.2, False) for i, o in enumerate((2, 3)))
        assert om.rel_err(gq.float().cpu(), ref) < (1e-5 if qd.dtype == torch.float32 else 2.0 ** -7)
    for i, o in enumerate((2, 3)):
        rows = om.route_rows(codes.numpy(), [o], 4, 0, R)[..., 0]
        keep = (rows >= 0) & masks[i].numpy()[..., None]
        at = torch.from_numpy((rows + (rs << (4 * o)))[keep])
        src = grad[..., i * 128:(i + 1) * 128].double()[torch.from_numpy(keep)]
        ref, mass = (torch.zeros(tables[i].shape, dtype=torch.float64) for _ in range(2))
        ref.index_add_(0, at, src)
        mass.index_add_(0, at, src.abs())
        n = torch.from_numpy(np.bincount(at.numpy(), minlength=ref.shape[0]))[:, None]
        assert bool(((gt[i].cpu().double() - ref).abs() <= n * 2.0 ** -24 * mass + 2.0 ** -8 * ref.abs()).all())
        assert bool((gt[i].cpu()[n[:, 0] == 0] == 0).all())


def test_gradients_not_wanted_and_inactive(dev):
    args = list(_inputs(CASES[5], dev)[-1])
    gq, gt = ops.lookup_grad(*args, (True, True, True))
    for want in ((True, False, False), (False, True, False), (False, False, True)):
        q2, t2 = ops.lookup_grad(*args, want)
        assert (q2 is not None) == want[0] and [x is not None for x in t2] == list(want[1:])
        assert q2 is None or torch.equal(q2, gq)
    args[9] = 0.0                                                     # scale 0: no route gradient
    q0, t0 = ops.lookup_grad(*args, (True, True, True))
    assert float(q0.abs().max()) == 0 and om.rel_err(t0[0].float().cpu(), gt[0].float().cpu()) < 2.0 ** -8


@pytest.mark.parametrize("R,exact", [(257, False), (4, True)])
def test_other_shapes_take_the_orders_kernels(dev, R, exact):
    args = list(_inputs((1, 9, R, 0, "random", torch.float32, torch.uint8, False), dev)[-1])
    args[10] = exact
    assert ops.lib().lng_lookup_grad_workspace_bytes(1, 9, R, 128, 4, ops.dtype_code(torch.bfloat16), int(exact)) == 0
    gq, gt = ops.lookup_grad(*args, (True, True, True))
    per = [ops.surrogate_grad(args[0][..., i * 128:(i + 1) * 128].contiguous(), None, args[1], args[2], args[3][i],
                              args[4][i], o, 4, 0, 0.8, 1.2, exact) for i, o in enumerate((2, 3))]
    assert torch.equal(gq, per[0] + per[1]) and gt[0].shape == args[3][0].shape


@pytest.mark.parametrize("mean", [0.0, 1.0])        # rows with a common part: their scores cancel
def test_no_further_from_fp64_than_order_by_order(dev, mean):
    B, T, R = 2, 200, 64
    codes, tables, q, grad, masks, args = _inputs((B, T, R, 0, "random", torch.float32, torch.uint8, False), dev)
    tables = [(t.float() * 0.04 + mean).to(torch.bfloat16) for t in tables]
    args = args[:3] + ([t.to(dev) for t in tables],) + args[4:]
    g, qd, cd, td, md = args[:5]
    gq, _ = ops.lookup_grad(*args, (True, False, False))
    per = [ops.surrogate_grad(g[..., i * 128:(i + 1) * 128].contiguous(), None, qd, cd, td[i], md[i], o, 4, 0, 0.8, 1.2,
                              False, workspace=False) for i, o in enumerate((2, 3))]
    ref = 0
    for i, o in enumerate((2, 3)):
        rows = om.route_rows(codes.numpy(), [o], 4, 0, R)[..., 0]
        hard = tables[i][torch.from_numpy(rows.clip(0))] * torch.from_numpy(rows >= 0)[..., None]
        ref = ref + om.surrogate_grad(grad[..., i * 128:(i + 1) * 128].double(), hard.double(), q.double(), codes.numpy(),
                                      tables[i].double(), masks[i], o, 4, 0, 0.8, 1.2, False).double()
    one, many = (float((x.cpu().double() - ref).norm()) for x in (gq, per[0] + per[1]))
    assert one <= 1.02 * many                        # 102 400 sums: the two norms are known to under 1 %


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_values_that_are_not_finite_stay_where_they_are(dev, bad):
    case = (1, 130, 8, 0, "random", torch.float32, torch.uint8, False)
    codes, _, _, grad, _, args = _inputs(case, dev)
    gq, gt = ops.lookup_grad(*args, (True, True, True))
    t, r = 60, 3
    args[0][0, t, r, 7] = bad                        # the order-2 part of one window's gradient
    bq, bt = ops.lookup_grad(*args, (True, True, True))
    keep = torch.ones(1, 130, 8, dtype=torch.bool)
    keep[0, t - 1:t + 1, r] = False                  # the logits of its two positions
    assert torch.equal(bq[keep], gq[keep]) and not torch.isfinite(bq[~keep]).all(-1).any()
    row = r * 256 + int(codes[0, t - 1, r] + 16 * codes[0, t, r])
    rows = torch.arange(bt[0].shape[0]) != row
    # a row's own sum may add its windows in another order from call to call
    assert torch.isfinite(bt[0][rows].float()).all() and not torch.isfinite(bt[0][row, 7].float())
    assert om.rel_err(bt[0][rows].float().cpu(), gt[0][rows].float().cpu()) < 2.0 ** -8
    assert torch.isfinite(bt[1].float()).all()


def test_tables_of_two_types_go_order_by_order(dev):
    """A module whose tables were given different types by hand: rows and gradients of each order's own path."""
    from ffnmem.memory.lngram_v2 import RouteNgramMemoryV2

    R, B, T = 5, 2, 40
    m = RouteNgramMemoryV2(1024, num_routes=R, readout_num_kv_heads=4, readout_head_dim=64, table_init_std_scale=1.0,
                           device=dev, dtype=torch.float32).train()
    t2, t3 = (m.tables[f"ngram_{o}"] for o in (2, 3))
    t3.to(torch.bfloat16)
    gen = torch.Generator(device=dev).manual_seed(3)
    codes = torch.randint(0, 16, (B, T, R), generator=gen, device=dev, dtype=torch.uint8)
    q = torch.randn(B, T, R, 4, generator=gen, device=dev, requires_grad=True)
    grad = torch.randn(B, T, R, 256, generator=gen, device=dev)
    rows = m._lookup_route_chunk(codes, q, 0, R, None, None)
    gq, g2, g3 = torch.autograd.grad(rows, [q, t2.weight, t3.weight], grad)
    want_q = 0
    for i, (o, tab, g) in enumerate(((2, t2.weight, g2), (3, t3.weight, g3))):
        part, w = grad[..., i * 128:(i + 1) * 128], tab.detach()
        assert torch.equal(rows[..., i * 128:(i + 1) * 128], ops.route_tokens(codes, [w], [o], 4).float())
        valid = m._valid_mask(o, B, T, dev, None, None)
        part = part.to(w.dtype)                      # the concatenation's backward gives each part its own type
        want_q = want_q + ops.surrogate_grad(part, None, q.detach(), codes, w, valid, o, 4, 0, m.q_surrogate_temperature,
                                             m.q_surrogate_scale, False)
        want = ops.table_grad_rows(part, codes, valid, o, 4, 0, w.shape[0], w.dtype)
        assert g.dtype == w.dtype and om.rel_err(g.float().cpu(), want.float().cpu()) < (1e-6 if i == 0 else 2.0 ** -8)
    assert om.rel_err(gq.cpu(), want_q.cpu()) < 1e-6


def test_the_logits_gradient_repeats_and_a_table_row_keeps_its_bound(dev):
    """The order of a row's windows may vary between calls: the logits' gradient does not depend on it, a
    table row of n windows by n * 2^-24 * sum|g| and one bf16 rounding at most."""
    codes, tables, q, grad, masks, args = _inputs((2, 700, 9, 0, "few", torch.float32, torch.uint8, False), dev)
    first = ops.lookup_grad(*args, (True, True, True))
    mass = ops.lookup_grad(args[0].abs(), *args[1:], (False, True, True))[1]
    for _ in range(5):
        gq, gt = ops.lookup_grad(*args, (True, True, True))
        assert torch.equal(gq, first[0])
        for a, b, m in zip(gt, first[1], mass):
            bound = 2 * 1400 * 2.0 ** -24 * 1.01 * m.float() + 2.0 ** -7 * torch.maximum(a.float().abs(), b.float().abs())
            assert bool(((a.float() - b.float()).abs() <= bound).all())
