"""The tiled route-token gather (``lng_route_tokens``) at its edges, bit for bit against the oracle's
rows: tiles of 64 positions, row widths of one piece to a block's threads, masks, route ranges and
tails, and outputs on both sides of the non-temporal store line."""

from __future__ import annotations

import pytest
import torch

from lngram_hip import ops
from lngram_hip._lib import check
from oracle import memory as om

pytestmark = pytest.mark.gpu

# (B, T, R, route_start, route_end, D, orders, bits, dtype, target_length, masked)
CASES = [
    (1, 1, 1, 0, 1, 8, (2, 3), 4, torch.bfloat16, None, False),          # small: one thread a piece
    (1, 63, 184, 0, 184, 128, (2, 3), 4, torch.bfloat16, None, True),    # 5.9 MB: one short tile
    (1, 64, 201, 3, 201, 64, (1, 2, 3, 4), 2, torch.bfloat16, None, True),
    (3, 65, 181, 0, 181, 128, (2, 3), 4, torch.bfloat16, 31, True),      # tails across tiles
    (64, 400, 11, 0, 11, 8, (2, 3), 4, torch.bfloat16, None, False),     # one-piece rows
    (2, 260, 3, 0, 3, 1024, (1,), 4, torch.float32, None, False),        # 4 KB rows: one row a block pass
    (9, 129, 40, 1, 39, 32, (2, 3), 4, torch.float32, None, True),
    (2, 300, 97, 0, 97, 24, (2, 3), 4, torch.bfloat16, None, True),      # 48 bytes: one thread a piece
    (5, 391, 33, 0, 33, 128, (2, 3), 4, torch.bfloat16, None, True),     # 33.0 MB: non-temporal stores
    (1, 63, 300, 0, 300, 128, (2, 3), 4, torch.bfloat16, None, True),    # past the tiled copy's line: one short tile
    (1, 96, 201, 3, 201, 64, (1, 2, 3, 4), 2, torch.bfloat16, None, True),
    (3, 260, 3, 0, 3, 1024, (1,), 4, torch.float32, None, False),        # 4 KB rows: one row a block pass
    (1, 4100, 20, 2, 19, 128, (2, 3), 4, torch.bfloat16, None, True),    # as many positions as rows a route
]


@pytest.mark.parametrize("case", CASES, ids=[f"{i}" for i in range(len(CASES))])
@pytest.mark.parametrize("codes_dtype", [torch.uint8, torch.int64])
def test_rows_equal_the_oracle(dev, case, codes_dtype):
    B, T, R, r0, r1, D, orders, bits, dt, tail, masked = case
    gen = torch.Generator().manual_seed(T)
    codes = torch.randint(0, 1 << bits, (B, T, R), generator=gen)
    tables = [torch.randn(R << (bits * o), D, generator=gen).to(dt) for o in orders]
    seg = val = None
    if masked:
        seg = torch.zeros(B, T, dtype=torch.int64)
        seg[:, T // 2:] = 1
        val = torch.rand(B, T, generator=gen) > 0.1
    got = ops.route_tokens(codes.to(codes_dtype).to(dev), [t.to(dev) for t in tables], orders, bits, r0, r1,
                           None if seg is None else seg.to(dev), None if val is None else val.to(dev), tail)
    rows = torch.from_numpy(om.route_rows(codes.numpy(), orders, bits, 0, R, segment_ids=None if seg is None else
                                          seg.numpy(), valid_tokens=None if val is None else val.numpy()))
    want = torch.cat([torch.where((rows[..., i] >= 0)[..., None], tab[rows[..., i].clamp_min(0)], torch.zeros(1, dtype=dt))
                      for i, tab in enumerate(tables)], -1)[:, :, r0:r1]
    want = want if tail is None else want[:, -tail:]
    assert torch.equal(got.cpu(), want)


def test_only_the_training_lookup_reads_ahead(dev, monkeypatch):
    """A gather cannot tell whether its tables are cached: only the step that knows they are not, because its
    backward came between, reads them first."""
    from ffnmem.memory.lngram_v2 import RouteNgramMemoryV2

    seen = []
    real = ops._prefetch_tables
    monkeypatch.setattr(ops, "_prefetch_tables", lambda *a: seen.append(1) or real(*a))
    m = RouteNgramMemoryV2(1024, num_routes=20, readout_num_kv_heads=4, readout_head_dim=64, table_init_std_scale=1.0,
                           device=dev, dtype=torch.bfloat16)
    codes = torch.randint(0, 16, (1, 4100, 20), dtype=torch.uint8, device=dev)
    q = torch.randn(1, 4100, 20, 4, device=dev, requires_grad=True)
    tables = [m.tables[f"ngram_{o}"].weight.detach() for o in (2, 3)]
    with torch.no_grad():
        want = ops.route_tokens(codes, tables, (2, 3), 4)
        m.eval()._lookup_route_chunk(codes, q, 0, 20, None, None)
    assert not seen
    assert torch.equal(m.train()._lookup_route_chunk(codes, q, 0, 20, None, None).detach(), want) and seen


@pytest.mark.parametrize("lo,n", [(0, 0), (1, 15), (0, 16), (8, 40), (3, 70001), (0, 64 << 20)])
def test_reading_ahead_changes_nothing(dev, lo, n):
    x = torch.arange(lo + n + 32, device=dev).to(torch.uint8)
    want = x.clone()
    check(ops.lib().lng_prefetch_rows(x.data_ptr() + lo, n, torch.cuda.current_stream(dev).cuda_stream), "prefetch_rows")
    assert torch.equal(x, want)
