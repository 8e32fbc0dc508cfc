"""A row of a bf16 projection has the same bits in every tile that may form it: its product, its row
statistics and its row scale, against the 256-row kernels with the row among many others (M past the
tiles' range), or with K padded by zeros to a multiple of 32 that the tiles do not take."""

from __future__ import annotations

import pytest
import torch

from lngram_hip import ops

pytestmark = pytest.mark.gpu


def _inputs(m, k, n, dev):
    gen = torch.Generator().manual_seed(m + k + n)
    return (torch.randn(m, k, generator=gen).to(torch.bfloat16).to(dev),
            torch.randn(n, k, generator=gen).to(torch.bfloat16).to(dev))


@pytest.mark.parametrize("k,n", [(1024, 1024), (256, 1000), (64, 136)])
def test_rows_of_the_projection_tiles(dev, k, n):
    x, w = _inputs(50000 if n < 200 else 8192, k, n, dev)      # past the tiles: 256-row projection kernel
    want, stats, scaled = ops.linear(x, w), ops.linear_rowsq(x, w)[1], ops.linear_rowscale(x, w, 1e-5)
    for m in (1024, 1281, 1500, 2331, 4000, 6000):             # 64 x 32, 64 x 64, 128 x 32 and 128 x 64 tiles
        y, sq = ops.linear_rowsq(x[:m], w)
        assert torch.equal(y, want[:m]) and torch.equal(ops.linear(x[:m], w), want[:m]), m
        assert torch.equal(sq, stats[:, :m]), m
        assert torch.equal(ops.linear_rowscale(x[:m], w, 1e-5), scaled[:m]), m


@pytest.mark.parametrize("m,k,n", [(65, 64, 1024), (200, 1024, 1024), (777, 192, 1000), (1023, 64, 72), (300, 128, 12)])
def test_rows_of_fewer_than_the_projection_kernels(dev, m, k, n):
    x, w = _inputs(m, k, n, dev)
    pad = [torch.cat((t, torch.zeros(len(t), 32, dtype=t.dtype, device=dev)), 1) for t in (x, w)]  # K % 64 == 32
    for got, want in zip(ops.linear_rowsq(x, w), ops.linear_rowsq(*pad)):
        assert torch.equal(got, want)
    assert torch.equal(ops.linear(x, w), ops.linear(*pad))


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_values_that_are_not_finite_stay_in_their_row(dev, bad):
    for m in (300, 1100, 2331, 4000):
        x, w = _inputs(m, 128, 1024, dev)
        want = ops.linear_rowsq(x, w)
        x[m // 2, 5] = bad
        got = ops.linear_rowsq(x, w)
        assert not torch.isfinite(got[0][m // 2].float()).any() and not torch.isfinite(got[1][:, m // 2]).any()
        keep = torch.arange(m, device=dev) != m // 2
        assert torch.equal(got[0][keep], want[0][keep]) and torch.equal(got[1][:, keep], want[1][:, keep])


@pytest.mark.parametrize("m,n,k", [(1, 1, 32), (5, 33, 64), (64, 32, 128), (512, 256, 1024), (1100, 1024, 96),
                                   (4100, 260, 160), (300, 33, 32)])
@pytest.mark.parametrize("kind", ["normal", "wide", "small"])
def test_fp32_products_are_fma_chains(dev, m, n, k, kind):
    """K padded by 16 zeros takes the VALU tile, one fmaf after another in K order: the matrix cores'
    fp32 products give the same bits, denormal sums among them."""
    gen = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn(m, k, generator=gen), torch.randn(n, k, generator=gen)
    if kind == "wide":
        x, w = (t * torch.exp2(torch.randint(-20, 21, t.shape, generator=gen).float()) for t in (x, w))
    if kind == "small":
        x, w = x * 1e-30, w * 1e-10
    x, w = x.to(dev), w.to(dev)
    px, pw = (torch.cat((t, torch.zeros(len(t), 16, device=dev)), 1) for t in (x, w))
    got, want = ops.linear(x, w), ops.linear(px, pw)
    assert torch.equal(got, want) and (got != 0).any()
    if n % 4 == 0:
        for a, b in zip(ops.router_codes(x, w, 4), ops.router_codes(px, pw, 4)):
            assert torch.equal(a, b)


@pytest.mark.parametrize("which", ["x", "w", "y"])
@pytest.mark.parametrize("m,n,k", [(70, 64, 128), (300, 36, 32)])
def test_fp32_buffers_of_any_alignment(dev, which, m, n, k):
    """fp32 buffers need 4-byte alignment only: views one element into their storage, and through the C
    ABI an output one element in."""
    gen = torch.Generator().manual_seed(m)

    def at(shape, off):
        return torch.empty(shape[0] * shape[1] + 4, device=dev)[off:off + shape[0] * shape[1]].view(shape)

    x, w = torch.randn(m, k, generator=gen).to(dev), torch.randn(n, k, generator=gen).to(dev)
    want, codes = ops.linear(x, w), ops.router_codes(x, w, 4)[1]
    x2, w2, y = at((m, k), which == "x").copy_(x), at((n, k), which == "w").copy_(w), at((m, n), which == "y")
    stream = torch.cuda.current_stream(dev).cuda_stream
    assert ops.lib().lng_linear(x2.data_ptr(), w2.data_ptr(), ops.dtype_code(torch.float32), m, n, k, y.data_ptr(), stream) == 0
    assert torch.equal(y, want)
    if which != "y":
        assert torch.equal(ops.linear(x2, w2), want)
        for a, b in zip(ops.router_codes(x2, w2, 4), (want, codes)):
            assert torch.equal(a, b)


@pytest.mark.parametrize("m,n,k", [(1, 256, 1024), (33, 4, 64), (200, 36, 128), (2560, 256, 192), (2561, 256, 64),
                                   (4097, 260, 128), (8192, 256, 1024), (20000, 64, 256), (3, 8, 4096),
                                   (33, 36, 4160), (1100, 1028, 4160), (5000, 260, 8192)])
def test_norm_and_product_in_one_pass(dev, m, n, k):
    gen = torch.Generator().manual_seed(m + n + k)
    x = (torch.randn(m, k, generator=gen) * torch.exp2(torch.randint(-30, 30, (m, 1), generator=gen).float()))
    x = x.to(torch.bfloat16).to(dev)
    if m > 4:
        x[1], x[2, 3], x[3, k - 1] = 0.0, float("inf"), float("nan")
    w, nw = (torch.randn(n, k, generator=gen) * 0.02).to(dev), (torch.rand(k, generator=gen) + 0.5).to(dev)
    assert ops.lib().lng_linear_split_workspace_bytes(n, k) > 0
    got = ops.norm_linear_fp32(x, nw, w, 1e-5)
    want = ops.linear(ops.rmsnorm(x.float(), nw, 1e-5), w)
    assert torch.equal(torch.nan_to_num(got, 7.0), torch.nan_to_num(want, 7.0))
    assert torch.equal(got.isnan(), want.isnan()) and (m <= 4 or bool(got[2:4].isnan().all()))


@pytest.mark.parametrize("which", ["x", "w", "both"])
def test_norm_and_product_of_rows_at_odd_addresses(dev, which):
    """The kernel reads whole 16-byte pieces: other views of x and w are copied by the binding, and the library
    takes a w of its own through an aligned copy in the workspace."""
    m, n, k = 100, 36, 128
    gen = torch.Generator().manual_seed(3)
    x = torch.randn(m, k, generator=gen).to(torch.bfloat16).to(dev)
    w, nw = (torch.randn(n, k, generator=gen) * 0.02).to(dev), (torch.rand(k, generator=gen) + 0.5).to(dev)
    want = ops.norm_linear_fp32(x, nw, w, 1e-5)

    def at(t, odd):
        return torch.empty(t.numel() + 8, dtype=t.dtype, device=dev)[odd:odd + t.numel()].view(t.shape).copy_(t)

    x2, w2 = at(x, int(which != "w")), at(w, int(which != "x"))
    assert torch.equal(ops.norm_linear_fp32(x2, nw, w2, 1e-5), want)
    nws = ops.lib().lng_linear_split_workspace_bytes(n, k)
    y, ws = torch.empty(m, n, device=dev), torch.empty(nws, dtype=torch.uint8, device=dev)
    stream = torch.cuda.current_stream(dev).cuda_stream

    def call(xt, space, size):
        return ops.lib().lng_linear_split(xt.data_ptr(), nw.data_ptr(), w2.data_ptr(), m, n, k, 1e-5, space, size,
                                          y.data_ptr(), stream)

    if which == "w":
        assert call(x2, None, 0) == -1 and call(x2, ws.data_ptr(), nws - 1) == -1
        assert call(x2, ws.data_ptr(), nws) == 0 and torch.equal(y, want)
    else:
        assert call(x2, ws.data_ptr(), nws) == -1
