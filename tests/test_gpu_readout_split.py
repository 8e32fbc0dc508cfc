"""The fused readout with a token's routes split over a block's waves: every token count around the
lines between its forms, route counts around the 32-route chunks, the first positions (no rows), and
the cached and supplied-row modes.

Against fp64 the readout is bf16 operands with fp32 sums (2e-2 norm-relative, the layer's bound); one
form against another is held to 2^-7 here, and bit for bit in ``test_gpu_readout_bits.py``."""

from __future__ import annotations

import math

import pytest
import torch

from lngram_hip import ops

pytestmark = pytest.mark.gpu

EPS = 1e-5


def _weights(R, dev, seed=0):
    gen = torch.Generator(device=dev).manual_seed(seed + R)

    def rnd(*shape, std):
        return (torch.randn(*shape, generator=gen, device=dev) * std).to(torch.bfloat16)

    kv = rnd(512, 256, std=0.05)
    return gen, rnd(R * 256, 128, std=0.02), rnd(R * 4096, 128, std=0.02), kv, rnd(256, std=1.0)


def _fp64(q, codes, t2, t3, kv, wm):
    B, T, R = codes.shape
    c, base = codes.long(), torch.arange(R, device=codes.device)
    x = torch.zeros(B, T, R, 256, dtype=torch.float64, device=codes.device)
    if T > 1:
        x[:, 1:, :, :128] = t2[base * 256 + c[:, :-1] + 16 * c[:, 1:]].double()
    if T > 2:
        x[:, 2:, :, 128:] = t3[base * 4096 + c[:, :-2] + 16 * c[:, 1:-1] + 256 * c[:, 2:]].double()
    x = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * wm.double()
    k = (x @ kv[:256].double().t()).view(B, T, R, 4, 64).permute(0, 1, 3, 4, 2)
    v = (x @ kv[256:].double().t()).view(B, T, R, 4, 64).permute(0, 1, 3, 2, 4)
    s = (q.double().view(B, T, 4, 4, 64) @ k) * 0.125
    p = torch.softmax(torch.cat((s, torch.full_like(s[..., :1], math.log(R))), -1), -1)[..., :-1]
    return (p @ v).reshape(B, T, 1024)


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30))


@pytest.mark.parametrize("B,T,R", [(1, 1, 184), (1, 3, 1), (4, 4, 32), (2, 8, 33), (1, 256, 181), (1, 257, 184),
                                   (2, 256, 256), (1, 513, 40), (1, 2048, 33), (1, 2049, 33), (5, 512, 33),
                                   (1, 2561, 33)])
def test_forms_match_fp64(dev, B, T, R):
    gen, t2, t3, kv, wm = _weights(R, dev)
    q = torch.randn(B, T, 1024, generator=gen, device=dev).to(torch.bfloat16) * 3
    codes = torch.randint(0, 16, (B, T, R), generator=gen, device=dev, dtype=torch.uint8)
    args = (t2, t3, ops.memory_readout_pack(kv), wm, EPS, 0.125, math.log(R))
    got = ops.memory_readout_fused(q, codes, *args)
    ref = _fp64(q, codes, t2, t3, kv, wm)
    assert torch.isfinite(got.float()).all() and bool((got[:, 0] == 0).all())
    if T > 1:
        assert _rel(got, ref) < 2e-2
    # the last tokens alone, read from the same codes as a cache: the form for few tokens
    n = min(T, 5)
    tail = ops.memory_readout_fused_at(q[:, T - n:].contiguous(), codes, T - n, *args)
    if T > 1:
        assert _rel(tail, got[:, T - n:]) < 2.0 ** -7
    # the same rows supplied by the caller give the same output bit for bit
    rows = ops.route_tokens(codes, [t2, t3], (2, 3), 4)[:, T - n:].contiguous()
    assert torch.equal(ops.memory_readout_fused_rows(q[:, T - n:].contiguous(), rows, *args[2:]), tail)


@pytest.mark.parametrize("n", [1, 7, 256, 300, 512])
def test_scaled_queries_and_device_positions(dev, n):
    R = 184
    gen, t2, t3, kv, wm = _weights(R, dev)
    rows = torch.randn(1, n, 1024, generator=gen, device=dev).to(torch.bfloat16)
    q = torch.randn(1, n, 1024, generator=gen, device=dev).to(torch.bfloat16) * 3
    codes = torch.randint(0, 16, (1, n + 9, R), generator=gen, device=dev, dtype=torch.uint8)
    args = (t2, t3, ops.memory_readout_pack(kv), wm, EPS, 0.125, math.log(R))
    got = ops.memory_readout_fused_at(q, codes, 9, *args, q_rows=rows, q_eps=EPS)
    scaled = (q.double() * torch.rsqrt(rows.double().pow(2).mean(-1, keepdim=True) + EPS))
    ref = _fp64(torch.cat((torch.zeros(1, 9, 1024, device=dev, dtype=torch.float64), scaled), 1), codes, t2, t3, kv, wm)
    assert _rel(got, ref[:, 9:]) < 2e-2
    pos = torch.tensor([9], dtype=torch.int32, device=dev)
    assert torch.equal(ops.memory_readout_fused_at(q, codes, 0, *args, q_rows=rows, q_eps=EPS, pos0_dev=pos), got)
    # large scores, and a query of zeros: the softmax states merge without overflow
    big = ops.memory_readout_fused_at(q * 1000, codes, 9, *args)
    assert torch.isfinite(big.float()).all()
    assert torch.isfinite(ops.memory_readout_fused_at(q * 0, codes, 9, *args).float()).all()


@pytest.mark.parametrize("n,H", [(1, 1), (16, 3), (300, 3), (700, 2), (64, 5)])
def test_windows_equal_their_gathered_rows(dev, n, H):
    R = 184
    gen, t2, t3, kv, wm = _weights(R, dev)
    q = torch.randn(1, n, 1024, generator=gen, device=dev).to(torch.bfloat16) * 3
    win = torch.randint(0, 16, (n, H, R), generator=gen, device=dev, dtype=torch.uint8)
    seg = torch.randint(0, 2, (n, H), generator=gen, device=dev, dtype=torch.int32)
    val = (torch.rand(n, H, generator=gen, device=dev) > 0.2).to(torch.uint8)
    tail = (ops.memory_readout_pack(kv), wm, EPS, 0.125, math.log(R))
    got = ops.memory_readout_fused_windows(q, win, seg, val, t2, t3, *tail, q_rows=q, q_eps=EPS)
    rows = ops.route_tokens(win, [t2, t3], (2, 3), 4, segment_ids=seg, valid_tokens=val, target_length=1)
    want = ops.memory_readout_fused_rows(q, rows.view(1, n, R, 256), *tail, q_rows=q, q_eps=EPS)
    assert torch.equal(got, want)
